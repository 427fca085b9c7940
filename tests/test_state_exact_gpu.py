"""Chunks of the recurrence whose q, k and v are bf16 values as they lie (the other
operand in three bf16 parts): values that are not finite in any operand, decays beyond
one, sums that leave fp32; and the rule that cuts such sequences into runs."""
import math

import pytest
import torch

from gpustack_amd import ops


def _walk32(src, cb, cc, H, N, P, a, state, hist):
    """Row by row in fp32, which decides what is finite."""
    T = src.shape[0]
    y = torch.zeros(T, H, P, device="cuda")
    S = state.clone() if hist else torch.zeros_like(state)
    for t in range(T):
        v = src[t, :H * P].float().view(H, P)
        k, q = (src[t, c:c + H * N].float().view(H, N) for c in (cb, cc))
        S = a[:, None, None] * S + k[:, :, None] * v[:, None, :]
        y[t] = (S * q[:, :, None]).sum(1)
    return y.view(T, H * P), S


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("size", [0, 64])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("where", ["q", "k", "v", "state", "large"])
@pytest.mark.parametrize("at", [0, 37, 129])
def test_not_finite_anywhere(where, bad, at, size):
    g = torch.Generator(device="cuda").manual_seed(at)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, H, N, P = 150, 2, 72, 64
    cb, cc = H * P, H * (P + N)
    src = rnd(T, H * (P + 2 * N)).bfloat16()
    state = rnd(1, H, N, P)
    if where == "state":
        state[0, 1, 5, 9] = bad
    elif where == "large":                 # finite, but not its products
        src[at, [3, cb + 4, cc + 5]] = 1e30
    else:
        src[at, {"q": cc, "k": cb, "v": 0}[where] + 7] = bad
    decay = torch.tensor([0.9, -0.97], device="cuda")
    ref, ref_s = _walk32(src, cb, cc, H, N, P, decay, state[0], True)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    y = torch.zeros(T, H * P, device="cuda")
    ops.state_scan(y, src, 0, cb, cc, None, 0, H, H, N, P, False, None, None,
                   None, decay, state, i32([0]), i32([T]), i32([0]),
                   i32(list(range(3, 3 + T))),
                   runs=ops.build_scan_chunks([0], [T], size, "cuda")
                   if size else None)
    for got, want in ((y, ref), (state[0], ref_s)):
        ok = want.isfinite()
        assert torch.equal(got.isfinite(), ok)
        # rows of one head that are large throughout stand beside others
        for h in range(H):
            o = ok.view(-1, H, P)[:, h] if got is y else ok[h]
            a, b = (t.view(-1, H, P)[:, h] if got is y else t[h]
                    for t in (got, want))
            if bool(o.any()):
                scale = float(b[o].abs().double().max())
                # two fp32 sums of a few hundred products each
                assert float((a[o].double() - b[o].double()).abs().max()) \
                    <= 2e-5 * scale


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("size", [0, 64, 160])
@pytest.mark.parametrize("N,P", [(32, 32), (48, 72), (128, 64), (120, 136)])
def test_decays_beyond_one(N, P, size):
    g = torch.Generator(device="cuda").manual_seed(N)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, H = 330, 3                          # 11 chunks, over two sets of decays
    cb, cc = H * P, H * (P + N)
    src = rnd(T, H * (P + 2 * N)).bfloat16()
    state = rnd(2, H, N, P)
    decay = torch.tensor([1.02, -1.01, 1.0], device="cuda")
    S = state[1].double()
    ref = torch.zeros(T, H, P, dtype=torch.float64, device="cuda")
    for t in range(T):
        v = src[t, :H * P].double().view(H, P)
        k, q = (src[t, c:c + H * N].double().view(H, N) for c in (cb, cc))
        S = decay.double()[:, None, None] * S + k[:, :, None] * v[:, None, :]
        ref[t] = (S * q[:, :, None]).sum(1)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    y = torch.zeros(T, H * P, device="cuda")
    ops.state_scan(y, src, 0, cb, cc, None, 0, H, H, N, P, False, None, None,
                   None, decay, state, i32([0]), i32([T]), i32([1]),
                   i32(list(range(5, 5 + T))),
                   runs=ops.build_scan_chunks([0], [T], size, "cuda")
                   if size else None)
    for got, want in ((y.view(T, H, P), ref), (state[1], S)):
        for h in range(H):                 # heads differ in size by e^6
            a, b = (t[:, h] if got.shape[0] == T else t[h] for t in (got, want))
            # fp32: the decay itself is off by 2^-25 a row, 330 rows of it
            assert float((a.double() - b).abs().max()) \
                <= 330 * 2.0 ** -24 * float(b.abs().max())


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("N,P,T", [(128, 128, 96), (64, 64, 90), (72, 40, 101)])
def test_weighted_values_are_rounded_not_cut(N, P, T):
    # decays that leave nothing of the row before: the state is one product, k v b
    g = torch.Generator(device="cuda").manual_seed(N)
    H = 4
    cb, cc, cdt = H * P, H * (P + N), H * (P + 2 * N)
    src = torch.randn(T, (cdt + H + 15) // 8 * 8, generator=g,
                      device="cuda").bfloat16()
    src[:, cdt:] = 0
    bias = 20 + torch.rand(H, generator=g, device="cuda") * 10   # softplus(b) = b
    state = torch.zeros(1, H, N, P, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    ops.state_scan(torch.zeros(T, H * P, device="cuda"), src, 0, cb, cc, src, cdt,
                   H, H, N, P, False, bias, torch.full((H,), 5., device="cuda"),
                   None, None, state, i32([0]), i32([T]), i32([0]),
                   i32(list(range(5, 5 + T))))
    v = src[-1, :cb].double().view(H, 1, P) * bias.double()[:, None, None]
    ref = src[-1, cb:cc].double().view(H, N, 1) * v
    ulp = torch.exp2(torch.floor(torch.log2(ref.abs().clamp(min=1e-30))) - 23)
    off = (state[0].double() - ref) * ref.sign() / ulp
    # half an ulp at the sum's end, half where its small terms meet the large one, a
    # quarter of v b's parts; towards 0 as often as away from it
    assert float(off.abs().max()) <= 1.25
    assert abs(float(off.mean())) < 0.05


def test_runs_of_exact_rows():
    rule = lambda news, heads, vdim: ops.scan_run_rows(news, heads, vdim, True)
    for n in (640, 1000, 4000, 8000, 100000):
        size = rule([n], 64, 64)
        assert size % 32 == 0
        # no more workgroups than the chip has places for
        assert -(-n // size) * 64 <= 512
        assert 0 <= size - max(n / 8, 12 * math.sqrt(n)) < 32
    assert rule([639], 64, 64) == 0 and rule([4000] * 3, 64, 64) == 0
    assert rule([301, 1900, 821, 1340, 1660, 1100], 64, 64) == 0
    assert rule([301, 1900, 821, 1340, 1660, 1100], 16, 128) > 0
    # too few rows a sequence for chunks
    assert rule([1900] + [1] * 85, 64, 64) == 0
    # a long one among many short ones is cut
    assert rule([87, 1, 19, 19, 33, 1389, 235, 2, 51, 13, 1, 1, 1, 1159, 5, 32, 4, 1,
                 345, 12, 34, 18, 313, 153], 64, 64) == 512

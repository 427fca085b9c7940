"""The recurrence in chunks against a walk row by row in float64: portions at
the edges of a chunk (32 rows), states that pad the tiles, decays from 1 to
next to nothing and below zero, fresh and continued sequences in one batch."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(),
                                 reason="needs a GPU")]


def _walk(src, cx, cb, cc, H, G, N, P, act, a, b, skip, state, news, hists,
          slots):
    f = lambda t: torch.nn.functional.silu(t) if act else t
    y = torch.zeros(src.shape[0], H, P, dtype=torch.float64, device="cuda")
    st = state.double()
    r0 = 0
    src = src.double()
    for n, hist, slot in zip(news, hists, slots):
        S = st[slot].clone() if hist else torch.zeros_like(st[slot])
        for t in range(r0, r0 + n):
            v = f(src[t, cx:cx + H * P]).view(H, P)
            k, q = (f(src[t, c:c + G * N]).view(G, N).repeat_interleave(
                H // G, 0) for c in (cb, cc))
            S = a[t][:, None, None] * S \
                + (b[t][:, None] * k)[:, :, None] * v[:, None, :]
            y[t] = (S * q[:, :, None]).sum(1)
            if skip is not None:
                y[t] += skip.double()[:, None] * v
        st[slot] = S
        r0 += n
    return y.view(src.shape[0], H * P), st


@pytest.mark.parametrize("kind", ["steps", "wide steps", "constants"])
@pytest.mark.parametrize("H,G,N,P", [(4, 2, 128, 64), (3, 3, 64, 128),
                                     (2, 1, 40, 72), (2, 2, 104, 32)])
@pytest.mark.parametrize("news", [[31, 32, 33, 1, 64], [200, 7], [130]])
def test_chunks(kind, H, G, N, P, news):
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(sum(news) + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, S = sum(news), len(news)
    hists = [0, 5, 0, 9, 3][:S]
    slots = [3, 0, 5, 1, 2][:S]
    cb, cc = 8 + H * P, 8 + H * P + G * N
    cdt = cc + G * N
    src = (rnd(T, (cdt + H + 15) // 8 * 8) * 0.7).bfloat16()
    state = rnd(7, H, N, P)
    act = kind == "constants"
    if act:
        decay = torch.tensor([1.0, 0.0, -0.5, 0.97], device="cuda")[:H]
        args = (None, 0, H, G, N, P, True, None, None, None, decay)
        a = decay.double().expand(T, H)
        b, skip = torch.ones_like(a), None
    else:
        # wide: decays down to e^-100, where a product underflows
        a_log = rnd(H) * 0.5 + (4.0 if kind == "wide steps" else 0.0)
        bias, skip = rnd(H) - 1, rnd(H)
        args = (src, cdt, H, G, N, P, False, bias, a_log, skip, None)
        b = torch.nn.functional.softplus(
            src[:, cdt:cdt + H].double() + bias.double())
        a = torch.exp(-torch.exp(a_log.double()) * b)
    ref_y, ref_s = _walk(src, 8, cb, cc, H, G, N, P, act, a, b, skip, state,
                         news, hists, slots)
    first = [sum(news[:i]) for i in range(S)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    pos = i32([h + j for h, n in zip(hists, news) for j in range(n)])
    y = torch.zeros(T, H * P, device="cuda")
    st = state.clone()
    ops.state_scan(y, src, 8, cb, cc, *args, st, i32(first), i32(news),
                   i32(slots), pos)
    # fp32 throughout: a row adds up to a few hundred products, each off by a
    # few 2^-24 of itself, and exponentials of sums that double keeps exact
    for got, ref in ((y, ref_y), (st, ref_s)):
        scale = float(ref.abs().max())
        assert float((got.double() - ref).abs().max()) <= 4e-6 * scale
    assert torch.equal(st[6], state[6])


@pytest.mark.parametrize("size", [32, 64, 96])
@pytest.mark.parametrize("kind", ["steps", "wide steps", "constants"])
@pytest.mark.parametrize("H,G,N,P", [(4, 2, 128, 64), (3, 3, 64, 128),
                                     (2, 1, 40, 72)])
@pytest.mark.parametrize("news", [[31, 65, 33, 1, 64], [200, 7], [97]])
def test_runs(size, kind, H, G, N, P, news):
    """Sequences cut into runs of rows (one to seven of them): as without."""
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(sum(news) + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, S = sum(news), len(news)
    hists, slots = [7, 5, 0, 9, 3][:S], [3, 0, 5, 1, 2][:S]
    cb, cc = 8 + H * P, 8 + H * P + G * N
    cdt = cc + G * N
    src = (rnd(T, (cdt + H + 15) // 8 * 8) * 0.7).bfloat16()
    state = rnd(7, H, N, P)
    if kind == "constants":
        decay = torch.tensor([1.0, 0.0, -0.5, 0.97], device="cuda")[:H]
        args = (None, 0, H, G, N, P, True, None, None, None, decay)
        a = decay.double().expand(T, H)
        b, skip = torch.ones_like(a), None
    else:
        a_log = rnd(H) * 0.5 + (4.0 if kind == "wide steps" else 0.0)
        bias, skip = rnd(H) - 1, rnd(H)
        args = (src, cdt, H, G, N, P, False, bias, a_log, skip, None)
        b = torch.nn.functional.softplus(
            src[:, cdt:cdt + H].double() + bias.double())
        a = torch.exp(-torch.exp(a_log.double()) * b)
    ref_y, ref_s = _walk(src, 8, cb, cc, H, G, N, P, kind == "constants", a, b,
                         skip, state, news, hists, slots)
    first = [sum(news[:i]) for i in range(S)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    pos = i32([h + j for h, n in zip(hists, news) for j in range(n)])
    y = torch.zeros(T, H * P, device="cuda")
    st = state.clone()
    ops.state_scan(y, src, 8, cb, cc, *args, st, i32(first), i32(news),
                   i32(slots), pos,
                   runs=ops.build_scan_chunks(first, news, size, "cuda"))
    # the bound of test_chunks: a state put together from runs has two more
    # roundings a run
    for got, ref in ((y, ref_y), (st, ref_s)):
        scale = float(ref.abs().max())
        assert float((got.double() - ref).abs().max()) <= 4e-6 * scale
    assert torch.equal(st[6], state[6])


@pytest.mark.parametrize("size", [0, 32])
@pytest.mark.parametrize("decay", [0.9, 0.0])
@pytest.mark.parametrize("hist", [0, 3])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("at", [5, 40, 90])
def test_not_finite_in_runs(at, bad, hist, decay, size):
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(at)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, H, N, P = 130, 2, 64, 96
    src = rnd(T, H * (P + 2 * N)).bfloat16()
    src[at, P + 70] = bad
    decay = torch.tensor([0.9, decay], device="cuda")
    state = rnd(2, H, N, P)
    cb, cc = H * P, H * (P + N)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    y = torch.zeros(T, H * P, device="cuda")
    a = decay.double().expand(T, H)
    ref, ref_s = _walk(src, 0, cb, cc, H, H, N, P, False, a,
                       torch.ones_like(a), None, state, [T], [hist], [0])
    ops.state_scan(y, src, 0, cb, cc, None, 0, H, H, N, P, False, None, None,
                   None, decay, state, i32([0]), i32([T]), i32([0]),
                   i32(list(range(hist, hist + T))),
                   runs=ops.build_scan_chunks([0], [T], size, "cuda")
                   if size else None)
    for got, want in ((y, ref), (state, ref_s)):
        ok = want.isfinite()
        assert torch.equal(got.isfinite(), ok)
        scale = float(want[ok].abs().max())    # fp32 sums, as above
        assert float((got[ok].double() - want[ok]).abs().max()) <= 4e-6 * scale


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("at", [5, 20, 47])
def test_not_finite(bad, at):
    """A value reaches its own row and the rows behind it, of its channel."""
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(at)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, H, N, P = 70, 2, 64, 96
    src = rnd(T, H * (P + 2 * N)).bfloat16()
    src[at, P + 70] = bad                      # head 1, channel 70
    decay = torch.tensor([0.9, -0.97], device="cuda")
    state = torch.zeros(2, H, N, P, device="cuda")
    cb, cc = H * P, H * (P + N)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    y = torch.zeros(T, H * P, device="cuda")
    ops.state_scan(y, src, 0, cb, cc, None, 0, H, H, N, P, False, None, None,
                   None, decay, state, i32([0]), i32([T]), i32([0]),
                   i32(list(range(T))))
    a = decay.double().expand(T, H)
    ref, ref_s = _walk(src, 0, cb, cc, H, H, N, P, False, a,
                       torch.ones_like(a), None,
                       torch.zeros(2, H, N, P, device="cuda"), [T], [0], [0])
    for got, want in ((y, ref), (state, ref_s)):
        ok = want.isfinite()
        assert torch.equal(got.isfinite(), ok)
        scale = float(want[ok].abs().max())    # fp32 sums, as above
        assert float((got[ok].double() - want[ok]).abs().max()) <= 4e-6 * scale
    assert bool(ref[:at].isfinite().all()) and not bool(
        ref[at:, P + 70].isfinite().any())


@pytest.mark.parametrize("bad", [None, float("inf"), float("nan")])
@pytest.mark.parametrize("news", [[20, 130, 64, 200, 31], [96, 97, 1, 60]])
def test_whole_sequences_behind_the_runs(news, bad):
    """Sequences of one run have no places in the workspace, also where their
    columns are walked again on the slot."""
    from gpustack_amd import ops

    g = torch.Generator(device="cuda").manual_seed(sum(news))
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, S, H, N, P = sum(news), len(news), 2, 64, 96
    hists, slots = [7, 5, 0, 9, 3][:S], [3, 0, 5, 1, 2][:S]
    src = rnd(T, H * (P + 2 * N)).bfloat16()
    first = [sum(news[:i]) for i in range(S)]
    if bad is not None:
        for f, n in zip(first, news):
            src[f + n // 2, P + 70] = bad
    decay = torch.tensor([0.9, -0.97], device="cuda")
    state = rnd(7, H, N, P)
    cb, cc = H * P, H * (P + N)
    a = decay.double().expand(T, H)
    ref, ref_s = _walk(src, 0, cb, cc, H, H, N, P, False, a,
                       torch.ones_like(a), None, state, news, hists, slots)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    y = torch.zeros(T, H * P, device="cuda")
    runs, cut = ops.build_scan_runs(first, news, 64, "cuda")
    assert 0 < cut < len(runs)
    spare = state[6].clone()
    ops.state_scan(y, src, 0, cb, cc, None, 0, H, H, N, P, False, None, None,
                   None, decay, state, i32(first), i32(news), i32(slots),
                   i32([h + j for h, n in zip(hists, news) for j in range(n)]),
                   runs=runs, cut=cut)
    for got, want in ((y, ref), (state, ref_s)):
        ok = want.isfinite()
        assert torch.equal(got.isfinite(), ok)
        scale = float(want[ok].abs().max())    # fp32 sums, as above
        assert float((got[ok].double() - want[ok]).abs().max()) <= 4e-6 * scale
    assert torch.equal(state[6], spare)

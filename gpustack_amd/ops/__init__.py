"""gpustack_amd.ops — dispatch layer for the CDNA4 HIP kernels.

On a GPU box the in-tree `_hip_ops.so` (hand-written gfx950 kernels) is
REQUIRED: there is no silent eager fallback — a missing extension raises at
first use so a broken build can't masquerade as the native path. On CPU-only
hosts the fp32 torch reference implementations run instead, which keeps the
engine/control-plane logic testable without hardware.
"""
from __future__ import annotations

import functools
import math
import os
from pathlib import Path

import torch

from . import torch_ref

_HIP_SO = Path(__file__).resolve().parent / "_hip_ops.so"
_HIP = None
_HIP_ERR: str | None = None


def _load_hip():
    global _HIP, _HIP_ERR
    if _HIP is not None or _HIP_ERR is not None:
        return _HIP
    try:
        import importlib.util

        so = _HIP_SO
        if not so.exists():
            raise ImportError(
                f"{so} not found — build it with `python -m gpustack_amd.ops.build` "
                "(hipcc --offload-arch=gfx950)"
            )
        spec = importlib.util.spec_from_file_location("gpustack_amd.ops._hip_ops", so)
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        _HIP = mod
    except Exception as e:  # noqa: BLE001
        _HIP_ERR = str(e)
        raise
    return _HIP


def hip_available() -> bool:
    if not torch.cuda.is_available():
        return False
    try:
        return _load_hip() is not None
    except Exception:  # noqa: BLE001
        return False


def to_device(parts, device) -> list[torch.Tensor]:
    """Host integers on the device: `parts` is a list of (values, dtype), values
    a list of ints, an array or a CPU tensor. On a GPU they go through pinned
    memory in ONE copy that waits for nothing, so that the host can prepare a
    step while the GPU works on the one before (torch's copies from ordinary
    memory wait for the stream, each of them)."""
    import array

    import numpy as np

    kinds = {torch.int32: ("i", np.int32), torch.int64: ("q", np.int64)}
    host = []
    for v, dtype in parts:
        if isinstance(v, list) and v and isinstance(v[0], int) \
                and dtype in kinds:
            # refuses what the type does not hold, as torch.tensor does
            v = np.frombuffer(array.array(kinds[dtype][0], v), kinds[dtype][1])
        host.append(torch.as_tensor(v, dtype=dtype))
    device = torch.device(device)
    if device.type != "cuda":
        return [t.to(device) for t in host]
    at, n = [], 0
    for t in host:                       # 16-byte places
        at.append(n)
        n += (t.numel() * t.element_size() + 15) // 16 * 16
    pin = torch.empty(max(n, 16), dtype=torch.uint8, pin_memory=True)
    part = lambda buf, t, o: buf[o:o + t.numel() * t.element_size()] \
        .view(t.dtype).view(t.shape)
    for t, o in zip(host, at):
        part(pin, t, o).copy_(t)
    dev = pin.to(device, non_blocking=True)
    return [part(dev, t, o) for t, o in zip(host, at)]


def _products():
    """The main library, or None in a checkout without it: the models that
    come with libraries of their own run there on the library's products."""
    if _HIP is None and not _HIP_SO.exists():
        return None
    return _load_hip()


def _backend(t: torch.Tensor):
    if t.is_cuda:
        return _load_hip()  # raises loudly if the native build is missing
    return None


def _oss_kernels_enabled() -> bool:
    """GPT-OSS CDNA4 kernel variants (head_dim-64 + attention sinks +
    sliding window in attn_decode/attn_prefill.hip) are written and
    compile-checked but not yet GPU-validated — opt in explicitly until
    the r3 numerics pass (tests/test_ops_gpu.py oss tests)."""
    return os.environ.get("GPUSTACK_AMD_OSS_KERNELS", "0") == "1"


def _mla_kernel_enabled() -> bool:
    return os.environ.get("GPUSTACK_AMD_MLA_KERNEL", "0") == "1"


def _sinks_f32(sinks):
    if sinks is not None and (sinks.dtype != torch.float32
                              or not sinks.is_contiguous()):
        sinks = sinks.float().contiguous()
    return sinks


# --- op surface -----------------------------------------------------------

def rms_norm(out, x, weight, eps: float) -> None:
    hip = _backend(x)
    if hip is not None:
        hip.rms_norm(out, x, weight, eps)
    else:
        torch_ref.rms_norm(out, x, weight, eps)


def add_rms_norm(x, residual, weight, eps: float):
    """residual += x and the norm of it, which is returned: in x, or where x is
    the parts of a product (linear_auto with `parts`) or the bf16 rows of each
    row's experts [T, k, H], in a tensor of its own."""
    if x.dim() == 3:
        out = torch.empty_like(residual)
        _load_hip().fused_add_rms_norm(out, residual, weight, eps, x)
        return out
    fused_add_rms_norm(x, residual, weight, eps)
    return x


def add_rms_norm_rows(x, residual, weight, eps: float, rows):
    """add_rms_norm's result at the given rows, residual left as it is or not:
    the last norm, of the rows whose logits are asked for. The caller has seen
    that there are such rows: the GPU clamps others."""
    if residual.is_cuda and residual.is_contiguous() and rows.is_cuda \
            and rows.dim() == 1 and rows.is_contiguous() \
            and residual.dtype == torch.bfloat16 and residual.dim() == 2 \
            and residual.shape[0] > 0 and rows.dtype == torch.int64:
        out = torch.empty(rows.shape[0], residual.shape[1],
                          dtype=residual.dtype, device=residual.device)
        _load_hip().add_rms_norm_rows(out, x, residual, weight, eps, rows)
        return out
    return add_rms_norm(x, residual, weight, eps)[rows]


def embed_rms_norm(tokens, embed, weight, eps: float):
    """(rows of the tokens, their norm). GPU only (embed_rms_norm_ok). The
    caller has seen that the table has such rows: others come out as zeros."""
    x = torch.empty(tokens.shape[0], embed.shape[1], dtype=embed.dtype,
                    device=embed.device)
    out = torch.empty_like(x)
    _load_hip().embed_rms_norm(out, x, tokens, embed, weight, eps)
    return x, out


def embed_rms_norm_ok(tokens, embed) -> bool:
    return (tokens.is_cuda and tokens.dim() == 1 and tokens.is_contiguous()
            and tokens.dtype == torch.int64 and embed.is_contiguous()
            and embed.dtype == torch.bfloat16 and embed.shape[1] % 8 == 0)


def fused_add_rms_norm(x, residual, weight, eps: float) -> None:
    hip = _backend(x)
    if hip is not None:
        hip.fused_add_rms_norm(x, residual, weight, eps)
    else:
        torch_ref.fused_add_rms_norm(x, residual, weight, eps)


def rotary_embedding(positions, q, k, cos_sin, head_dim: int, rot_dim: int,
                     mode: str = "neox") -> None:
    hip = _backend(q)
    if hip is not None:
        if mode != "neox":
            raise NotImplementedError(
                "pairwise (GPT-J style) rotary is not in the CDNA4 kernel "
                "yet (Ernie/Hunyuan/MiniMax GPU serving lands with it in "
                "r3); CPU serving is available")
        hip.rotary_embedding(positions, q, k, cos_sin, head_dim, rot_dim)
    else:
        torch_ref.rotary_embedding(positions, q, k, cos_sin, head_dim,
                                   rot_dim, mode=mode)


def silu_and_mul(out, x) -> None:
    hip = _backend(x)
    if hip is not None:
        hip.silu_and_mul(out, x)
    else:
        torch_ref.silu_and_mul(out, x)


def reshape_and_cache(k, v, k_cache, v_cache, slots) -> None:
    hip = _backend(k)
    if hip is not None:
        hip.reshape_and_cache(k, v, k_cache, v_cache, slots)
    else:
        torch_ref.reshape_and_cache(k, v, k_cache, v_cache, slots)


def qkv_store_ok(qkv, head_dim: int, rot_dim: int, mode: str) -> bool:
    """True where ops.qkv_store takes a fused projection: bf16 rows on the
    GPU, whole heads of 64, 128 or 256 channels rotated in halves."""
    return (qkv.is_cuda and qkv.dtype == torch.bfloat16 and qkv.dim() == 2
            and qkv.is_contiguous() and mode == "neox"
            and rot_dim == head_dim and head_dim in (64, 128, 256))


def qkv_store(qkv, q_heads: int, kv_heads: int, q_norm, k_norm, cos_sin,
              positions, slots, k_cache, v_cache, eps: float,
              parts=None) -> None:
    """qkv [T, (q_heads + 2 kv_heads) * D]: weighted RMS norm of every q and k
    head (where weights are given), rotation of q and k in place, keys and
    values to their slots (-1: none). `parts` (linear_auto): the rows are
    their sum, and qkv is only written. GPU only (qkv_store_ok)."""
    _load_hip().qkv_store(qkv, q_heads, kv_heads, q_norm, k_norm, cos_sin,
                          positions, slots, k_cache, v_cache, eps, parts)


def greedy_sample_into(out, logits, host=None) -> None:
    """`host`: the words once more, pinned where the logits are on the GPU; they
    are there when work behind this call is (a copy less: 2 to 3 us of a step)."""
    if logits.is_cuda and logits.dtype == torch.float32:
        # fp32-logit models: whichever fp32-stream library is loaded
        (_PAGED if _PAGED is not None else _load_latent()).argmax_f32(
            out, logits, host)
        return
    hip = _backend(logits)
    if hip is not None:
        hip.greedy_sample(out, logits, host)
    else:
        torch_ref.greedy_sample(out, logits)
        if host is not None:
            host.copy_(out)


def greedy_sample(logits) -> torch.Tensor:
    out = torch.empty(logits.shape[0], dtype=torch.long, device=logits.device)
    if logits.is_cuda and logits.dtype == torch.float32:
        _load_latent().argmax_f32(out, logits)  # fp32-logit models
        return out
    hip = _backend(logits)
    if hip is not None:
        hip.greedy_sample(out, logits)
    else:
        torch_ref.greedy_sample(out, logits)
    return out


def paged_attn_decode(out, q, k_cache, v_cache, block_tables, seq_lens,
                      scale: float, sinks=None, window: int = 0,
                      softcap: float = 0.0) -> None:
    hip = _backend(q)
    if hip is not None:
        if (sinks is not None or window or softcap or q.shape[-1] != 128) \
                and not _oss_kernels_enabled():
            # the sinks/window/softcap and D!=128 kernel variants are
            # written but not yet GPU-validated — fail loudly rather than
            # silently mis-attend (opt in with GPUSTACK_AMD_OSS_KERNELS=1;
            # r3 flips the default after the validation pass)
            raise NotImplementedError(
                "sinks/window/softcap/D!=128 CDNA4 decode kernel variants "
                "are unvalidated — set GPUSTACK_AMD_OSS_KERNELS=1 to opt in")
        hip.paged_attn_decode(out, q, k_cache, v_cache, block_tables, seq_lens,
                              scale, sinks=_sinks_f32(sinks), window=window,
                              softcap=softcap)
    else:
        torch_ref.paged_attn_decode(out, q, k_cache, v_cache, block_tables,
                                    seq_lens, scale, sinks=sinks,
                                    window=window, softcap=softcap)


def paged_attn_decode_rows_ok(rows, q_heads: int, kv_heads: int, head_dim: int,
                              k_cache, v_cache, block_tables, *norms) -> bool:
    """Whether paged_attn_decode_rows takes a step: heads of 128 channels, two to
    eight of them (not three) a kv head, without sinks, window or score cap, pools and
    head norms (`norms`, or None) at 16-byte addresses; and where it is the faster one.
    It saves 1.2 to 2.7 us up to four workgroups a CU whatever the lengths (128 rows of 8 kv heads 14.5 -> 13.4 at 40 keys, 41.9 ->
    39.2 at 256 to 383). Behind them it loses contexts under 80 keys (256 rows of 40
    to 58 21.9 -> 22.8, 512 36.8 -> 40.7) and gains longer ones (80 to 109 54.5 ->
    54.7, 100 to 149 67.6 -> 64.5): it is taken where the block table has room for
    128. fp8 pages, whose steps are shorter, up to two a CU (64 rows 9.8 -> 8.4 and
    17.0 -> 15.3; 128 15.7 -> 17.1 at 80 to 109 keys, 27.2 -> 26.8 at 256 to 383)."""
    group = q_heads // kv_heads
    groups, pages = block_tables.shape[0] * kv_heads, block_tables.shape[1]
    return (rows.is_cuda and head_dim == 128 and q_heads % kv_heads == 0
            and group in (2, 4, 5, 6, 7, 8)
            and (groups <= 512 if k_cache.element_size() == 1
                 else groups <= 1024 or pages >= 8)
            and not any(t.data_ptr() % 16 for t in (k_cache, v_cache, *norms)
                        if t is not None))


def paged_attn_decode_rows(out, rows, q_heads: int, kv_heads: int, q_norm, k_norm,
                           cos_sin, positions, slots, k_cache, v_cache,
                           block_tables, seq_lens, eps: float, scale: float) -> None:
    """qkv_store and paged_attn_decode in one launch, for batches of ONE row a
    sequence, each the last of its sequence: rows is the projection [N, (q_heads + 2
    kv_heads) * 128] or its fp32 parts (linear_auto). GPU only
    (paged_attn_decode_rows_ok)."""
    _load_hip().paged_attn_decode_rows(
        out, rows, q_heads, kv_heads, q_norm, k_norm, cos_sin, positions, slots,
        k_cache, v_cache, block_tables, seq_lens, eps, scale)


def mla_decode(ctx_out, q_cat, lat_cache, block_tables, seq_lens,
               scale: float) -> None:
    """MLA absorbed decode (DeepSeek): ctx_out[N,H,512] f32 = softmax
    (q_cat · lat) · lat[:, :512] over the paged latent pool. GPU-only —
    the CPU oracle lives in models/llama.py MLAAttention."""
    hip = _backend(q_cat)
    if hip is None:
        raise NotImplementedError("mla_decode is the CDNA4 kernel entry; "
                                  "CPU serving uses the torch MLA path")
    hip.mla_decode(ctx_out, q_cat, lat_cache, block_tables, seq_lens, scale)


_PREFILL_BQ = 64
# rows of a workgroup of the prompt kernels: a list of such tiles has no entry
# that they pass over (in a list of 64-row tiles every second one is)
PREFILL_ROWS = 128


def build_prefill_tiles(seq_lens: list[int], device,
                        rows: int = _PREFILL_BQ) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Map varlen sequences to q tiles of `rows` (64 or PREFILL_ROWS) for the
    MFMA kernel."""
    return tuple(to_device([(a, torch.int32) for a in
                            prefill_tile_rows(seq_lens, rows)], device))


def prefill_tile_rows(seq_lens: list[int], rows: int = _PREFILL_BQ):
    """The lists of build_prefill_tiles: each tile's sequence's first row, its
    own first row in the sequence, the sequence's length."""
    starts, q0s, lens = [], [], []
    tok = 0
    for L in seq_lens:
        for q0 in range(0, L, rows):
            starts.append(tok)
            q0s.append(q0)
            lens.append(L)
        tok += L
    return starts, q0s, lens


def varlen_prefill_attn(out, q, k, v, seq_lens: list[int], scale: float,
                        tiles=None, sinks=None, window: int = 0,
                        softcap: float = 0.0) -> None:
    hip = _backend(q)
    if hip is not None:
        d_ok = (q.shape[-1] == 128
                or (q.shape[-1] == 192 and _mla_kernel_enabled()))
        if (sinks is not None or window or softcap or not d_ok) \
                and not _oss_kernels_enabled():
            raise NotImplementedError(
                "sinks/window/softcap/D!=128 CDNA4 prefill kernel variants "
                "are unvalidated — set GPUSTACK_AMD_OSS_KERNELS=1 (or "
                "GPUSTACK_AMD_MLA_KERNEL=1 for the 192/128 MLA expand "
                "shape) to opt in")
        if tiles is None or tiles[0] is None:
            tiles = build_prefill_tiles(seq_lens, q.device, PREFILL_ROWS)
        hip.flash_prefill(out, q, k, v, tiles[0], tiles[1], tiles[2], scale,
                          sinks=_sinks_f32(sinks), window=window,
                          softcap=softcap)
    else:
        torch_ref.varlen_prefill_attn(out, q, k, v, seq_lens, scale,
                                      sinks=sinks, window=window,
                                      softcap=softcap)


def build_paged_prefill_tiles(seq_starts: list[int], seq_hists: list[int],
                              seq_news: list[int], device,
                              rows: int = _PREFILL_BQ):
    """Map per-seq suffix rows to q tiles of `rows` (64 or PREFILL_ROWS) for
    the paged prefill-with-history kernel (one entry set per (seq, q-tile))."""
    return tuple(to_device([(a, torch.int32) for a in paged_prefill_tile_rows(
        seq_starts, seq_hists, seq_news, rows)], device))


def paged_prefill_tile_rows(seq_starts: list[int], seq_hists: list[int],
                            seq_news: list[int], rows: int = _PREFILL_BQ):
    """The lists of build_paged_prefill_tiles: each tile's sequence's first
    row, its own first row there, cached tokens, new rows, sequence."""
    qstart, q0s, hists, news, seqi = [], [], [], [], []
    for i, (st, h, n) in enumerate(zip(seq_starts, seq_hists, seq_news)):
        for q0 in range(0, n, rows):
            qstart.append(st)
            q0s.append(q0)
            hists.append(h)
            news.append(n)
            seqi.append(i)
    return qstart, q0s, hists, news, seqi


def paged_prefill_attn(out, q, k_cache, v_cache, block_tables,
                       seq_starts: list[int], seq_hists: list[int],
                       seq_news: list[int], scale: float, tiles=None,
                       sinks=None, window: int = 0,
                       softcap: float = 0.0) -> None:
    """Prefill-with-history: suffix/chunk rows attend to cached paged KV +
    their own freshly written positions through the MFMA flash kernel
    (removes the r1-measured ~3.5x paged-decode-row penalty)."""
    hip = _backend(q)
    if hip is not None:
        if (sinks is not None or window or softcap or q.shape[-1] != 128) \
                and not _oss_kernels_enabled():
            raise NotImplementedError(
                "sinks/window/softcap/D!=128 CDNA4 paged-prefill kernel "
                "variants are unvalidated — set GPUSTACK_AMD_OSS_KERNELS=1 "
                "to opt in")
        if tiles is None:
            tiles = build_paged_prefill_tiles(seq_starts, seq_hists,
                                              seq_news, q.device,
                                              PREFILL_ROWS)
        hip.flash_prefill_paged(out, q, k_cache, v_cache, block_tables,
                                tiles[0], tiles[1], tiles[2], tiles[3],
                                tiles[4], scale, sinks=_sinks_f32(sinks),
                                window=window, softcap=softcap)
    else:
        torch_ref.paged_prefill_attn(out, q, k_cache, v_cache, block_tables,
                                     seq_starts, seq_hists, seq_news, scale,
                                     sinks=sinks, window=window,
                                     softcap=softcap)


def gemm8(x, w, out=None, safe: bool = False):
    """8-phase pipelined 256x256 MFMA GEMM: out[M,N] = x[M,K] @ w[N,K]^T
    (bf16, f32 accumulate). GPU-only; requires N%256==0, K%128==0 —
    falls back to F.linear otherwise. `safe=True` runs the fully-drained
    variant (race isolation for tests)."""
    import torch.nn.functional as F

    M, K = x.shape
    N = w.shape[0]
    if not x.is_cuda or N % 256 != 0 or K % 128 != 0:
        return F.linear(x, w, None)
    if out is None:
        out = torch.empty(M, N, dtype=x.dtype, device=x.device)
    hip = _backend(x)
    if hip is None:
        return F.linear(x, w, None)
    hip.gemm8(out, x.contiguous(), w, 1 if safe else 0)
    return out


def skinny_gemm(x, w, out=None, splitk: int | None = None, version: int = 1):
    """Split-K decode GEMM: out[M,N] = x[M,K] @ w[N,K]^T (bf16, f32 acc).
    GPU-only (falls back to F.linear elsewhere or for unsupported shapes)."""
    import torch.nn.functional as F

    M, K = x.shape
    N = w.shape[0]
    if not x.is_cuda or N % 128 != 0 or K % 64 != 0:
        return F.linear(x, w, None)
    if splitk is None:
        mt = (M + 255) // 256
        nt = N // 128
        splitk = 1
        while (mt * nt * splitk < 400 and splitk < 8
               and K % (64 * splitk * 2) == 0):
            splitk *= 2
    if out is None:
        out = torch.empty(M, N, dtype=x.dtype, device=x.device)
    ws = None
    if splitk > 1:
        ws = torch.empty(splitk * M * N, dtype=torch.float32, device=x.device)
    _load_hip().skinny_gemm(out, x, w, ws, splitk, version)
    return out


def _rows_gemm_wins(M: int, N: int, K: int) -> bool:
    """Where the decode product (ops/csrc/rows_gemm.hip) measured faster than
    the library, us at 1 / 8 / 16 rows, weights out of HBM:
    small weights, whose time is latency: 4096x4096 9.5 / 10.1 / 10.7 against
    15.6, 2048x4096 8.5 / 9.6 / 10.8 against 14.8, 5120x2048 8.0 / 9.0 / 10.6
    against 12.3 (24 rows of 4096x4096: 12.9 against 13.4; 6144x4096 13.0 /
    15.6 / 18.3 against 14.6);
    many columns (22016x4096 36 / 39 / 41 against 52 and 28672x4096 43 / 47 / 53
    against 54, where the tiled product is better still): 16384x2048 14 / 15 /
    16 against 18, 49152x2048 34 / 37 / 42 against 47, 65536x4096 88 / 93
    against 120 (49152x3072 at 16 rows 65 against 60, 16384x5120 34 / 37 / 42
    against 34);
    wide heads of narrow models: 102400x1536 71 / 77 / 80 against 115,
    151936x2048 127 / 135 / 144 against 205, 200064x2560 220 / 236 / 260
    against 325 (128256x3072 135 / 150 / 173 against 146, 102400x1024 50 / 52 /
    53 against 42)."""
    if M > 16 or K % 128 != 0 or not 1024 <= K <= 4096:
        return False
    if N >= 100000:
        return 1536 <= K <= 2560
    return N * K <= 17 << 20 or (
        N >= 12288 and N * K <= (280_000_000 if M <= 8 else 130_000_000))


def _rows_tile_plan(M: int, N: int, K: int):
    """(columns of a tile, parts of K) where the tiled product of up to 512
    rows (rows_tile_kernel in ops/csrc/rows_gemm.hip) measured fastest, else
    None. Above 128 rows _tall_tile_plan has the rule. The split aims at one workgroup a CU (256); us against the library,
    or up to 16 rows against the better of it and the decode product, weights
    out of HBM:
    up to 10240 columns, 48 rows: 4096x14336 26.0 / 36.3, 4096x4096 11.8 / 13.8,
    5120x2048 10.7 / 12.9, 3072x8192 15.3 / 21.7; 96 rows: 4096x14336 30.1 / 50.1,
    4096x4096 14.9 / 17.1; but 8192x4096 18.5 / 18.1 and 2048x4096 at 96 rows
    13.5 / 12.8;
    more columns, where the library loses on rows a multiple of 4 KB apart:
    28672x4096 41.2 / 50.7 at 48 rows and 45.7 / 57.5 at 96, 128256x4096
    182 / 254, 16384x2048 15.7 / 18.0, 65536x6144 144 / 178, 28672x8192
    85 / 129, but 51200x3072 72 / 62, 40960x5120 97 / 91, 22016x2560 31 / 30
    (18944 columns make 296 tiles, two for some CUs and one for most: 31 / 27
    at 2560), and a fourth or fifth round of tiles of long rows (49152x8192
    137 / 149, 57344x8192 172 / 161, 69632x8192 230 / 224, 86016x8192 249 / 295;
    57344x6144 142 / 147).
    At 96 rows: 16384x2048 18.3 / 18.8, 16384x4096 32 / 35, 65536x2048 60 / 70,
    65536x4096 99 / 129, 51200x6144 137 / 147, 22016x8192 82 / 82, 128256x8192
    372 / 416; rows of 5120, 3072 and 2560 lose (51200 of each: 121 / 104,
    73 / 68, 65 / 58), so do longer ones (51200x10240 224 / 200, 102400x12288 at
    112 rows 557 / 504) and 12288x4096 33 / 30. Tiles of 128 columns fill the
    256 CUs in rounds, and one that is not nearly full loses on rows of more
    than 4096 (73728x8192 302 / 279, 77824x6144 250 / 237, 143360x8192 at 80
    rows 477 / 428), above 96 rows on rows of 4096 too, where it is the second
    or third (at 128: 36864x4096 84 / 75, 77824x4096 166 / 153, 40960x8192
    160 / 154).
    up to 16 rows: 28672x4096 40 / 43 at one and 41 / 53 at 16, 4096x11008
    17 / 31, 22016x4096 32 / 39, 128256x4096 175 / 178, but 16384x4096 at one
    row 27 / 26."""
    if not 0 < M <= 512 or K % 64 != 0 or N % 8 != 0 or min(N, K) < 1024:
        return None
    if M > 128:
        return _tall_tile_plan(M, N, K)
    t64, t128 = -(-N // 64), -(-N // 128)
    if N > 10240:
        wide = 160 <= t128 <= 256 or t128 >= 500 or M > 64 and t128 > 256
        if 256 < t64 < 400 and not wide:
            return None
        if M <= 16:
            wins = (N <= 32768 and K >= 2560 and (
                M > 4 or N >= 22016 or K >= 11008)
                or N >= 100000 and K >= 3072)
        elif M <= 64:
            wins = K % 2048 == 0 and (K <= 8192 or N <= 32768) and not (
                K > 6144 and 768 < t64 <= 1280)
        else:
            wins = K % 2048 == 0 and K <= 8192 and N >= 16384 and not (
                M > 96 and (K > 4096 and 256 < t128 < 500 or K > 2048 and (
                    256 < t128 < 300 or 512 < t128 < 768))
                or K > 4096 and (512 < t128 < 768 or 1024 < t128 < 1280))
        plan = (128 if wide else 64), 1
    elif K <= 2048:
        wins = 16 < M <= 64 and (K == 1024 and N >= 2560
                                 or 5120 <= N <= 8192)
        plan = 32, 1
    else:
        if M <= 16:
            wins = K >= 11008 or N > 8448
        elif M <= 64:
            wins = K >= 11008 or K >= 4096 and not 6144 < N <= 8448
        else:
            wins = N >= 3072 <= K or N >= 2048 and K >= 7168
        parts = min(8, 256 // t64)
        if t64 <= 24:
            plan = 32, 8
        elif parts * t64 >= 216 or parts == 8:
            plan = 64, parts
        else:
            plan = 128, 256 // t128
    return plan if wins else None


def _tall_tile_plan(M: int, N: int, K: int):
    """_rows_tile_plan for 129 to 512 rows: long rows of up to 10240 columns,
    which leave the library's tiles few and its chip idle; more row tiles leave
    it less so, and the lines come down with their number. Cut over k into as
    many parts as two workgroups a CU take, at most 8 (4096x14336 at 256 rows:
    four parts 45 without their join, eight 39), and into 5 or 7 nowhere: the 8
    XCDs take workgroups in turn, so that an odd number of parts brings all of x
    to each of their L2s, an even one half of it or less (176 rows of 4608x9216
    in 7 parts 48, in 6 37; 240 of 5632x11008 in 5 78, in 4 54; 384 of
    4096x11008 66, 54; but 136 of 6144x8192 39, 43). us against the library,
    with the join, weights out of HBM:
    160 rows: 4096x14336 42 / 82, 4608x9216 36 / 57, 5120x5120 26 / 36; 176
    rows: 4608x9216 37 / 41, 2560x6144 22.4 / 22.5, 8192x5120 36 / 34 (x4096 34 /
    28); 256 rows: 4096x14336 48 / 61, 6144x12288 63 / 110, 1032x6144 17 / 22,
    2048x6144 20 / 23, but 10240x10240 100 / 89; 384 rows: 5120x14336 71 / 88,
    4096x11008 54 / 63, 2560x6144 27 / 28; 512 rows: 4096x14336 71 / 82,
    4096x6144 38 / 43, 3072x7168 40 / 42, but 5120x11008 97 / 93. The library is
    uneven in M: between 4608 and 5120 columns it is up to a tenth the faster one
    at 136 to 152 and at 168 to 184 rows (184 rows of 4864x8192 43 / 36), and half
    as fast as the tiles at 160 and from 192 on (192 of 5120x8192 .62)."""
    rows = -(-M // 128)
    if N > (10240, 5120, 4096)[rows - 2] \
            or K < (5120 if rows == 2 and N >= 3072 else 6144):
        return None
    t128 = rows * -(-N // 128)
    if t128 < 32:
        return 64, 8
    parts = min(8, 512 // t128)
    return 128, parts - parts % 2 if parts > 4 else parts


def _parts_plan(M: int, N: int, K: int):
    """(columns of a tile, parts of K) of a small product whose consumer adds
    the parts up, where that beats the product of _rows_tile_plan, the library
    or the decode product, else None: short rows leave whole tiles few and
    their chain long. us with an RMS norm behind, parts against the best of the
    others.
    Up to 16 rows, against the decode product (which wants k in 128s, and whose
    workgroups of 16 columns fill the chip from 2049 to 4096 of these) from 3072
    k there and from 2048 k elsewhere: at one row 2048x2048 7.7 / 7.8, 2048x3072
    8.6 / 9.6, 4608x2048 10.8 / 11.8, but 4096x3072 11.2 / 10.9; at 16 rows 8.1 /
    9.3, -, 11.4 / 14.3, 11.5 / 12.2; 4096x2048 at 8 rows 10.4 / 9.7. Where only
    the library is beside it, at any k: 3072x1088 at 8 rows 8.1 / 12.5, 2048x5120
    at one 11 / 21, 4096x5120 14 / 23, 1024x8192 10 / 15, 6144x4096 17 / 20,
    4096x8192 19.4 / 20.8, 8192x3072 at 16 rows 17 / 24, and about even on 5632
    to 7168 columns of 8192 k (28 / 29 at one row, 31 / 30 at 16).
    More rows: up to 4096 columns at any k, beyond from where whole tiles of 32
    columns stop (2048 k): 24 rows of 2048x2048 8.2 / 14.0, 3072x1024 8.3 / 8.6,
    6144x2112 13.4 / 19.5, but 6144x2048 12.9 / 12.5; 64 rows of 3072x1024 9.6 /
    9.9, x1088 9.7 / 14.9, 4096x2048 12.2 / 15.9, but 4608x1024 12.2 / 10.8; 128
    rows of 2048x2048 12.3 / 14.5. Above 64 rows _rows_tile_plan cuts rows from
    3072 k on itself, from as many columns (128 rows of 2560x3072 16 / 24), and
    up to 64 rows those from 4096 k on, up to 6144 columns (64 rows of 7168x10240
    38 / 49)."""
    if not 0 < M <= 128 or K % 64 != 0 or N % 8 != 0 or min(N, K) < 1024 \
            or N > 8192 or K >= 11008:
        return None
    if M <= 16:
        wins = K >= (3072 if 2048 < N <= 4096 else 2048) \
            or not _rows_gemm_wins(M, N, K)
    elif K >= 4096:
        wins = N > 6144 and M <= 64
    elif M > 64 and K >= 3072:
        wins = N < 3072
    else:
        wins = N <= 4096 or K > 2048
    if not wins:
        return None
    if M <= 16 and K >= 4096 and N <= 5120:
        # long rows: as many parts as leave one workgroup a CU. Cuts of 4 KB
        # meet on few memory channels, the more workgroups the more (3 / 4
        # parts at 8192 k: 4096 columns .91, 3840 .96, 3584 1.03, 3072 1.13)
        if N <= 2048:
            return 32, min(8, 256 // -(-N // 32))
        if K % 8192 == 0 and N > 3584:
            return 64, 3
        return 64, min(4, 256 // -(-N // 64))
    if N <= 4096:
        return 32 if N <= 2048 else 64, 4
    # the same for four cuts of rows a multiple of 8 KB apart (8192 columns: .88
    # at 4096 k, .77 at 8192, but 1.02 at 4032 and 1.0 at 8320)
    return 128, 3 if K % 4096 == 0 else 4


def router_plan(T: int, E: int, H: int):
    """(columns of a tile, parts over k) of a router's product, whose parts the
    choice of the experts adds up, or None. us for both launches against a
    cast, an fp32 library product and the choice, at 64 / 1024 / 4188 / 16384
    rows: 64 experts of 2048 8.1 / 9.8 / 14.5 / 26 against 12 / 17 / 36 / 77, 128
    of 2048 8.5 / 11 / 18 / 34 against 14 / 20 / 53 / 115, 256 of 4096 12 / 17 / 30 / 73
    against 13 / 30 / 102 / 297; 512 of 2048 (with a choice that took 4 more) 22 / 27 / 37 /
    102 against 23 / 39 / 96 / 311, but at 128 rows 25 against 24. Eight parts of narrow
    tiles fill the chip for few rows (32 experts of 4096, eight / four parts: 64 rows 7.8
    / 9.4, 8000 19.7 / 22.3; 64 of 2048 8.1 / 8.6, 2000 rows 11.4 / 11.8; 128 of 2048 at
    1024 11.3 / 12.2, but 2000 14.8 / 13.5, 256 of 4096 at 64 14.0 / 11.6); later the
    parts' own traffic counts (4188 rows of 64 experts 64 x 4 14.5, 32 x 4 16.5; of 128
    64 x 2 17.7, 32 x 4 19.4, 128 x 2 21.7; of 256 128 x 4 30, 128 x 2 34), and one
    is the best of 256 experts at 16384 (73, two 82)."""
    if E % 4 != 0 or H % 64 != 0 or H < 1024 or E > 512 or T == 0:
        return None
    if E > 256:
        if 64 < T < 256:
            return None
        return (64, 2) if T <= 2048 else (128, 2)
    if E <= 32:
        return 32, 8
    if E <= 64:
        return (32, 8) if T <= 2500 else (64, 4) if T <= 12000 else (64, 2)
    if E <= 128:
        return (32, 8) if T <= 1400 else (32, 4) if T <= 2500 \
            else (64, 2) if T <= 6000 else (128, 2)
    return (32, 4) if T <= 2500 else (128, 4) if T <= 6000 \
        else (128, 2) if T <= 12000 else (128, 1)


def choose_sorts(T: int, E: int) -> bool:
    """True where the choice of the experts sorts the assignments too (moe_choose): one
    workgroup's work up to 8 rows, of up to 64 experts 16. us, two launches against one:
    128 experts 8 rows 7.1 / 5.7, 16 rows 7.0 / 7.0, 256 8 rows 7.4 / 7.1, 16 rows 7.5 /
    8.6; 64 16 rows 6.4 / 5.7, 24 rows 6.4 / 6.6 (moe_gemm.hip)."""
    return 0 < T <= (16 if E <= 64 else 8) and E <= 256


def moe_few_wins(rows: int, E: int, K: int, down: bool) -> bool:
    """Whether an expert product of `rows` assignments takes 16 rows at a time straight
    from memory (moe_few) in the place of tiles of 128 x 128 (moe_tile): the first product
    up to 4 rows an expert, the second up to 768 k to 4 where its blocks of 64 k are the same
    for the four waves, else to 2, to one of rows beyond 3072, else to 3/4. More than 16 rows of an expert read its weights again, so the lines
    allow for uneven routing. us, tiles / this, E experts of N x K, even routing: first, 128
    of 768 x 2048 8 assignments 22.1 / 13.5, 64 71 / 56, 256 128 / 116, 512 142 / 133, 768
    145 / 137, 64 of 1024 x 2048 128 101 / 79, 32 of 2048 x 1024 128 42.7 / 40.1, 256 43.5
    / 44.6, 8 of 14336 x 4096 16 303 / 263, 32 350 / 314; second, 128 of 2048 x 768 8 9.8 /
    7.4, 256 64 / 59, 512 72 / 70, 64 of 2048 x 1408 48 42 / 33, 384 64 / 66, 64 of 1024 x
    896 32 11.3 / 11.2, 64 15.4 / 16.0, 512 20.1 / 22.2, 16 of 4096 x 6400 16 106 / 90, 64
    140 / 142. Uneven, half of 64 rows to one of the experts and 114 of 128 with any, 768 x
    2048 512 134 / 127 and 2048 x 768 65.8 / 66.0; 96 rows of them, 68 to one,
    140 / 142 and 70.7 / 75.6. The second at 2 / 3 / 4 rows an expert by k, of the tiles' time:
    128 of 2048 columns 512 .83 / .90 / .93, 640 .88 / .98 / 1.03, 704 .85 / .93 / .97, 768 .85 /
    .92 / .95, 832 .93 / .96 / .99, 896 .89 / .96 / .98, 1024 .98 / 1.0 / 1.02; 64 of 1024 512
    .92 / 1.05 / 1.07, 640 1.02 / 1.05 / 1.10, 704 1.02 / 1.03 / 1.07, 768 .95 / .97 / .98, 832
    1.03 / 1.06 / 1.05, 1024 1.02 / 1.09 / 1.10; beyond 768 k what is left at 1 row is .73 to .95,
    at 3/4 .67 to 1.02."""
    if rows <= 0:
        return False
    if not down:
        return rows <= 4 * E
    if K <= 768:
        return rows <= (4 if K % 256 == 0 else 2) * E
    return rows <= E if K > 3072 else 4 * rows <= 3 * E


def moe_wide_wins(rows: int, E: int, N: int, K: int, down: bool) -> bool:
    """Where an expert product of `rows` assignments in tiles of up to 320 rows
    (ops/csrc/moe_wide.hip) measured faster than tiles of 128 (moe_gemm.hip). From
    128 rows an expert, where these begin to read its weights twice, and where its
    256 workgroups' rounds are filled, but for one round, or rows that fill the
    tiles. us, 128-row tiles / this, first and second product: 128 experts of 2048
    x 768 at 112 rows each 172 / 169 + 106 / 113, 128 198 / 173 + 119 / 116, 256
    283 / 209 + 176 / 149, 340 (two tiles for each) 340 / 296 + 209 / 194, 800
    721 / 539 + 434 / 383; 8 of 4096 x 14336 at 128 492 / 387 + 301 / 246, at 320,
    two rounds of .69, 748 / 624 + 413 / 516: the second stays. Of 108 pairs of
    products from 128 to 800 rows an expert, of ten models' sizes, 99 and 95 are
    taken, none of them slower by more than 3 %; with routing drawn even, by
    (e + 1)^-1/2 or (e + 1)^-1, of 260 products 10, all of the last two, to 1.09 (64
    experts, 1508 rows by eight, 94 / 103), .85 on average."""
    if E < 1 or E > 256 or rows < 128 * E or K % 64 != 0 or K < 192 or N % 8 != 0 \
            or rows >= 1 << 30:
        return False
    # offsets of 32 bits of bytes
    if ((1 if down else 2) * N + 192) * K >= (1 << 31) - (1 << 19) \
            or rows * (N if down else K) >= (1 << 31) - (1 << 19) \
            or 320 * max(N, K) >= (1 << 31) - (1 << 19):
        return False
    mean = rows // E
    parts = -(-(mean + math.isqrt(mean)) // 320)   # some experts have more rows
    tiles = E * parts * -(-N // (192 if down else 96))
    rounds = -(-tiles // 256)
    return rounds == 1 or tiles >= .8 * 256 * rounds or mean >= 240 * parts


# us of rows_tile_kernel's whole products by tile of 32, 64 and 128 columns, and of
# rows_gemm_kernel (0), for up to so many rows: a launch, and for every 64 k (r: workgroups
# by 256) with one workgroup a CU the second and r^3 times the third, with more the fourth,
# r times the fifth and ceil(r / 2) times the sixth; of rows_gemm_kernel the second and r
# times the third where its workgroups have 16 columns, the fourth and r times the fifth
# where they have 32. Fitted to 3000 sizes of 1024 to 4096 k, weights out of HBM (3 to 6 %
# off on average, 25 at most).
_FEW_TIMES = {
    8: {32: (2.41, .157, .043, .055, .133, .081), 64: (2.04, .271, .104, .088, .262, .159), 128: (2.08, .358, .476, .134, .546, .285), 0: (2.01, .045, .095, .066, .178, 0)},
    16: {32: (2.42, .157, .043, .046, .146, .081), 64: (2.11, .272, .102, .073, .275, .167), 128: (2.1, .375, .458, .118, .563, .311), 0: (2.06, .05, .123, .05, .21, 0)},
    32: {32: (2.42, .162, .048, .04, .163, .083), 64: (2.23, .274, .108, .063, .295, .165), 128: (2.22, .399, .439, .089, .563, .364)},
    64: {32: (2.33, .246, .037, .067, .181, .133), 64: (2.52, .306, .107, .057, .331, .177), 128: (2.87, .484, .344, .055, .564, .455)},
}


def _few_time(rows: int, cols: int, N: int, K: int) -> float:
    base, one, full, two, each, pair = _FEW_TIMES[rows][cols]
    steps = K / 64
    if cols == 0:
        narrow = N // 32 < 512
        r = -(-N // (16 if narrow else 32)) / 256
        return base + steps * (one + r * full if narrow else two + r * each)
    r = -(-N // cols) / 256
    return base + steps * (one + r ** 3 * full if r <= 1 else
                           two + r * each + math.ceil(r / 2) * pair)


@functools.lru_cache(maxsize=4096)
def _few_rows_plan(M: int, N: int, K: int, plan, rows: bool):
    """(tile plan, whether rows_gemm) of a whole product of up to 64 rows of 1024 to 4096
    k, given what _rows_tile_plan and _rows_gemm_wins say: the form of the least time
    (_few_time), where it is 8 % less than that of theirs; in the library's place one of
    the two, but beyond 16 rows only where it is no more than the library takes at its
    best (8 us, below 3072 columns 6, and 5.4 TB/s), and neither up to 8192 columns of 4096
    k. Of 2233 sizes up to 64 rows (8 us everywhere) these take 1.024 of the time of the
    best form, the two rules alone 1.114; 41 more than with the two rules by over 4 %. us: 16 rows of 151936 x 2048 130 -> 117, 8 of 10304 x 2048 14.7 -> 12.5, 16 of 8192 x
    2048 11.0 -> 8.3, 16 of 102400 x 1536 71 -> 63, 32 of 14336 x 1024 21.4 -> 7.7.
    Of 620 sizes of 17 to 64 rows of 1024 to 3968 k that the two rules leave to the library
    439 are taken, .867 of the time on average, 20 more by over 3 %, to 1.09 (64 rows of
    27648 x 2560). Below 3072 columns up to 96 of the 256 CUs have a tile, and the library
    cuts k: with 8 us there 41 took more, to 1.26 (32 of 1536 x 2816 7.4 / 9.3).
    Of 4096 k the library has numbers that it has not of 4032 (library / tiles of 32 at 1, 8,
    16, 32, 64 rows: 8192 columns of 4096 17.1 / 17.8, 17.2 / 17.7, 17.1 / 17.4, 17.6 / 17.1,
    20.1 / 21.0; of 4032 20.3 / 14.1, 20.5 / 14.0, 20.5 / 14.2, 23.0 / 15.3, 29.1 / 21.9), and
    the tiles' rows lie a power of two apart; of 6144 columns the tiles would take 13.4 to
    14.2 for 14.3 to 15.3 up to 32 rows, 19.0 for 17.9 at 64; beyond, 9216, 23.5 for 26.0."""
    if not (0 < M <= 64 and 1024 <= K <= 4096 and N >= 1024) or K % 64 or N % 8 \
            or plan and plan[1] > 1:
        return plan, rows
    upto = next(m for m in _FEW_TIMES if m >= M)
    forms = [c for c in _FEW_TIMES[upto] if c or K % 128 == 0]
    time = {c: _few_time(upto, c, N, K) for c in forms}
    best = min(time, key=time.get)
    now = plan[0] if plan else 0 if rows else None
    if now is None:
        if N <= 8192 and K == 4096 \
                or M > 16 and time[best] > (8 if N >= 3072 else 6) + 2e-6 * N * K / 5.4:
            return plan, rows
    elif time[best] >= .92 * time[now]:
        return plan, rows
    return ((best, 1), False) if best else (None, True)


def linear_auto(x, w, parts: bool = False):
    """Shape-gated GEMM dispatch: the products for few rows
    (_rows_tile_plan, _rows_gemm_wins, _few_rows_plan) and for many
    (_wide_parts_plan, _wide_rows_tile), the split-K skinny kernel where it
    measured faster than hipBLASLt (scripts/bench_skinny_gemm.py on MI355X:
    down_proj-like N=4096 K>=8192 M>=384 at splitk=4, 824 TF vs hipBLASLt 680),
    F.linear everywhere else. `parts`: a product that is cut over k may come
    as its fp32 parts [n, M, N], for a consumer that adds them up itself
    (add_rms_norm, qkv_store, add_layer_norm) and saves the join's launch."""
    import torch.nn.functional as F

    if _own_products(x, w):
        M, K = x.shape
        N = w.shape[0]
        wide = _wide_parts_plan(M, N, K) if parts else None
        if wide and _wide_take(x, w):
            return _load_hip().wide_parts(x, w, wide[1], *wide[0])
        plan = parts and _parts_plan(M, N, K) or _rows_tile_plan(M, N, K)
        plan, rows = _few_rows_plan(M, N, K, plan, _rows_gemm_wins(M, N, K))
        wide = None if parts and plan and plan[1] > 1 else _wide_rows_tile(M, N, K)
        if wide and _wide_take(x, w):
            out = torch.empty(M, N, dtype=x.dtype, device=x.device)
            _load_hip().wide_rows(out, x, w, *wide)
            return out
        if (plan or rows) and _rows_take(x, w):
            if parts and plan and plan[1] > 1:
                return _load_hip().rows_tile_parts(x, w, *plan)
            out = torch.empty(M, N, dtype=x.dtype, device=x.device)
            if plan:
                _load_hip().rows_tile(out, x, w, *plan)
            else:
                _load_hip().rows_gemm(out, x, w)
            return out
        if (N == 4096 and K >= 8192 and 384 <= M <= 1024
                and K % 256 == 0 and _products() is not None
                and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
                and x.is_contiguous() and w.is_contiguous()):
            return skinny_gemm(x, w, splitk=4)
    return F.linear(x, w)


def _own_products(x, w) -> bool:
    import os

    return (x.is_cuda and x.dim() == 2 and w.dim() == 2
            and os.environ.get("GPUSTACK_AMD_SKINNY_GEMM", "1") == "1")


def _rows_take(x, w) -> bool:
    """Operands that the products for few rows take."""
    return (x.shape[0] > 0 and _products() is not None
            and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and w.is_contiguous() and w.data_ptr() % 16 == 0
            and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0
            and not (x.requires_grad or w.requires_grad))


def _wide_take(x, w) -> bool:
    """Operands that the products of many rows take: _rows_take, and offsets inside
    a tile's rows within 32 bits of bytes."""
    return x.stride(0) <= 1 << 22 and _rows_take(x, w)


def _silu_plan(M: int, N: int, K: int):
    """_rows_tile_plan of a product of N columns, gate and up, that ends in the
    activation, else None. Tiles of 64 columns bring 32 rows of each, which for
    most widths take longer to come than 64 neighbours where rows are 8 KB (4096
    k) apart. us with the activation behind / in it, 16 rows: 16384x4096 29.7 /
    37.4, 12288x4096 25.3 / 27.9, 48 rows of 36864x4096 73 / 85 (11264 and 14336
    columns would gain 5 to 8 %); other lengths gain at every width (in it / behind
    at 48 rows: 16384x2048 .77, x6144 .92, x8192 .96)."""
    plan = _rows_tile_plan(M, N, K)
    if not plan or plan[1] > 1 or plan[0] < 64 or N % 8 != 0 \
            or plan[0] == 64 and K == 4096:
        return None
    return plan


# Tiles of wide_kernel (ops/csrc/wide_tiles.hip), in 32 rows and 32 weight rows: us of
# a round's end, of a round's step of 64 k, and what a step takes more where all 256
# workgroups have a tile (the card's power). Fitted to 6600 sizes, off by 4 % of a time
# on average (8 x 8) to 9 % (4 x 2); the tile of the least time by them costs .6 % more
# than the best of them with the activation and 1.4 % without.
_WIDE_TILES = {
    (8, 8): (5.7, .92, .43), (8, 7): (6.2, .82, .37), (8, 6): (4.4, .73, .31),
    (8, 5): (3.9, .67, .24), (8, 4): (3.1, .56, .22), (6, 8): (4.2, .77, .29),
    (6, 6): (3.4, .65, .20), (4, 6): (2.1, .51, .17), (4, 4): (1.3, .38, .15),
    (4, 2): (.4, .26, .10)}
_WIDE_SILU = ((8, 8), (8, 7), (8, 6), (8, 5), (8, 4), (6, 8))
_WIDE_ROWS = ((8, 8), (8, 7), (8, 6), (8, 4), (6, 8), (6, 6), (4, 6), (4, 4), (4, 2))
_WIDE_PARTS = ((8, 8), (8, 6), (8, 4), (6, 8), (6, 6), (4, 6), (4, 4))


def _wide_time(M: int, N: int, K: int, tile, parts: int = 1) -> float:
    end, step, full = _WIDE_TILES[tile]
    n = -(-M // (32 * tile[0])) * -(-N // (32 * tile[1])) * parts
    rounds = -(-n // 256)
    return 2 + end * rounds + math.ceil(K / 64 / parts) * (step * rounds + full * n / 256)


def _wide_tile(M: int, N: int, K: int, tiles, base: float, products: float,
               host: float):
    """The tile of the least time for N weight rows, where that is no more than the
    library takes for its fixed part, `base`, its bytes at 6 TB/s and its products (the
    root of their squares), else None.
    Short products wait for the host where the step is not captured: a call of the library
    costs it 18 to 20 us, one of these 7, and a step of a few hundred rows is such calls (a
    prompt of 312 rows in the hybrid stack 847 us with the library's products of 2048 k,
    754 with these). Their fixed part is `host`, up to 5 us more as _wide_time has them,
    which is 1.2 to 1.45 below their times. Captured steps take the same kernels as their
    warm-up, though some take the device longer: 512 rows of 1536x2048 12.5 / 15.3."""
    if K % 64 != 0 or K < 128 or (N + 512) * K >= 1 << 31 \
            or N >= 1 << 21 or M * max(N, K) >= 1 << 40:
        return None

    time, best = min((_wide_time(M, N, K, tile), tile) for tile in tiles)
    moved = 2 * (N * K + M * (N + K)) / 6e6
    library = base + math.hypot(moved, products)
    short = host + min(5, math.hypot(moved, 2 * M * N * K / 1250e6))
    return best if time <= max(library, short) else None


@functools.lru_cache(maxsize=4096)
def _wide_silu_tile(M: int, N: int, K: int):
    """The tile of a product of many rows that ends in the activation, or None where
    the library's product and the activation behind it are as good; N columns, gate
    and up. Of 6668 drawn sizes that it takes by 11 (1024 to 30000 weight rows, 1024 to 15360 k,
    129 to 8192 rows, weights out of HBM) 63 are slower by more than 3 %, most beyond
    6912 k (256 rows of 19712x15104 the worst, 1.12), .80 of the other's time on average.
    Short ones, with 13 us for the library's fixed part and the activation's, are slower on
    the device as often as not, where both calls cost the host 25 (512 rows of 1280x1024
    11.8 / 15.1, 256 of 4096x1024 14.7 / 16.8). us,
    library and activation / this, 4096 k: 512 rows of 28672 108 / 93, 2039 411 / 337,
    8192 1422 / 1286; 512 of 22016 99 / 80; but 136 of 16384 columns and 3072 k are
    left, .91."""
    if N % 16 != 0 or M <= 128:
        return None
    return _wide_tile(M, N, K, _WIDE_SILU, 11, 2 * M * N * K / 1250e6, 13)


@functools.lru_cache(maxsize=4096)
def _wide_parts_plan(M: int, N: int, K: int):
    """(tile, parts over k) of a product of many rows whose consumer adds the parts up
    (wide_kernel in ops/csrc/wide_tiles.hip), or None. As many parts as let its 256
    workgroups have one tile each, at most 8 and each of 1024 k and more, or half as many:
    the tile and the parts of the least time with the parts' own bytes, where that is 3 %
    (up to 256 rows 5) less than a whole product's; both with the norm behind, which reads
    4 bytes a part and element. Not below 3584 k, where a part is hardly more than its
    start (3072 k, us with an RMS norm behind, before / so: 256 rows of 1024 columns 13.3 /
    17.4, of 2048 19.2 / 22.8), up to 512 rows of 2048 columns and fewer, which the
    library fills with small tiles, not below 5120 (256 of 1024x4096 15.2 / 18.0).
    Up to 512 rows it takes the place of _tall_tile_plan: of 2568 sizes of 1408 to 10240
    columns and 5120 to 28672 k .89 of its time on average, from .96 at 5120 k to .83 at
    28672, 38 of them slower by more than 3 %, most at 11008 and 16384 k (192 rows of
    8192x16384 the worst, 90 / 106); but of fewer columns a third loses (1024 1.02 on
    average, 1152 .96, 1280 .97, 1408 .88).
    us with the norm, weights out of HBM, before / so: 512 rows of 4096x4096 36 / 34, of
    6144x4096 49 / 42, of 4096x14336 73 / 66, 264 of 4096x14336 64 / 53, 136 of 4096x4096
    27 / 22, 640 of 4096x14336 143 / 84, 1024 159 / 107, 2039 217 / 197; but 1024 rows of
    4096x4096 47 / 48. Of 3026 drawn sizes that it takes (1024 to 10240 columns, to 15360
    k, 129 to 8192 rows) 31 are slower than before by more than 3 % (228 rows of 1024x5120
    the worst, 1.14), .83 of the time on average."""
    if M <= 128 or K < (5120 if M <= 512 and N <= 2048 else 3584) or K % 64 != 0 \
            or N % 8 != 0 or (N + 512) * K >= 1 << 31 or N >= 1 << 21 \
            or M <= 512 and N <= 1280 and _tall_tile_plan(M, N, K):
        return None
    out = M * N / 1e6
    best = None
    for tile in _WIDE_PARTS:
        n = -(-M // (32 * tile[0])) * -(-N // (32 * tile[1]))
        most = min(8, 256 // n, K // 1024)
        for parts in {most, -(-most // 2)}:
            if parts >= 2:
                plan = _wide_time(M, N, K, tile, parts) + parts * out, tile, parts
                best = min(best or plan, plan)
    behind = 10 + N * K / 20e6 + .85 * out
    whole = min(_wide_time(M, N, K, tile) for tile in _WIDE_ROWS) + .3 * out
    if best is None or best[0] + behind > (.97 if M > 256 else .95) * (whole + behind):
        return None
    return best[1:]


@functools.lru_cache(maxsize=4096)
def _wide_rows_tile(M: int, N: int, K: int):
    """The tile of a product of many rows, or None for the library. Whole tiles of 256
    x 256 that fill their rounds are the library's too, and as often slower (.84 to 1.2
    of its time): those are left to it, what fills smaller tiles better is taken.
    The library is uneven: its times spread by 14 % around any such sum, and rows and
    columns that its tiles divide are its fast ones. The sum is that of whole tiles of 128
    x 256, each with 192 k for its end, at 1250 TFLOP/s, and 6 us beside. (By M N K, and
    9 us, it lost more where products are longer than the library's call: 384 rows of
    3584x2560 18.4 / 23.3 us, library / this.) Of 7762 drawn sizes (1024 to 30000 columns,
    1024 to 15360 k, 257 to 8192 rows) 6390 are taken by that, 237 of them slower on the
    device by more than 3 %, 10 by more than 10, to 1.21, .87 of the library's time on
    average, and 257 short ones, 121 of them slower by more than 3 %, to 1.33;
    of a grid of numbers that its tiles divide 1539 of 1698, 107 and 7, to 1.12, .91 (5000
    rows of 4096x11008 355 / 380), and 42, 21 of them, to 1.23.
    us, weights out of HBM, before / this: 2039 rows of 6144x4096 99 / 89, of 4096x4096
    72 / 64, of 4096x14336 216 / 191; but 512 of 4096x2560 and long rows of few columns
    (384 rows of 3584x7168 35 / 47) are left."""
    if M <= 256 or N % 8 != 0:
        return None
    rows, columns = (M + 127) // 128 * 128, (N + 255) // 256 * 256
    tile = _wide_tile(M, N, K, _WIDE_ROWS, 6, 2 * rows * columns * (K + 192) / 1250e6, 9)
    return None if tile == (8, 8) else tile


def linear_silu(x, w):
    """silu(gate) * up of the product with w = [gate rows; up rows], or None
    where the activation is a launch of its own: the tiled product of up to
    128 rows (_rows_tile_plan), not cut over k, and the one of many rows
    (_wide_silu_tile) end in it."""
    if not _own_products(x, w):
        return None
    M, K = x.shape
    plan = _silu_plan(M, w.shape[0], K)
    wide = None if plan else _wide_silu_tile(M, w.shape[0], K)
    if not (plan or wide) or not (_wide_take if wide else _rows_take)(x, w):
        return None
    out = torch.empty(M, w.shape[0] // 2, dtype=x.dtype, device=x.device)
    if wide:
        _load_hip().wide_rows(out, x, w, *wide, silu=True)
    else:
        _load_hip().rows_tile(out, x, w, *plan, silu=True)
    return out


def mfma_probe(a, b):
    return _load_hip().mfma_probe(a, b)


build_cos_sin_cache = torch_ref.build_cos_sin_cache


# --- fp32-residual op family ------------------------------------------------
# Kernels for models that keep the residual stream, norms, attention scores
# and routers in fp32 (ModelSpec.fp32_residual): ops/csrc/resid32.hip and
# ops/csrc/latent_attn.hip, built into their own small extension so a
# checkout that serves only such a model compiles nothing else. Activations
# entering GEMMs are bf16 or fp32 (the engine dtype); every kernel is
# instantiated for both.

_LATENT = None
_PAGED = None


def _load_paged():
    """Load `_hip_paged.so` (row kernels of the pre/post-norm fp32 stream
    and paged rotary attention), compiling it in-tree first when no built
    library is there."""
    global _PAGED
    if _PAGED is not None:
        return _PAGED
    import importlib.util

    from .build import PAGED_SO_PATH, build_paged

    if not PAGED_SO_PATH.exists():
        build_paged()
    spec = importlib.util.spec_from_file_location(
        "gpustack_amd.ops._hip_paged", PAGED_SO_PATH)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    _PAGED = mod
    return mod


def _paged_backend(t: torch.Tensor):
    return _load_paged() if t.is_cuda else None


def _load_latent():
    """Load `_hip_latent.so`, compiling it in-tree first when no built
    library is there (a fresh checkout on a GPU box)."""
    global _LATENT
    if _LATENT is not None:
        return _LATENT
    import importlib.util

    from .build import LATENT_SO_PATH, build_latent

    if not LATENT_SO_PATH.exists():
        build_latent()
    spec = importlib.util.spec_from_file_location(
        "gpustack_amd.ops._hip_latent", LATENT_SO_PATH)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    _LATENT = mod
    return mod


def _lat_backend(t: torch.Tensor):
    return _load_latent() if t.is_cuda else None


ACT_MODES = {"relu2": 0, "gelu": 1, "gelu_tanh": 2, "silu": 3, "tanh": 4}


def embed_pair_hash(x, h, tokens, prev, embed, pair_table, buckets: int,
                    mul_prev: int, mul_cur: int) -> None:
    k = _lat_backend(x)
    if k is not None:
        k.embed_pair_hash(x, h, tokens, prev, embed, pair_table,
                          buckets, mul_prev, mul_cur)
    else:
        torch_ref.embed_pair_hash(x, h, tokens, prev, embed, pair_table,
                                  buckets, mul_prev, mul_cur)


def rms_scale_add(x, a, weight, scale, eps: float, h) -> None:
    k = _lat_backend(x)
    if k is not None:
        k.rms_scale_add(x, a, weight, scale, eps, h)
    else:
        torch_ref.rms_scale_add(x, a, weight, scale, eps, h)


def rms_norm_f32(out, x, weight, eps: float) -> None:
    k = _lat_backend(x)
    if k is not None:
        k.rms_norm_f32(out, x, weight, eps)
    else:
        torch_ref.rms_norm_f32(out, x, weight, eps)


def latent_norm_store(cache, src, col0: int, weight, slots, eps: float) -> None:
    k = _lat_backend(src)
    if k is not None:
        k.latent_norm_store(cache, src, col0, weight, slots, eps)
    else:
        torch_ref.latent_norm_store(cache, src, col0, weight, slots, eps)


_LAT_GROUP = 16   # (row, head) pairs sharing one key stream per workgroup


def build_latent_tiles(seq_starts, seq_hists, seq_news, heads: int, device):
    """Group the batch's (row, head) pairs into tiles of at most 16 pairs
    that belong to ONE sequence, so a workgroup streams that sequence's
    latents once for all of them. Long portions tile as 16 rows x 1 head;
    short ones (decode rows above all) pack rows x heads. Returns int32
    [ntiles, 6]: row0, nrows, head0, nheads, seq, pos0."""
    import numpy as np

    G = _LAT_GROUP
    parts = []
    for i, (st, hist, new) in enumerate(zip(seq_starts, seq_hists, seq_news)):
        if new >= G:
            nh, nr = 1, G
        else:
            nh = min(heads, G)
            nr = max(1, min(new, G // nh))
        r0 = np.arange(0, new, nr, dtype=np.int32)
        h0 = np.arange(0, heads, nh, dtype=np.int32)
        rr, hh = np.meshgrid(r0, h0, indexing="ij")
        rr, hh = rr.reshape(-1), hh.reshape(-1)
        t = np.empty((rr.size, 6), dtype=np.int32)
        t[:, 0] = st + rr
        t[:, 1] = np.minimum(nr, new - rr)
        t[:, 2] = hh
        t[:, 3] = np.minimum(nh, heads - hh)
        t[:, 4] = i
        t[:, 5] = hist + rr
        parts.append(t)
    tiles = (np.concatenate(parts) if parts
             else np.empty((0, 6), dtype=np.int32))
    return to_device([(tiles, torch.int32)], device)[0]


def latent_attention_mfma_ok(cache) -> bool:
    """True when ops.latent_attention takes the MFMA kernel for this pool:
    bf16, both page planes, 16-token pages, width % 32 == 0 (<= 1024). Only
    then may q_lat / ctx be bf16 and arbitrarily strided."""
    return (cache.is_cuda and cache.dtype == torch.bfloat16
            and cache.shape[1] == 2 and cache.shape[2] == 16
            and cache.shape[3] % 32 == 0 and cache.shape[3] <= 1024)


def latent_attention(ctx, q_lat, cache, block_tables, row_seq, positions,
                     scale: float, tiles=None, exact: bool = False,
                     max_ctx: int = 0) -> None:
    """ctx / q_lat: [T, H, R] views (last axis contiguous). `exact` forces
    the fp32 vector-ALU kernel where the MFMA kernel would run. `max_ctx`
    (longest context in the batch, a host number) lets a batch of few tiles
    over long contexts split each tile's keys over several workgroups."""
    k = _lat_backend(q_lat)
    if k is not None:
        if tiles is None:
            raise ValueError("latent_attention on GPU needs the tile list "
                             "(build_latent_tiles)")
        nsplit = 1
        nt = tiles.shape[0]
        if not exact and max_ctx >= 512 and 0 < nt < 512:
            nsplit = max(1, min(16, 1024 // nt, max_ctx // 128))
        k.latent_attention(ctx, q_lat, cache, block_tables, tiles, positions,
                           scale, exact, nsplit)
    else:
        torch_ref.latent_attention(ctx, q_lat, cache, block_tables, row_seq,
                                   positions, scale)


def act_inplace(x, mode: str) -> None:
    # the kernel ships in both fp32-stream libraries: whichever is loaded
    k = _PAGED if (_PAGED is not None and x.is_cuda) else _lat_backend(x)
    if k is not None:
        k.act_inplace(x, ACT_MODES[mode])
    else:
        torch_ref.act_inplace(x, mode)


def route_grouped_topk(experts, weights, logits, n_experts: int, groups: int,
                       keep: int, scale: float) -> None:
    k = _lat_backend(logits)
    if k is not None:
        k.route_grouped_topk(experts, weights, logits, n_experts, groups,
                             keep, scale)
    else:
        torch_ref.route_grouped_topk(experts, weights, logits, n_experts,
                                     groups, keep, scale)


def moe_combine(out, y, inv, weights, shared, gate_logits, gate_col: int) -> None:
    k = _lat_backend(out)
    if k is not None:
        k.moe_combine(out, y, inv, weights, shared, gate_logits, gate_col)
    else:
        torch_ref.moe_combine(out, y, inv, weights, shared, gate_logits,
                              gate_col)


def grouped_ff_available(x, width: int, ff: int) -> bool:
    """The sync-free grouped expert kernels take bf16 on the GPU with
    width % 64 == 0 and ff % 64 == 0."""
    return (x.is_cuda and x.dtype == torch.bfloat16
            and width % 64 == 0 and ff % 64 == 0)


def grouped_up_act(u, x, up_w, s_tok, offs, counts, mode: str) -> None:
    """up_w [E, ff, W], or [E, 2 ff, W] (gate rows, then up rows) for the
    gated form."""
    _load_latent().grouped_up_act(u, x, up_w, s_tok, offs, counts,
                                  ACT_MODES[mode])


def grouped_down(y, u, down_w, offs, counts) -> None:
    _load_latent().grouped_down(y, u, down_w, offs, counts)


def softcap_(logits, cap: float) -> None:
    k = _lat_backend(logits)
    if k is not None:
        k.softcap(logits, cap)
    else:
        torch_ref.softcap_(logits, cap)


# --- pre/post-norm fp32 stream + paged rotary attention -------------------
# ops/csrc/rowmix32.hip and ops/csrc/ragged_attn.hip in `_hip_paged.so`.

def embed_rows_f32(x, tokens, embed) -> None:
    k = _paged_backend(x)
    if k is not None:
        k.embed_rows_f32(x, tokens, embed)
    else:
        torch_ref.embed_rows_f32(x, tokens, embed)


def rms_norm_rows(out, x, weight, eps: float) -> None:
    """fp32 rows -> weighted RMS norm in out's dtype."""
    k = _paged_backend(x)
    if k is not None:
        k.sandwich_add_norm(x, None, None, 0.0, eps, None, weight, out)
    else:
        torch_ref.rms_norm_f32(out, x, weight, eps)


def sandwich_add_norm(x, a, post_w, mult: float, eps: float, extra, next_w,
                      h, center: bool = False) -> None:
    """`center`: both norms are weight-only layer norms (the mean comes off
    first) instead of RMS norms."""
    k = _paged_backend(x)
    if k is not None:
        k.sandwich_add_norm(x, a, post_w, mult, eps, extra, next_w, h, center)
    else:
        torch_ref.sandwich_add_norm(x, a, post_w, mult, eps, extra, next_w, h,
                                    center)


def build_page_groups(seq_starts, seq_hists, seq_news, block_size: int,
                      device):
    """Runs of batch rows that fall into ONE cache page in order, for
    page-wise value stores: int32 [n, 2] = first row, rows. A sequence that
    brings rows for positions hist..hist+new-1 is cut at multiples of the
    page size."""
    import numpy as np

    parts = []
    for st, hist, new in zip(seq_starts, seq_hists, seq_news):
        first = np.arange(hist - hist % block_size, hist + new, block_size)
        lo = np.maximum(first, hist)
        hi = np.minimum(first + block_size, hist + new)
        parts.append(np.stack([st + lo - hist, hi - lo], axis=1))
    g = (np.concatenate(parts) if parts else np.empty((0, 2))).astype(np.int32)
    return to_device([(g, torch.int32)], device)[0]


def rotary_norm_store(q_out, qkv, nq: int, nk: int, q_norm_w, k_norm_w,
                      inv_freq, pos32, head_dim: int, k_cache, v_cache, slots,
                      eps: float, tied: bool, page_groups=None) -> None:
    """`page_groups` (build_page_groups; GPU, prompts): the value rows are
    written page by page instead of row by row."""
    k = _paged_backend(qkv)
    if k is not None:
        k.rotary_norm_store(q_out, qkv, nq, nk, q_norm_w, k_norm_w, inv_freq,
                            pos32, head_dim, k_cache, v_cache, slots, eps,
                            tied, page_groups)
    else:
        torch_ref.rotary_norm_store(q_out, qkv, nq, nk, q_norm_w, k_norm_w,
                                    inv_freq, pos32, head_dim, k_cache,
                                    v_cache, slots, eps, tied)


_ATT_GROUP = 16   # (row, score map) pairs sharing one key stream per workgroup


def build_attn_tiles(seq_starts, seq_hists, seq_news, heads: int,
                     kv_heads: int, maps: int, device):
    """Group the batch's (row, score map) pairs into tiles of at most 16
    pairs that share ONE key stream: same sequence, same kv head, same map.
    Long portions tile as 16 rows x 1 query head; short ones (decode rows
    above all) pack rows x the query heads of a kv group. Score map a =
    head * maps + map, so the heads of one kv group and one map are `maps`
    apart. Returns int32 [ntiles, 6]: row0, nrows, a0, n_a, seq, a_step."""
    import numpy as np

    G = _ATT_GROUP
    rep = heads // kv_heads
    parts = []
    for i, (st, hist, new) in enumerate(zip(seq_starts, seq_hists, seq_news)):
        if new >= G or rep == 1:
            nh, nr = 1, G
        else:
            nh = min(rep, G)
            nr = max(1, min(new, G // nh))
        r0 = np.arange(0, new, nr, dtype=np.int32)
        # first score map of every (kv head, chunk of nh heads, map)
        g0 = np.arange(0, rep, nh, dtype=np.int32)
        a0 = ((np.arange(kv_heads, dtype=np.int32)[:, None, None] * rep
               + g0[None, :, None]) * maps
              + np.arange(maps, dtype=np.int32)[None, None, :])
        na = np.broadcast_to(np.minimum(nh, rep - g0)[None, :, None],
                             a0.shape).reshape(-1)
        a0 = a0.reshape(-1)
        rr, ai = np.meshgrid(r0, np.arange(a0.size), indexing="ij")
        rr, ai = rr.reshape(-1), ai.reshape(-1)
        t = np.empty((rr.size, 6), dtype=np.int32)
        t[:, 0] = st + rr
        t[:, 1] = np.minimum(nr, new - rr)
        t[:, 2] = a0[ai]
        t[:, 3] = na[ai]
        t[:, 4] = i
        t[:, 5] = maps
        parts.append(t)
    tiles = (np.concatenate(parts) if parts
             else np.empty((0, 6), dtype=np.int32))
    return to_device([(tiles, torch.int32)], device)[0]


# Portions of at least this many rows go to the prompt kernel where it fits.
PROMPT_PORTION = 32


def prompt_kernel_wins(seq_news, max_ctx: int, heads: int, window: int) -> bool:
    """Where the prompt kernel is the faster one. Tiles of 16 rows are many
    workgroups that may cut a long walk over the keys into parts, tiles of 128
    few that read every key once, so the line is the number of 16-row tiles, three
    workgroups a CU; a whole prompt of up to 64 rows is one tile either way. us, 16-row
    tiles (paged_attn_waves_kernel) / prompt kernel, 16 heads on 4: one whole prompt of
    64 rows 8.6 / 8.6, 100 8.9 / 11.6, 300 11.9 / 15.7; 100 behind 200 11.4 / 18.1; 512
    rows (512 tiles) 16 / 23, behind 1000 35 / 54, behind 4000 90 / 133, behind 8000 162
    / 248, in a window of 1024 there 28 / 44; 2 x 300 (608) behind 8000 210 / 239; 700
    (704) behind 1000 49 / 57, behind 8000 237 / 248; 1000 rows (1008) behind 1000 69 /
    67, behind 8000 319 / 262; 200 (208) behind 4000 53 / 124. Of 940 batches (8 to 64
    heads, 32 to 2000 rows) 16 are on the wrong side by more than 3 %, to 1.22."""
    tiles = sum((n + 15) // 16 for n in seq_news if n >= PROMPT_PORTION) * heads
    span = min(max_ctx, window) if window > 0 else max_ctx
    return tiles >= 768 or tiles > 0 and span <= 64


def build_prompt_tiles(seq_starts, seq_hists, seq_news, device):
    """Tiles of PREFILL_ROWS rows of every portion of at least PROMPT_PORTION
    rows, int32 [5, ntiles]: the lists of paged_prefill_tile_rows."""
    lists = paged_prefill_tile_rows(
        seq_starts, seq_hists,
        [n if n >= PROMPT_PORTION else 0 for n in seq_news], PREFILL_ROWS)
    return to_device([([v for one in lists for v in one], torch.int32)],
                     device)[0].view(5, -1)


def prompt_attention_fits(q_dim: int, v_dim: int, maps: int, keep_first: int,
                          softcap: float, chunk: int, gate: bool, scale: float,
                          k_cache) -> bool:
    """What the prompt kernel of paged_attention takes: heads of 128 channels
    on values of 128 in bf16 pages of 16, one score map, a window, sinks and
    slopes, and no other option."""
    return (q_dim == 128 and v_dim == 128 and maps == 1 and keep_first == 0
            and softcap == 0 and chunk == 0 and not gate and scale > 0
            and k_cache.is_cuda and k_cache.dtype == torch.bfloat16
            and k_cache.shape[2] == 16)


@functools.lru_cache(maxsize=4096)
def _paged_wave_parts(nt: int, span: int) -> int:
    """Parts of `span` keys for `nt` tiles of paged_attn_waves_kernel, each of 128
    keys and more and no more than 2048 workgroups in all: those of the least time by 8
    us for a thousand keys on the CU with the most workgroups (on an average one for half
    of it: contexts differ, and the others make up for it), 2 us for a merge and .6 for
    each part in it. us at 1 / 2 / 3 / 4 / 6 parts, 16 heads on 4, and of a workgroup to a
    tile of 64 keys, with scores through the LDS: 33 rows behind 1000 to 8000 keys 113 /
    103 / 83 / 86 / 75 (5 taken, 78; 85), 40 rows 116 / 106 / 92 / 92 / 91 (3; 95), 33
    behind 200 to 3000 46 / 37 / 39 / 38 / 38 (3; 41), 64 of them in a window of 1024 27 /
    31 / 32 / 37 / 39 (1; 35), 300 rows of a prompt behind 8000 153 / 125 / 114 / 108 /
    116 (5, 107; 147). Of 307 batches of 1 to 200 sequences one is slower than that by more
    than 2 % (65 / 64), .83 of its time on average, 1.2 % above the best number of each."""
    def time(parts):
        most = nt * parts / 256
        return 4e-3 * span * (math.ceil(most) + max(most, 1)) / parts \
            + (parts > 1) * (2 + .6 * parts)

    return min(range(1, max(1, min(16, span // 128, 2048 // nt)) + 1), key=time)


def paged_attention(out, q, k_cache, v_cache, block_tables, row_seq, positions,
                    scale: float, maps: int = 1, window: int = 0,
                    keep_first: int = 0, sinks=None, tiles=None,
                    exact: bool = False, max_ctx: int = 0,
                    slopes=None, softcap: float = 0.0, chunk: int = 0,
                    gate=None, prompt_tiles=None) -> None:
    """q: [T, A, D], out: [T, A, VW] (A = heads * maps score maps; views
    whose last axis is contiguous). On the
    GPU the MFMA kernel runs for bf16 pools of fitting sizes, the fp32
    vector-ALU kernel otherwise (always for fp32 pools, or with `exact`).
    `max_ctx` (longest context in the batch, a host number) lets a batch of
    few tiles over long contexts split each tile's keys over workgroups.
    `slopes` (fp32, per head): slope * distance is taken off every scaled
    score. `softcap` > 0: scaled scores pass softcap * tanh(s / softcap).
    `chunk` > 0: keys of the row's own chunk of positions only. `gate`
    ([T, heads] view in q's dtype): a head's output times sigmoid(gate).
    `prompt_tiles` (build_prompt_tiles; GPU, where prompt_attention_fits):
    these portions' rows take the prompt kernel, `tiles` the others."""
    k = _paged_backend(q)
    if k is not None:
        if tiles is None:
            raise ValueError("paged_attention on GPU needs the tile list "
                             "(build_attn_tiles)")
        if prompt_tiles is not None:
            k.paged_prompt_attention(out, q, k_cache, v_cache, block_tables,
                                     prompt_tiles, scale, window, sinks,
                                     slopes)
            if tiles.shape[0] == 0:
                return
        nsplit = 1
        nt = tiles.shape[0]
        span = min(max_ctx, window + keep_first) if window > 0 else max_ctx
        if chunk > 0:
            span = min(span, chunk)
        if span >= 512 and 0 < nt < 2048:
            if (q.shape[-1] == 128 and 64 < out.shape[-1] <= 128
                    and q.dtype == torch.bfloat16):
                nsplit = _paged_wave_parts(nt, span)
            else:
                # 1024 workgroups, or up to 2048 while the split stays <= 4 (a
                # wider split pays more for the merge than it gains in
                # occupancy), each of at least 128 keys
                nsplit = max(1, min(16, span // 128,
                                    max(1024 // nt, min(4, 2048 // nt))))
        k.paged_attention(out, q, k_cache, v_cache, block_tables, tiles,
                          positions, scale, maps, window, keep_first, sinks,
                          exact, nsplit, slopes, softcap, chunk, gate)
    else:
        torch_ref.paged_attention(out, q, k_cache, v_cache, block_tables,
                                  row_seq, positions, scale, maps, window,
                                  keep_first, sinks, slopes, softcap, chunk,
                                  gate)


def head_rope_store(q_out, src, col_q: int, q_heads: int, q_dim: int, q_w,
                    q_norm_dims: int, q_rot0: int, col_k: int, k_heads: int,
                    k_dim: int, k_w, k_norm_dims: int, k_rot0: int, col_v: int,
                    inv_freq, half_layout: bool, amplitude: float, pos32,
                    k_cache, v_cache, slots, eps: float,
                    page_groups=None) -> None:
    """Per-head norm + rotation + cache write (torch_ref.head_rope_store
    has the semantics). `page_groups` (build_page_groups; GPU, prompts,
    values read from src): the value rows are written page by page."""
    k = _paged_backend(src)
    if k is not None:
        k.head_rope_store(q_out, src, col_q, q_heads, q_dim, q_w, q_norm_dims,
                          q_rot0, col_k, k_heads, k_dim, k_w, k_norm_dims,
                          k_rot0, col_v, inv_freq, half_layout, amplitude,
                          pos32, k_cache, v_cache, slots, eps, page_groups)
    else:
        torch_ref.head_rope_store(q_out, src, col_q, q_heads, q_dim, q_w,
                                  q_norm_dims, q_rot0, col_k, k_heads, k_dim,
                                  k_w, k_norm_dims, k_rot0, col_v, inv_freq,
                                  half_layout, amplitude, pos32, k_cache,
                                  v_cache, slots, eps)


def dual_rms_mix(out, a, wa, b, wb, eps: float) -> None:
    k = _paged_backend(a)
    if k is not None:
        k.dual_rms_mix(out, a, wa, b, wb, eps)
    else:
        torch_ref.dual_rms_mix(out, a, wa, b, wb, eps)


def head_gate(out, o_hts, gate_src, col: int) -> None:
    k = _paged_backend(o_hts)
    if k is not None:
        k.head_gate(out, o_hts, gate_src, col)
    else:
        torch_ref.head_gate(out, o_hts, gate_src, col)


def diff_combine(out, a, lam, diff: float, eps: float) -> None:
    k = _paged_backend(a)
    if k is not None:
        k.diff_combine(out, a, lam, diff, eps)
    else:
        torch_ref.diff_combine(out, a, lam, diff, eps)


def act_and_mul(out, gu, mode: str) -> None:
    k = _paged_backend(gu)
    if k is not None:
        k.act_and_mul(out, gu, ACT_MODES[mode])
    else:
        torch_ref.act_and_mul(out, gu, mode)


# --- layer-norm fp32 stream, attention without rotation, recurrent mixers ---
# ops/csrc/lnrows32.hip and ops/csrc/state_scan.hip in `_hip_state.so`.

_STATE = None


def _load_state():
    """Load `_hip_state.so` (layer-norm row kernels, head-norm cache write,
    short convolution, matrix-state scan, gated norms, scored routing),
    compiling it in-tree first when no built library is there."""
    global _STATE
    if _STATE is not None:
        return _STATE
    import importlib.util

    from .build import STATE_SO_PATH, build_state

    if not STATE_SO_PATH.exists():
        build_state()
    spec = importlib.util.spec_from_file_location(
        "gpustack_amd.ops._hip_state", STATE_SO_PATH)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    _STATE = mod
    return mod


def _state_backend(t: torch.Tensor):
    return _load_state() if t.is_cuda else None


def embed_rows_scaled(x, tokens, embed, scale: float) -> None:
    k = _state_backend(x)
    if k is not None:
        k.embed_rows_scaled(x, tokens, embed, scale)
    else:
        torch_ref.embed_rows_scaled(x, tokens, embed, scale)


def add_layer_norm(x, a, w, b, eps: float, h) -> None:
    """x += a and h = its layer norm; a may be the parts of a product
    (linear_auto)."""
    k = _state_backend(x)
    if k is not None:
        k.add_layer_norm(x, a, w, b, eps, h)
    else:
        torch_ref.add_layer_norm(x, a, w, b, eps, h)


def add_layer_norm_rows(x, a, w, b, eps: float, rows, dtype):
    """The layer norm of the given rows of x + a, x getting the sum or not: the
    end of a stream, of the rows whose logits are asked for. With an `a` the
    caller has seen that there are such rows: the GPU clamps others."""
    k = _state_backend(x)
    h = torch.empty(rows.shape[0], x.shape[1], dtype=dtype, device=x.device)
    if k is not None and a is not None and rows.is_cuda and x.shape[0] > 0 \
            and rows.dtype == torch.int64 and rows.is_contiguous() \
            and k.add_layer_norm(x, a, w, b, eps, h, rows):
        return h
    if a is not None:
        add_layer_norm(x, a, None, None, eps, None)
    add_layer_norm(x[rows].contiguous(), None, w, b, eps, h)
    return h


def head_norm_parts_ok(T: int, head_dim: int, nv: int, k_cache) -> bool:
    """Whether head_norm_store adds a projection's parts up: whole lanes of 8
    channels, a key pool at a 16-byte address, rows whose weights bound the product
    (64 rows of 3072 x 2048 12.0 us in the library, 6.5 cut over k)."""
    return T <= 128 and head_dim in (64, 128, 256) and nv % 8 == 0 \
        and k_cache.data_ptr() % 16 == 0


def head_norm_store(q_out, qkv, nq: int, nk: int, q_w, k_w, head_dim: int,
                    temp_coef: float, temp_every: float, pos32, v_first, lam,
                    k_cache, v_cache, slots, eps: float,
                    page_groups=None, parts=None) -> None:
    """`page_groups` (build_page_groups; GPU, prompts): the value rows are
    written page by page instead of row by row. `parts` (linear_auto; GPU,
    head_norm_parts_ok): the rows are their sum, of which qkv is left the
    values."""
    k = _state_backend(qkv)
    if k is not None:
        k.head_norm_store(q_out, qkv, nq, nk, q_w, k_w, head_dim, temp_coef,
                          temp_every, pos32, v_first, lam, k_cache, v_cache,
                          slots, eps, page_groups, parts)
    else:
        torch_ref.head_norm_store(q_out, qkv, nq, nk, q_w, k_w, head_dim,
                                  temp_coef, temp_every, pos32, v_first, lam,
                                  k_cache, v_cache, slots, eps)


def short_conv(out, src, col0: int, w, b, conv_state, seq_first, seq_rows,
               state_slots, row_seq, pos32, silu: bool = True,
               single: bool = False) -> None:
    """Short causal convolution per channel, with or without SiLU
    (torch_ref.short_conv has the semantics). `single` (a host-side hint):
    every sequence brings one row; the slot moves on in the same launch."""
    if src.is_cuda:
        # the kernel ships in both libraries: whichever is loaded
        k = _STATE or _STREAMS or _load_streams()
        k.short_conv(out, src, col0, w, b, conv_state, seq_first, seq_rows,
                     state_slots, row_seq, pos32, silu, single)
    else:
        torch_ref.short_conv(out, src, col0, w, b, conv_state, seq_first,
                             seq_rows, state_slots, pos32, silu)


def causal_conv_silu(out, src, col0: int, w, b, conv_state, seq_first,
                     seq_rows, state_slots, row_seq, pos32,
                     single: bool = False) -> None:
    if src.is_cuda:
        _load_state()       # models that call this run on that library
    short_conv(out, src, col0, w, b, conv_state, seq_first, seq_rows,
               state_slots, row_seq, pos32, single=single)


# Rows a sequence, on average, from which state_scan takes its chunk kernel
# (CHUNK_ROWS in ops/csrc/state_scan.hip)
SCAN_CHUNK_ROWS = 24


def scan_run_rows(seq_news, heads: int, vdim: int,
                  exact: bool = False) -> int:
    """Rows of a run for state_scan, or 0 where whole sequences do as well: up
    to half of the chip's 512 places for workgroups (64 value channels of a
    head) would work through the longest sequence alone. us whole / in runs of
    an eighth of it and 64 rows: 64 heads of 64 channels, 1 x 4000 rows 723 /
    266, 1 x 1000 191 / 107, 1 x 500 97 / 70, 1 x 250 50 / 50, 2 x 2000 364 /
    259, six of 301 to 1900 433 / 353, but 8 x 500 141 / 250, 4 x 200 47 / 91;
    16 heads of 128 1 x 4000 918 / 260, 1 x 500 121 / 77, the six 428 / 241,
    8 x 500 133 / 173, 32 x 125 91 / 145. Of 345 batches that it cuts 20 take
    longer, most at about 256 rows (49 / 54), at worst where the others fill the
    chip anyway (400 beside 12 x 200 rows of 32 heads 93 / 115). Batches of so many
    short sequences that no chunk kernel runs have none either.
    `exact`: rows that no activation is put on, whose chunks take a quarter to half
    of the time. Runs pay for the second walk later, and want to be longer: as long
    as the longest sequence's root has it, or as many as the chip has places.
    64 heads of 64, 1 x 500 rows 37 / 43, 1 x 1000 69 / 51, 1 x 4000 254 / 120, 2 x
    2000 130 / 98, but 3 x 2000 132 / 149, six of 301 to 1900 155 / 187; 16 heads of
    128 the six 124 / 97, 4 x 1000 69 / 62; 8 of 64 4 x 4000 253 / 105. Whole ones pay
    where a long sequence stands among many short ones: up to 185 places of a row of
    the longest the sum of 12 uneven batches is .86 of it in runs (24 sequences, 1389 of
    3928 rows in one, 311 / 146; but 657 of 913 70 / 84), beyond about even. Of 261
    uneven batches none takes longer than on fp32 instructions by more than 1 %, .57 on average,
    1.05 of the best of ten lengths each; at worst 2.1 (3322 of 5527 rows in one of 8,
    128 heads 593 / 280)."""
    longest, rows = max(seq_news, default=0), sum(seq_news)
    groups = heads * ((vdim + 63) // 64)
    if exact:
        if longest < 640 or longest * 185 <= rows * groups \
                or rows < SCAN_CHUNK_ROWS * len(seq_news):
            return 0
        size = max(12 * math.sqrt(longest), rows * groups / 512)
        return (int(size) + 31) // 32 * 32
    if longest < 256 or longest * 256 <= rows * groups:
        return 0
    if rows < SCAN_CHUNK_ROWS * len(seq_news):
        return 0
    return (longest // 8 + 64 + 31) // 32 * 32


def state_scan(y, src, col_x: int, col_b: int, col_c: int, dt_src,
               col_dt: int, heads: int, groups: int, n_state: int, vdim: int,
               act_silu: bool, dt_bias, a_log, skip, decay, state, seq_first,
               seq_rows, state_slots, pos32, single: bool = False,
               runs=None, cut: int | None = None) -> None:
    """`single` (a host-side hint): every sequence brings one row, as in a
    decode step; the GPU then streams the states through its step kernel.
    `runs` (build_scan_runs; a prompt): the GPU cuts the sequences into runs of
    rows that workgroups take side by side. `cut`: how many of the list, its
    first, belong to sequences of several runs (None: all may); two states of
    all heads are kept for each of these during the call."""
    k = _state_backend(src)
    if k is not None:
        k.state_scan(y, src, col_x, col_b, col_c, dt_src, col_dt, heads,
                     groups, n_state, vdim, act_silu, dt_bias, a_log, skip,
                     decay, state, seq_first, seq_rows, state_slots, pos32,
                     single, runs, cut)
    else:
        torch_ref.state_scan(y, src, col_x, col_b, col_c, dt_src, col_dt,
                             heads, groups, n_state, vdim, act_silu, dt_bias,
                             a_log, skip, decay, state, seq_first, seq_rows,
                             state_slots, pos32)


def gated_group_norm(out, y, gate, w, groups: int, eps: float,
                     gate_first, y_scale=None) -> None:
    """gate_first: True / 1 = silu gate, then norm; False / 0 = norm, then
    sigmoid gate; 2 = norm, then silu gate. y_scale [T, groups] multiplies
    the parts of y first."""
    k = _state_backend(y)
    if k is not None:
        k.gated_group_norm(out, y, gate, w, groups, eps, int(gate_first),
                           y_scale)
    else:
        torch_ref.gated_group_norm(out, y, gate, w, groups, eps, gate_first,
                                   y_scale)


def route_topk(experts, weights, logits, correction, n_experts: int,
               groups: int, keep: int, group_top: int, sigmoid: bool,
               renorm: bool, scale: float) -> None:
    k = _state_backend(logits)
    if k is not None:
        k.route_topk(experts, weights, logits, correction, n_experts, groups,
                     keep, group_top, sigmoid, renorm, scale)
    else:
        torch_ref.route_topk(experts, weights, logits, correction, n_experts,
                             groups, keep, group_top, sigmoid, renorm, scale)


def delta_scan(y, src, col_q: int, col_k: int, col_v: int, gate_src,
               col_a: int, col_b: int, heads: int, groups: int, n_state: int,
               vdim: int, dt_bias, a_log, state, seq_first, seq_rows,
               state_slots, pos32, single: bool = False) -> None:
    """Gated delta rule over the state pool (torch_ref.delta_scan has the
    semantics). `single`: every sequence brings one row (a decode step)."""
    k = _state_backend(src)
    if k is not None:
        k.delta_scan(y, src, col_q, col_k, col_v, gate_src, col_a, col_b,
                     heads, groups, n_state, vdim, dt_bias, a_log, state,
                     seq_first, seq_rows, state_slots, pos32, single)
    else:
        torch_ref.delta_scan(y, src, col_q, col_k, col_v, gate_src, col_a,
                             col_b, heads, groups, n_state, vdim, dt_bias,
                             a_log, state, seq_first, seq_rows, state_slots,
                             pos32)


def rope_table(pos32, inv_freq):
    """cos / sin of pos * f for every row, [T, 2, half] fp32: the table a
    prompt's memory_scan reads (None on the CPU, whose reference turns the
    rows itself)."""
    if not pos32.is_cuda:
        return None
    out = torch.empty(pos32.numel(), 2, inv_freq.numel(), dtype=torch.float32,
                      device=pos32.device)
    _load_state().rope_table(out, pos32, inv_freq)
    return out


def memory_scan(y, q, k, v, state, seq_first, seq_rows, state_slots, pos32, *,
                q_scale: float = 1.0, k_scale: float = 1.0, decay=None,
                chan=None, w0=None, bonus=None, gates=None, i_b=None,
                f_b=None, cap: float = 0.0, extra=None, rden=None,
                inv_freq=None, rot=None, single: bool = False) -> None:
    """Matrix memory over the state pool (torch_ref.memory_scan has the
    semantics). `single`: every sequence brings one row (a decode step).
    `rot`: the step's rope_table, shared by the layers of a prompt (None: the
    op makes its own)."""
    b = _state_backend(q)
    if b is not None:
        b.memory_scan(y, q, k, v, q_scale, k_scale, decay, chan, w0, bonus,
                      rot, inv_freq, gates, i_b, f_b, cap, state, extra, rden,
                      seq_first, seq_rows, state_slots, pos32, single)
    else:
        torch_ref.memory_scan(y, q, k, v, state, seq_first, seq_rows,
                              state_slots, pos32, q_scale, k_scale, decay,
                              chan, w0, bonus, gates, i_b, f_b, cap, extra, rden,
                              inv_freq)


# --- parallel residual streams, token shift, gated recurrence --------------
# ops/csrc/hyperrows32.hip, gru_scan.hip and short_conv.hip in
# `_hip_streams.so`.

_STREAMS = None


def _load_streams():
    """Load `_hip_streams.so` (stream rows, token shift, gated recurrence,
    short convolution), compiling it in-tree first when no built library is
    there."""
    global _STREAMS
    if _STREAMS is not None:
        return _STREAMS
    import importlib.util

    from .build import STREAMS_SO_PATH, build_streams

    if not STREAMS_SO_PATH.exists():
        build_streams()
    spec = importlib.util.spec_from_file_location(
        "gpustack_amd.ops._hip_streams", STREAMS_SO_PATH)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    _STREAMS = mod
    return mod


def _streams_backend(t: torch.Tensor):
    return _load_streams() if t.is_cuda else None


def embed_streams(x, tokens, embed, scale: float) -> None:
    k = _streams_backend(x)
    if k is not None:
        k.embed_streams(x, tokens, embed, scale)
    else:
        torch_ref.embed_streams(x, tokens, embed, scale)


def stream_step(x, a, gate, gate_b, mix, out_w, in_w, norm_w, eps: float, h,
                shift=None) -> None:
    """Close one sublayer on the streams and open the next
    (torch_ref.stream_step has the semantics). `shift` = (hs, mu, state,
    row_seq, state_slots, pos32), for batches of single rows: the token
    shift of h (one or several, as in token_shift) runs in the same
    launch."""
    k = _streams_backend(x)
    if k is not None:
        k.stream_step(x, a, gate, gate_b, mix, out_w, in_w, norm_w, eps, h,
                      *(shift or (None,) * 6))
        return
    torch_ref.stream_step(x, a, gate, gate_b, mix, out_w, in_w, norm_w, eps, h)
    if shift is not None:
        hs, mu, state, row_seq, slots, pos32 = shift
        one = torch.ones_like(row_seq)
        torch_ref.token_shift(hs, h, mu, state,
                              torch.arange(h.shape[0], device=h.device), one,
                              slots[row_seq.long()], pos32)


def token_shift(hs, h, mu, state, seq_first, seq_rows, state_slots, row_seq,
                pos32) -> None:
    k = _streams_backend(h)
    if k is not None:
        k.token_shift(hs, h, mu, state, seq_first, seq_rows, state_slots,
                      row_seq, pos32)
    else:
        torch_ref.token_shift(hs, h, mu, state, seq_first, seq_rows,
                              state_slots, pos32)


SCAN_CHUNK = 64   # rows of one sequence a workgroup of the scan walks


def build_scan_chunks(seq_starts, seq_news, size: int, device):
    """Runs of at most `size` rows of one sequence in order, for scans that
    split a prompt over workgroups: int32 [n, 4] = first row, rows,
    sequence, list index of the sequence's first run."""
    return to_device([(_scan_chunks(seq_starts, seq_news, size,
                                    range(len(seq_news))), torch.int32)],
                     device)[0]


def build_scan_runs(seq_starts, seq_news, size: int, device):
    """(build_scan_chunks' list with the sequences of one run at its end, the
    number of entries in front of them)."""
    order = sorted(range(len(seq_news)), key=lambda i: seq_news[i] <= size)
    runs = to_device([(_scan_chunks(seq_starts, seq_news, size, order),
                       torch.int32)], device)[0]
    return runs, sum(-(-n // size) for n in seq_news if n > size)


def _scan_chunks(seq_starts, seq_news, size: int, order):
    import numpy as np

    parts, n = [], 0
    for i in order:
        st, new = seq_starts[i], seq_news[i]
        lo = np.arange(0, new, size)
        t = np.empty((lo.size, 4), dtype=np.int32)
        t[:, 0] = st + lo
        t[:, 1] = np.minimum(size, new - lo)
        t[:, 2] = i
        t[:, 3] = n
        n += lo.size
        parts.append(t)
    return np.concatenate(parts) if parts else np.empty((0, 4), dtype=np.int32)


def gru_scan(y, src, col_z: int, col_u: int, col_g: int, z_b, u_b, state,
             seq_first, seq_rows, state_slots, pos32, chunks=None) -> None:
    """Gated recurrence with one state value per channel
    (torch_ref.gru_scan has the semantics). `chunks` (build_scan_chunks; a
    prompt): rows are split over workgroups, whose partial recurrences are
    joined; None: one workgroup walks all rows of a sequence."""
    k = _streams_backend(src)
    if k is not None:
        k.gru_scan(y, src, col_z, col_u, col_g, z_b, u_b, state, seq_first,
                   seq_rows, state_slots, pos32, chunks)
    else:
        torch_ref.gru_scan(y, src, col_z, col_u, col_g, z_b, u_b, state,
                           seq_first, seq_rows, state_slots, pos32)

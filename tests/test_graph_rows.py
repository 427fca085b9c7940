"""Captured steps that store and attend in one launch: only where every row is a sequence
of its own, and to the bit what the two launches give."""
from types import SimpleNamespace

import pytest
import torch

from gpustack_amd import ops
from gpustack_amd.engine import EngineConfig
from gpustack_amd.engine.graph_runner import DecodeGraphRunner
from gpustack_amd.engine.model_runner import ModelRunner
from gpustack_amd.engine.scheduler import Scheduler
from gpustack_amd.engine.sequence import SamplingParams, Sequence, SeqStatus


@pytest.mark.parametrize("drafted", [0, 3])
def test_rows_of_one_sequence_are_refused(drafted):
    """A row of such a step would read the pool while another one of its sequence
    writes there."""
    cfg = SimpleNamespace(max_num_seqs=4, max_model_len=64, block_size=16,
                          speculative={"num_draft_tokens": drafted} if drafted else None)
    graphs = DecodeGraphRunner(SimpleNamespace(
        cfg=cfg, device=torch.device("cpu"), ragged=False,
        kv=SimpleNamespace(pad_block=7, state_allocator=None)))
    graphs.graphs = {4: object()}
    batch = lambda n: SimpleNamespace(is_prefill=False, is_suffix=False, rows_per_seq=n,
                                      seqs=[None] * 2)
    assert graphs._meta(2).own_rows is (drafted == 0)
    assert graphs.can_run(batch(1))
    assert graphs.can_run(batch(2)) is (drafted > 0)
    for name in ("is_prefill", "is_suffix"):
        b = batch(1)
        setattr(b, name, True)
        assert not graphs.can_run(b)


def _runner(lens, kv_dtype, model, layers):
    cfg = EngineConfig(model=model, device="cuda:0", max_num_seqs=len(lens),
                       max_model_len=1200, kv_cache_blocks=sum(lens) // 16 + 40,
                       kv_cache_dtype=kv_dtype, seed=5, admission_min_seqs=1)
    cfg.spec.num_layers, cfg.spec.vocab_size = layers, 2048
    runner = ModelRunner(cfg)
    kv = runner.init_kv_cache()
    sch, g = Scheduler(cfg, kv), torch.Generator().manual_seed(3)
    for i, n in enumerate(lens):
        s = Sequence("r%d" % i, torch.randint(2, 2048, (n + 1,), generator=g).tolist(),
                     SamplingParams(max_tokens=99, ignore_eos=True))
        s.block_table = kv.allocator.allocate(kv.blocks_needed(n))
        s.num_cached_tokens, s.status = n, SeqStatus.RUNNING
        sch.running.append(s)
    return runner, sch.schedule()


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("model", ["llama-3-8b", "qwen3-14b"])
def test_captured_steps(monkeypatch, kv_dtype, model):
    """Up to 1100 keys in several parts, head norms, pools in bf16 and fp8; other numbers
    in the pools, and work of others, between the replays."""
    lens, steps, taken = [1100, 15, 64, 377, 900], [], []
    rows = ops.paged_attn_decode_rows
    monkeypatch.setattr(ops, "paged_attn_decode_rows",
                        lambda *a: (taken.append(1), rows(*a)))
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(ops, "paged_attn_decode_rows_ok", lambda *a: False)
        n = len(taken)
        runner, batch = _runner(lens, kv_dtype, model, 2)
        assert (len(taken) > n) is fused
        assert runner.graph_runner.can_run(batch)
        pools = [*runner.kv.k_caches, *runner.kv.v_caches]
        bucket = next(b for b in runner.graph_runner.buckets if b >= len(lens))
        for seed in range(3):
            g = torch.Generator(device="cuda").manual_seed(seed)
            for t in pools:
                t.copy_(torch.randn(t.shape, generator=g, device="cuda").to(t.dtype))
            runner.execute_async(batch, reuse_tokens=False)
            steps.append([runner.graph_runner.outs[bucket][:len(lens)].clone()]
                         + [t.view(torch.uint8).clone() for t in pools])
            torch.cuda.synchronize()
            torch.ones(1 << 20, device="cuda").sum().item()
        del runner, pools
    assert bool(steps[0][0].isfinite().all())
    for a, b in zip(steps[:3], steps[3:]):
        for u, v in zip(a, b):
            assert torch.equal(u, v)

"""Token ids outside the vocabulary and logit rows outside the batch are refused,
also where the kernel that gathers by them would not."""
import pytest
import torch

from gpustack_amd import ops
from gpustack_amd.engine import EngineConfig, LLMEngine
from gpustack_amd.engine.graph_runner import DecodeGraphRunner
from gpustack_amd.engine.scheduler import ScheduledBatch
from gpustack_amd.engine.sequence import Sequence

DEVICES = ["cpu", pytest.param("cuda:0", marks=[
    pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(),
                                        reason="needs a GPU")])]


def _engine(device="cpu"):
    if device != "cpu":
        cfg = EngineConfig(model="llama-3-8b", device=device, max_model_len=128,
                           max_num_seqs=4, gpu_memory_utilization=0.2)
        cfg.spec.num_layers = 2
        return LLMEngine(cfg)
    return LLMEngine(EngineConfig(model="tiny", device=device,
                                  max_model_len=128, max_num_seqs=4,
                                  kv_cache_blocks=64))


def _batch(eng, ids, prefill=True, **kw):
    seq = Sequence("t", list(ids))
    seq.block_table = eng.scheduler.kv.allocator.allocate(2)
    n = len(ids)
    return ScheduledBatch(
        is_prefill=prefill, seqs=[seq], token_ids=list(ids),
        positions=list(range(n)), seq_lens=[n],
        slot_mapping=eng.scheduler.kv.slots_for(seq.block_table, 0, n), **kw)


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("bad", [-1, "vocab", 2 ** 40])
@pytest.mark.parametrize("prefill", [True, False])
def test_ids_outside_the_vocabulary(device, bad, prefill):
    eng = _engine(device)
    V = eng.cfg.spec.vocab_size
    bad = V if bad == "vocab" else bad
    ids = [3, V - 1, bad] if prefill else [bad]
    with pytest.raises(IndexError):
        eng.runner.forward_logits(_batch(eng, ids, prefill))
    with pytest.raises(IndexError):
        eng.runner.execute(_batch(eng, ids, prefill))
    with pytest.raises(IndexError):
        eng.runner.embed([[1, 2], [bad]])
    with pytest.raises(IndexError):
        eng.runner.score_tokens([[1, 2], [bad]], [1])
    assert eng.runner.forward_logits(_batch(eng, [0, V - 1])).shape[-1] == V


def test_long_lists_and_arrays_of_ids():
    import numpy as np

    run = _engine().runner
    V = run.cfg.spec.vocab_size
    for n in (0, 1, 512, 513, 5000):
        ids = [i % V for i in range(n)]
        for form in (ids, np.asarray(ids, dtype=np.int64)):
            assert list(run.in_vocab(form)) == ids
        for bad in (-1, V):
            for at in {0, n // 2, n - 1} if n else ():
                wrong = ids[:at] + [bad] + ids[at + 1:]
                for form in (wrong, np.asarray(wrong)):
                    with pytest.raises(IndexError):
                        run.in_vocab(form)


def test_a_captured_step_refuses_them():
    eng = _engine()
    graphs = DecodeGraphRunner(eng.runner)
    with pytest.raises(IndexError):
        graphs.run(_batch(eng, [eng.cfg.spec.vocab_size], False))


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("row", [3, -4])
def test_logit_rows_outside_the_batch(device, row):
    eng = _engine(device)
    with pytest.raises(IndexError):
        eng.runner.forward_logits(_batch(eng, [1, 2, 3], logit_rows=[0, row]))
    got = eng.runner.forward_logits(_batch(eng, [1, 2, 3],
                                           logit_rows=[2, -1]))
    assert torch.equal(got[0], got[1])


def test_what_nobody_checked_goes_to_torch(monkeypatch):
    """The gathers without a refusal of their own are for checked steps."""
    eng = _engine()
    tokens, meta = eng.runner._meta(_batch(eng, [1, 2, 3]))
    want = eng.runner.model(tokens, meta, eng.runner.kv)

    def never(*a):
        raise AssertionError("an unchecked step")

    monkeypatch.setattr(ops, "embed_rms_norm_ok", lambda *a: True)
    monkeypatch.setattr(ops, "embed_rms_norm", never)
    monkeypatch.setattr(ops, "add_rms_norm_rows", never)
    meta.checked = False
    assert torch.equal(eng.runner.model(tokens, meta, eng.runner.kv), want)
    with pytest.raises(IndexError):
        eng.runner.model(tokens + eng.cfg.spec.vocab_size, meta, eng.runner.kv)

"""Host integers on their way to the device (ops.to_device)."""
import numpy as np
import pytest
import torch

from gpustack_amd import ops

DEVICES = ["cpu", pytest.param("cuda", marks=[
    pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(),
                                        reason="needs a GPU")])]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("n", [0, 1, 3, 8191])
def test_values_and_types(device, n):
    ids = list(range(5, 5 + n))
    parts = [(ids, torch.long), (ids, torch.int32),
             (np.arange(n, dtype=np.int64), torch.int32),
             (np.arange(2 * n, dtype=np.int32).reshape(2, n), torch.int32),
             ([np.int64(7), 8], torch.long),
             (torch.arange(n), torch.long)]
    want = [torch.as_tensor(np.asarray(v), dtype=t) for v, t in parts]
    got = ops.to_device(parts, device)
    assert [g.dtype for g in got] == [w.dtype for w in want]
    assert all(g.device.type == device and torch.equal(g.cpu(), w)
               for g, w in zip(got, want))


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("value", [2 ** 31, -2 ** 31 - 1, 2 ** 40])
def test_values_that_a_type_does_not_hold(device, value):
    """Refused, as torch.tensor refuses them, not wrapped."""
    with pytest.raises(RuntimeError):
        torch.tensor([3, value], dtype=torch.int32)
    with pytest.raises((RuntimeError, OverflowError)):
        ops.to_device([([3, value], torch.int32)], device)
    ends = [2 ** 31 - 1, -2 ** 31]
    assert ops.to_device([(ends, torch.int32)], device)[0].tolist() == ends


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_copies_queued_behind_work_keep_their_values():
    """The pinned memory of a copy that has not run is not handed out again."""
    a = torch.randn(4096, 4096, device="cuda")
    for _ in range(20):
        b = a @ a
    got = [ops.to_device([([i] * 4000, torch.long)], "cuda")[0]
           for i in range(50)]
    assert all(bool((g == i).all()) for i, g in enumerate(got)), b.shape

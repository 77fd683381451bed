"""ri_append_kv: the token's rows land at their position and nowhere else."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BG,stride,pos,on_device", [(1, 1, 0, False), (3, 70, 69, False), (16, 69, 0, True),
                                                     (37, 324, 100, True), (37, 324, 324, True), (5, 8, -1, True)])
def test_append_kv(dev, BG, stride, pos, on_device):
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(BG)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(dev)
    k, v, zk, zv = bf(BG, 128), bf(BG, 128), bf(BG, stride, 128), bf(BG, stride, 128)
    want = [zk.clone(), zv.clone()]
    if 0 <= pos < stride:
        want[0][:, pos], want[1][:, pos] = k, v
    at = torch.tensor([pos], dtype=torch.int64, device=dev) if on_device else None
    kernels.append_kv(k, v, zk, zv, 0 if on_device else pos, at)
    assert torch.equal(zk, want[0]) and torch.equal(zv, want[1])
    if not on_device:
        with pytest.raises(RuntimeError):
            kernels.append_kv(k, v, zk, zv, stride)

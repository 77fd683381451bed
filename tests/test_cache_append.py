"""The host side of appending a token to the steady zone (CPU): what is refused, and which rows take which way."""
import pytest
import torch

from retrievalattention_amd import kernels
from retrievalattention_amd.cache_hub import retroinfer_cache


def _cache(monkeypatch, rows, filled, **attributes):
    """A cache of one layer, one sequence and two KV heads, with only what the append looks at."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    c = object.__new__(retroinfer_cache)
    zone = lambda: [torch.zeros(1, 2, rows, 128, dtype=torch.bfloat16)]
    c.__dict__.update(dict(
        layer_num=1, context=filled, static_pattern_start=4, static_pattern_end=64, static_pattern_total=filled,
        device_positions=False, steady_zone_keys=zone(), steady_zone_values=zone(), _row_shape=(1, 1, 2, 128)), **attributes)
    return c


@pytest.mark.parametrize("device_positions", [False, True])
def test_full_steady_zone_refuses_a_token(monkeypatch, device_positions):
    c = _cache(monkeypatch, 70, 69, device_positions=device_positions, steady_pos_dev=torch.tensor([69]))
    row = torch.ones(1, 1, 2, 128, dtype=torch.bfloat16)
    c.decode_update_kv_cache(row, row, 0)
    assert c.static_pattern_total == 70 and bool((c.steady_zone_keys[0][:, :, 69] == 1).all())
    c.steady_pos_dev.fill_(3)      # (a position inside the zone: the host counter alone has to refuse)
    with pytest.raises(IndexError):
        c.decode_update_kv_cache(2 * row, row, 0)
    assert c.static_pattern_total == 70 and not c.steady_zone_keys[0][:, :, :69].any()


def test_replayed_token_without_a_row_is_reported(monkeypatch):
    c = _cache(monkeypatch, 70, 69, device_positions=True)
    c.token_replayed()             # the zone's last row
    with pytest.raises(IndexError, match="zone is full"):
        c.token_replayed()
    assert c.context == 70 and c.static_pattern_total == 70


class _OnDevice:
    """What the checks before a native call ask of a device tensor, for a device of choice."""
    is_cuda, dtype = True, torch.bfloat16

    def __init__(self, device, *shape):
        self.index, self.device, self.shape = device, torch.device("cpu"), torch.Size(shape)

    def get_device(self):
        return self.index

    def is_contiguous(self):
        return True

    def data_ptr(self):
        return 256

    def numel(self):
        return self.shape.numel()


@pytest.mark.parametrize("row_device,zone_device,native", [(0, 0, True), (1, 1, True), (1, 0, False), (0, 1, False)])
def test_native_calls_take_tensors_of_one_device(monkeypatch, row_device, zone_device, native):
    """Rows and queries of another device than the layer's buffers go the general way (copies across devices)."""
    c = _cache(monkeypatch, 70, 69)
    calls = []
    monkeypatch.setattr(kernels, "append_kv", lambda *a: calls.append(a))
    c.steady_zone_keys = c.steady_zone_values = [_OnDevice(zone_device, 1, 2, 70, 128)]
    row = _OnDevice(row_device, 1, 1, 2, 128)
    assert c._append(row, row, 0) is native and len(calls) == native

    class Taken(Exception):
        pass

    def plan(*a):
        raise Taken("prepared")

    def select(*a, **k):
        raise Taken("general")

    c.__dict__.update(batch_size=1, num_heads=8, batch_groups=2, group_size=4, head_dim=128, dtype=torch.bfloat16,
                      overlap_miss_staging=False, es_cluster_num=3, cache_blocks=1, cache_size=1, page_size=8,
                      centroids=[_OnDevice(zone_device, 2, 8, 128)], _plan=plan, _host_plan=plan, _select=select)
    q = _OnDevice(row_device, 1, 1, 8, 128)
    q.view = lambda *a: q
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: None)
    for compute in (lambda: c._compute_device(q, 0, 69, 0),
                    lambda: c._compute_host_in_place(q, 0, None, 69, 0, 1, True, False)):
        with pytest.raises(Taken, match="prepared" if native else "general"):
            compute()

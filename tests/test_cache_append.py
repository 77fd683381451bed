"""The host side of a decode step (CPU): which tokens the steady zone refuses, which tensors take which way, and when a
prepared call is prepared again."""
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

    def new_empty(self, shape):
        return torch.empty(shape, dtype=self.dtype)

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


@pytest.mark.parametrize("residency", ["device", "host"])
def test_prepared_call_follows_its_buffers(monkeypatch, residency):
    """Replacing any buffer whose address a prepared call holds prepares it again, once."""
    prepared = []

    class Plan:
        def __init__(self, key, *a):
            self.key = key
            prepared.append(self)

        def valid(self, key):
            return self.key == key

    monkeypatch.setattr(kernels, "DecodeStepPlan", Plan)
    monkeypatch.setattr(kernels, "HostStepPlan", Plan)
    new = lambda: torch.zeros(4, dtype=torch.int32)
    per_layer = ["centroids", "centroids_mask", "cluster_size_i32", "cluster_start", "value_sum", "cluster_size",
                 "steady_zone_keys", "steady_zone_values", "list_keys", "list_values", "ret_ids", "est_ids", "valid_lengths"]
    single = ["logits"]
    if residency == "device":
        single += ["ret_tok_off", "ret_start", "meta", "steady_len_dev"]
    else:
        per_layer += ["cache_keys", "cache_values", "hit_unit_idices", "hit_unit_sizes", "hit_unit_sizes_cumsum",
                      "hit_num_units", "miss_unit_idices", "miss_unit_sizes", "miss_unit_sizes_cumsum", "miss_num_units",
                      "update_buffer_indices", "update_unit_sizes", "update_cache_indices", "update_num_units"]
    c = _cache(monkeypatch, 70, 69, device_positions=residency == "device", _plans={}, nprobe=2, es_cluster_num=3,
               page_size=8, buffer_size=16, cache_size=1, dtype=torch.bfloat16, use_cluster_estimation=False, RSQRT_DIM=1.0)
    c.__dict__.update({n: [new()] for n in per_layer}, **{n: new() for n in single})
    c.layouts = [[new() for _ in range(4)]]
    lru = kernels.DeviceLru(2, 8, 16, 4, 4, 8, "cpu")
    c.device_lru = [lru]
    plan = c._plan if residency == "device" else c._host_plan
    replace = [lambda n=n: setattr(c, n, [new()]) for n in per_layer] + [lambda n=n: setattr(c, n, new()) for n in single]
    if residency == "host":
        replace += [lambda i=i: c.layouts[0].__setitem__(i, new()) for i in (2, 3)]
        replace += [lambda n=n: setattr(lru, n, getattr(lru, n).clone())
                    for n in ("blk_off", "stamp", "order", "blk_ids", "free_list", "free_count", "epoch")]
    keep = [plan(0, 0)]
    for i, move in enumerate(replace):
        held = {**c.__dict__, **lru.__dict__, "layouts": list(c.layouts[0])}   # (the old buffers keep their addresses)
        keep.append(held)
        move()
        assert plan(0, 0) is prepared[-1] and plan(0, 0) is prepared[-1]
        assert len(prepared) == i + 2, i

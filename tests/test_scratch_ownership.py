"""Whose scratch a decode step works in: caches may decode on different streams at a time, so each has its own arrival
counters, partials and scores' statistics, from before its first step on and also when its index grows."""
import gc

import pytest
import torch

from retrievalattention_amd import kernels
from retrievalattention_amd.cache_hub import retroinfer_cache


@pytest.fixture
def no_gpu(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(kernels, "_need", lambda *a, **k: None)


def _host_cache(nc=64):
    """What a cache of one layer and two groups lays down for its decode steps, in host memory."""
    c = object.__new__(retroinfer_cache)
    z = lambda *s, dt=torch.bfloat16: [torch.zeros(s, dtype=dt)]  # noqa: E731
    i32 = torch.int32
    c.__dict__.update(
        layer_num=1, layer_mapping={"0": "cpu"}, batch_size=1, batch_groups=2, head_dim=128, group_size=4, n_centroids=nc,
        nprobe=2, es_cluster_num=3, max_compute_cluster_num=5, kv_residency="device", block_cache="device",
        use_cluster_estimation=False, device_positions=False, page_size=8, buffer_size=64, dtype=torch.bfloat16,
        RSQRT_DIM=128 ** -0.5, _plans={}, _centred_keys={}, centroids=z(2, nc, 128), centroids_mask=z(2, nc, dt=torch.bool),
        cluster_size_i32=z(2, nc, dt=i32), cluster_start=z(2, nc, dt=i32), value_sum=z(2, nc, 128), cluster_size=z(2, nc),
        steady_zone_keys=z(1, 2, 70, 128), steady_zone_values=z(1, 2, 70, 128), list_keys=z(1, 2, 99, 128),
        list_values=z(1, 2, 99, 128))
    c.allocate_computation_buffer()
    c.prepare_cache()
    return c


def _areas(plan):
    return [plan._tensors[name] for name in ("score_workspace", "attn_workspace")]


def test_caches_have_scratch_of_their_own(no_gpu):
    a, b = _host_cache(), _host_cache()
    mine, other = _areas(a._plan(0, 0)), _areas(b._plan(0, 0))
    general = [kernels._workspace(256, torch.device("cpu"), tag) for tag in ("score0", "attn0")]
    spans = sorted((t.data_ptr(), t.data_ptr() + t.numel()) for t in mine + other + general)
    assert all(x[1] <= y[0] for x, y in zip(spans, spans[1:])), "scratch areas overlap"
    assert [t.data_ptr() for t in _areas(a._plan(0, 0))] == [t.data_ptr() for t in mine]


def test_nothing_of_a_step_is_allocated_during_its_capture(no_gpu, monkeypatch):
    c = _host_cache()
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    areas = _areas(c._plan(0, 0))
    for tag, mine in zip(("score0", "attn0"), areas):   # nor of the same operators by themselves
        assert kernels._workspace(mine.numel(), torch.device("cpu"), tag).data_ptr() != mine.data_ptr()
    with pytest.raises(RuntimeError, match="during a stream capture"):
        c._scratch.area(1 << 30, torch.device("cpu"), "attn0")


def test_outgrown_scratch_lives_as_long_as_its_owner(no_gpu):
    c = _host_cache()
    plan = c._plan(0, 0)
    before = plan._tensors["score_workspace"]
    c._scratch.area(4 * before.numel(), torch.device("cpu"), "score0")
    assert not plan.valid(plan.key) and any(t is before for t in c._scratch.retired)
    owner = c._scratch
    assert any(s is owner for s in kernels._all_scratch())
    kernels.release_cached_graphs()
    assert owner.retired == []
    count = len(kernels._all_scratch())
    del c, plan, owner
    gc.collect()
    assert len(kernels._all_scratch()) == count - 1


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,nc,nprobe,es", [(4096, 256, 26, 60), (8192, 512, 52, 118), (16384, 1024, 18, 237)])
def test_captured_steps_of_two_caches_on_two_streams(dev, tokens, nc, nprobe, es):
    """Replays that overlap give what the same replays give one after the other, bit for bit.  (Steps whose rows several
    workgroups of a group attend, in one launch and in two.)"""
    heads, gs, new = 2, 8, 8
    draw = torch.Generator(device=dev).manual_seed(tokens)
    bf = lambda *s: torch.randn(s, generator=draw, device=dev).to(torch.bfloat16)  # noqa: E731
    steps = []
    for _ in range(2):
        c = retroinfer_cache([0], 2, 1, tokens + 68 + new, heads, heads * gs, 128, torch.bfloat16,
                             {"0": "cuda:0", "1": "cuda:0"}, new, 4, 64, 2, nc, 1, nprobe, nprobe + es, 8, 3 * nprobe, 1, 0,
                             kv_residency="device", device_positions=True)
        for layer in range(2):
            c.prefill_update_kv_cache(None, bf(1, tokens + 68, heads, 128), bf(1, tokens + 68, heads, 128), layer, 0)
            c.sync(layer, 0)
        c.prepare_cache()
        q, k, v = bf(1, 1, heads * gs, 128), bf(1, 1, heads, 128), bf(1, 1, heads, 128)

        def replayed():   # (the first layer only: the position stays where it is)
            c.decode_update_kv_cache(k, v, 0)
            return c.compute(q, 0)

        replayed()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = [replayed() for _ in range(8)]
        steps.append((graph, out, torch.cuda.Stream(), c, q, k, v))   # (a graph holds addresses only)
    areas = [t.data_ptr() for _, _, _, c, *_ in steps for t in _areas(c._plan(0, 0))]
    assert len(set(areas)) == 4
    want = []
    for graph, out, *_ in steps:
        graph.replay()
        torch.cuda.synchronize()
        want.append([o.clone() for o in out])
    assert not torch.equal(want[0][0], want[1][0])
    torch.cuda.synchronize()
    for _ in range(25):
        for graph, _, stream, *_ in steps:
            with torch.cuda.stream(stream):
                graph.replay()
    torch.cuda.synchronize()
    for (_, out, *_), w in zip(steps, want):
        for got, expected in zip(out, w):
            assert torch.equal(got, expected)

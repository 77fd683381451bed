"""Which captured clustering a call of segment_k_means_csr replays (CPU, with the launches and the graphs stood in for)."""
import contextlib
from types import SimpleNamespace

import pytest
import torch

from retrievalattention_amd import kernels
from retrievalattention_amd.cache_hub import kmeans


@pytest.mark.parametrize("change", [
    dict(dtype=torch.float16), dict(shape=(2, 32, 128)), dict(num_iters=9), dict(num_segments=2), dict(num_centroids=32),
    dict(init_indices=torch.arange(64)), dict(key_store=torch.zeros(1))], ids=lambda c: next(iter(c)))
def test_a_captured_clustering_is_replayed_for_its_own_kind_of_call(monkeypatch, change):
    """Keys at the same address, but of another type or shape or with other parameters: not the captured launches."""
    monkeypatch.setattr(kmeans, "_GRAPHS", kmeans.collections.OrderedDict())
    monkeypatch.setattr(kmeans, "_SEEN", kmeans.collections.OrderedDict())
    result = lambda: SimpleNamespace(**{f: None for f in ("centroids", "assign", "counts", "offsets", "members")})
    launched, replayed = [], []
    monkeypatch.setattr(kmeans, "_cluster", lambda key, *a: launched.append(key.dtype) or result())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: SimpleNamespace(replay=lambda: replayed.append(1)))
    monkeypatch.setattr(torch.cuda, "graph", lambda g: contextlib.nullcontext())
    for name in ("kmeans_value_sum", "kmeans_store_rows"):
        monkeypatch.setattr(kernels, name, lambda *a, **k: None)
    memory = torch.zeros(1 * 64 * 128, dtype=torch.int16)

    def call(dtype=torch.bfloat16, shape=(1, 64, 128), num_centroids=64, **options):
        key = memory.view(dtype).view(shape)
        kmeans.segment_k_means_csr(key, key, num_centroids, reuse_graph=True, **options)

    for _ in range(3):
        call()
    assert len(launched) == 2 and len(replayed) == 2     # launched, captured and replayed, replayed
    call(**change)
    assert len(launched) == 3 and len(replayed) == 2


def test_a_captured_clustering_keeps_no_buffer_of_its_caller(monkeypatch):
    """Initial centroids that the caller hands over are the result's, by their address: neither they nor the keys stay alive with
    the graph, and other ones are another clustering."""
    import weakref
    monkeypatch.setattr(kmeans, "_GRAPHS", kmeans.collections.OrderedDict())
    monkeypatch.setattr(kmeans, "_SEEN", kmeans.collections.OrderedDict())
    replayed = []
    monkeypatch.setattr(kmeans, "_cluster", lambda key, *a: SimpleNamespace(
        centroids=a[-1], assign=None, counts=None, offsets=None, members=None))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: SimpleNamespace(replay=lambda: replayed.append(1)))
    monkeypatch.setattr(torch.cuda, "graph", lambda g: contextlib.nullcontext())
    monkeypatch.setattr(kernels, "kmeans_value_sum", lambda *a, **k: None)
    key, centroids, other = (torch.zeros(1, 64, 128, dtype=torch.bfloat16) for _ in range(3))
    call = lambda c: kmeans.segment_k_means_csr(key, key, 64, reuse_graph=True, centroids=c)
    for _ in range(3):
        assert call(centroids).centroids is centroids
    assert len(replayed) == 2 and call(other).centroids is other and len(replayed) == 2
    held = weakref.ref(centroids)
    del centroids
    assert held() is None

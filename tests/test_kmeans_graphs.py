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


def test_a_captured_clustering_is_found_by_its_keys_alone(monkeypatch):
    """Initial centroids that the caller hands over become a captured clustering's own, and later calls for the same keys are told
    to use them: a caller that comes after another one, with keys at the same address, replays at once.  Other ones are copied.
    The keys do not stay alive with the graph."""
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
    key = torch.zeros(1, 64, 128, dtype=torch.bfloat16)
    own = lambda: kmeans.initial_centroids(key, 64)
    call = lambda c: kmeans.segment_k_means_csr(key, key, 64, reuse_graph=True, centroids=c).centroids
    first, second = own(), own()
    assert first is not second and first.shape == (1, 64, 128) and first.dtype == key.dtype
    assert call(first) is first and call(second) is second and len(replayed) == 1   # launched; captured and replayed
    assert own() is second and call(own()) is second and len(replayed) == 2
    other = torch.ones(1, 64, 128, dtype=torch.bfloat16)
    assert call(other) is second and len(replayed) == 3 and torch.equal(second, other)
    for change in (dict(num_iters=9), dict(num_segments=2), dict(final_means=False)):
        assert kmeans.initial_centroids(key, 64, **change) is not second
    assert kmeans.initial_centroids(key, 32) is not second
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert own() is not second
    held = weakref.ref(key)
    del key
    assert held() is None

"""segment_k_means with the reference's signature and return values
(cache_hub/kmeans.py:224-259 of the reference), driven by the gfx950 kernels.

Differences that a caller can observe, both within what the reference leaves open:
  * cluster sums are accumulated in a fixed order (fp32: ascending token order in blocks of 256
    tokens, block sums added in block order) instead of by atomics, so the result is
    reproducible run to run;
  * tokens inside a cluster list are ascending (the reference's order is whatever its atomics
    produced).
"""
import collections

import torch

from .. import kernels


def init_centroid_indices(num_tokens, num_centroids, device):
    """kmeans.py:234-236: float32 arithmetic, truncated to int64."""
    idx = torch.arange(num_centroids, dtype=torch.float32, device=device) * (num_tokens / num_centroids)
    idx += num_tokens / num_centroids / 2
    return idx.to(torch.int64)


class KMeansResult:
    """CSR form of the clustering, kept on the device."""
    __slots__ = ("centroids", "value_sum", "assign", "counts", "offsets", "members")


def _cluster(key, num_centroids, num_iters, num_segments, init_indices, final_means=True, centroids=None):
    """Everything of the clustering that reads the keys: centroids, assignment, inverted lists.  final_means off: the
    caller takes the last means over the lists, which it makes itself where kmeans_store_makes_lists says so.
    centroids: the initial ones, which become the result's."""
    G, N, D = key.shape
    dev = key.device
    nc, S = num_centroids, num_segments
    if centroids is not None:
        pass
    elif init_indices is None:
        centroids = torch.empty((G, nc, D), dtype=key.dtype, device=dev)
        kernels.kmeans_init(key, centroids, G, N, nc)
    else:
        centroids = torch.index_select(key, 1, init_indices).contiguous()
    nseg, ncs = N // S, nc // S
    P = G * S
    assign = None
    if nseg > 0 and num_iters > 1:
        assign = torch.empty((P, nseg), dtype=torch.int32, device=dev)
        kernels.kmeans_iterate(key, centroids, assign, P, nseg, ncs, S, N, num_iters - 1, S == 1)
    r = KMeansResult()
    r.counts = torch.empty((G, nc), dtype=torch.int32, device=dev)
    r.offsets = torch.empty((G, nc + 1), dtype=torch.int32, device=dev)
    r.members = torch.empty((G, N), dtype=torch.int32, device=dev)
    if assign is not None and S == 1:   # (the segment is the sequence: the last pass over all centroids was one of them)
        r.assign = assign
    else:
        r.assign = torch.empty((G, N), dtype=torch.int32, device=dev)
        kernels.kmeans_assign(key, centroids, r.assign, G, N, nc, 1, N)
    if not final_means and kernels.kmeans_store_makes_lists(G, N, nc):
        pass
    elif N <= kernels.KMEANS_DIRECT_MAX_TOKENS and not final_means:
        kernels.kmeans_lists_direct(r.assign, r.counts, r.offsets, r.members, G, N, nc)
    elif N <= kernels.KMEANS_DIRECT_MAX_TOKENS:
        kernels.kmeans_update_direct(key, r.assign, centroids, G, N, nc, 1, N, False,
                                     (r.counts, r.offsets, r.members))
    else:
        kernels.kmeans_build_lists(r.assign, r.counts, r.offsets, r.members, G, N, nc)
        if final_means:
            kernels.kmeans_update(key, r.counts, r.offsets, r.members, centroids, G, N, nc, 1, N, False)
    r.centroids = centroids
    return r


# Captured clusterings, newest last: (key pointer, type, shape, parameters) -> (graph, result).  A clustering is
# about a hundred short launches; replayed as one HIP graph it loses the gaps between them.  The graph
# reads the key tensor afresh on every replay, so only the address has to stay the same, not the content.
_GRAPHS = collections.OrderedDict()
_SEEN = collections.OrderedDict()
_MAX_GRAPHS = 4


def _graph_key(key, nc, num_iters, S, final_means, init_indices, given):
    return (key.data_ptr(), key.dtype, key.shape, key.device, nc, num_iters, S, final_means,
            None if init_indices is None else init_indices.data_ptr(), given)


def initial_centroids(key, num_centroids, num_iters=10, num_segments=1, final_means=True):
    """[G, nc, 128] tensor for the initial centroids of a call of segment_k_means_csr with reuse_graph (final_means: without
    key_store): a captured clustering's own, which its replays start from and end in, else a new one."""
    hit = None
    if not torch.cuda.is_current_stream_capturing():
        hit = _GRAPHS.get(_graph_key(key, num_centroids, num_iters, num_segments, final_means, None, True))
    if hit is not None:
        return hit[1].centroids
    return torch.empty((key.shape[0], num_centroids, key.shape[2]), dtype=key.dtype, device=key.device)


def segment_k_means_csr(key, value, num_centroids, num_iters=10, num_segments=1, init_indices=None,
                        reuse_graph=False, value_sum=None, value_store=None, store_stride=0, key_rows=None, key_mean=None,
                        key_store=None, index=None, centroids=None):
    """Runs the clustering and returns a KMeansResult (no dense cluster lists, no host copy).
    key/value [G, N, 128] bfloat16 or float16 device tensors, keys contiguous.

    value_sum: [G, nc, 128] tensor for the sums (else a new one).  value_store: where the value rows are also
    written cluster by cluster, store_stride rows from group to group.  key_store (with value_store): the same for
    key_rows, the [G, N, 128] keys before key_mean was subtracted.  index (with key_mean): the tensors that
    kernels.prefill_index fills, filled here, with key_store in its launches.  centroids: [G, nc, 128] tensor with what
    kernels.kmeans_init gives for the keys, best in an initial_centroids(); it is written over, and the result's centroids are
    in it or in the captured clustering's.

    reuse_graph (off unless asked for): the second call with keys at the same address and of the same
    type, shape and parameters captures the launches into a HIP graph, and later such calls replay it.
    Results of replayed calls live in the graph's own memory: THEY ARE OVERWRITTEN by the next replay
    for the same key tensor, so only a caller that consumes or copies them before its next call may
    turn this on (prefill_update_kv_cache does: it copies everything into the cache's tensors at once;
    value sums are always fresh)."""
    G, N, D = key.shape
    if D != 128 or key.dtype not in (torch.bfloat16, torch.float16) or not key.is_contiguous():
        raise ValueError("segment_k_means: expected contiguous bfloat16 or float16 [G, N, 128] keys")
    if value.dtype != key.dtype:
        raise ValueError("segment_k_means: keys and values must have the same element type")
    if num_centroids % num_segments != 0:
        raise AssertionError("num_centroids must be divisible by num_segments")
    nc, S = num_centroids, num_segments
    if (nc // S) % 32 != 0 or nc % 32 != 0:
        raise AssertionError("centroids per segment must be a multiple of 32")  # kmeans.py:99
    r = None
    if reuse_graph and not torch.cuda.is_current_stream_capturing():
        gkey = _graph_key(key, nc, num_iters, S, key_store is None, init_indices, centroids is not None)
        hit = _GRAPHS.get(gkey)
        if hit is None and gkey in _SEEN:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                res = _cluster(key, nc, num_iters, S, init_indices, key_store is None, centroids)
            hit = (graph, res, init_indices)          # (the index tensor stays alive with the graph, as given centroids do)
            _GRAPHS[gkey] = hit
            while len(_GRAPHS) > _MAX_GRAPHS:
                _GRAPHS.popitem(last=False)
        if hit is not None:
            _GRAPHS.move_to_end(gkey)
            if centroids is not None and centroids is not hit[1].centroids:
                hit[1].centroids.copy_(centroids)
            hit[0].replay()
            r = KMeansResult()
            for f in ("centroids", "assign", "counts", "offsets", "members"):
                setattr(r, f, getattr(hit[1], f))
        else:
            _SEEN[gkey] = True
            while len(_SEEN) > 64:
                _SEEN.popitem(last=False)
    if r is None:
        r = _cluster(key, nc, num_iters, S, init_indices, key_store is None, centroids)
    r.value_sum = torch.empty((G, nc, D), dtype=value.dtype, device=key.device) if value_sum is None else value_sum
    if key_store is not None:
        kernels.kmeans_store_rows(kernels.aligned_rows(value), key_rows, key_mean, r.counts, r.offsets, r.members,
                                  r.value_sum, r.centroids, value_store, key_store, G, N, nc, store_stride, index,
                                  r.assign if kernels.kmeans_store_makes_lists(G, N, nc) else None)
        return r
    kernels.kmeans_value_sum(kernels.aligned_rows(value), r.counts, r.offsets, r.members, r.value_sum, G, N, nc,
                             store=value_store, store_stride=store_stride)
    if index is not None:
        kernels.prefill_index(r.centroids, key_mean, r.counts, r.offsets, *index)
    return r


def csr_to_dense(counts, offsets, members):
    """[G, nc, max_cluster_size] zero-padded lists as triton_reverse_index returns them
    (kmeans.py:155-173)."""
    G, nc = counts.shape
    mx = max(int(counts.max().item()), 1)
    col = torch.arange(mx, device=counts.device)[None, None, :]
    valid = col < counts[:, :, None]
    src = (offsets[:, :nc, None].long() + col).clamp_max(members.shape[1] - 1)
    dense = torch.gather(members.long()[:, None, :].expand(G, nc, -1), 2, src)
    return torch.where(valid, dense, torch.zeros_like(dense)).to(torch.int32)


def segment_k_means(key, value, num_centroids, num_iters=10, num_segments=1):
    """Reference signature: returns (centroids, value_sum, clusters, cluster_size), tensors of the
    caller's own (no captured graph: its results would be overwritten by a later call)."""
    r = segment_k_means_csr(key.contiguous(), value, num_centroids, num_iters, num_segments, reuse_graph=False)
    return r.centroids, r.value_sum, csr_to_dense(r.counts, r.offsets, r.members), r.counts

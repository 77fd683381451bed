"""Torch-facing wrappers of the C ABI.  The first block keeps the names and argument order of
the reference's `retroinfer_kernels` extension and of `weighted_flash_decoding`
(library/retroinfer/retroinfer_kernels/src/*.cu, *.cpp pybind sections), so code written
against the reference runs unchanged; the second block exposes the fused MI355X entry points.

Tensors only provide memory and the current stream; all arithmetic happens in the library.
"""
import contextlib
import ctypes
import functools
import math
import threading
import weakref

import torch

from ._lib import DecodeStep, Lru, lib, check, step_calls

# 16-bit element types of the reference's operators and cache (batch_gemm_softmax.cu:185-197,
# gather_copy.cu:63-67): every wrapper takes either and calls the entry point of that type (name or name_f16).
_DT = (torch.bfloat16, torch.float16)


def _fn(name, dtype):
    """The entry point `name` for 16-bit tensors of `dtype`."""
    if dtype not in _DT:
        raise RuntimeError("Only Half and BFloat16 are supported")
    return getattr(lib(), name + "_f16" if dtype == torch.float16 else name)

# Named profiler ranges around the stages of a decode step, with the names the reference gives its NVTX
# ranges (cache_hub/retroinfer_cache.py:558-678); torch's nvtx calls are roctx ranges on ROCm, so
# rocprofv3 --marker-trace shows them.  Off except inside `with profiler_ranges(True)`, which a cache built
# with profiler_ranges=True holds around its own calls (so one cache's ranges do not switch on another's).
PROFILER_RANGES = False


@contextlib.contextmanager
def profiler_ranges(enabled):
    global PROFILER_RANGES
    before, PROFILER_RANGES = PROFILER_RANGES, bool(enabled)
    try:
        yield
    finally:
        PROFILER_RANGES = before


def _ranged(name):
    def deco(fn):
        @functools.wraps(fn)
        def wrapper(*args, **kwargs):
            if not PROFILER_RANGES:
                return fn(*args, **kwargs)
            torch.cuda.nvtx.range_push(name)
            try:
                return fn(*args, **kwargs)
            finally:
                torch.cuda.nvtx.range_pop()
        return wrapper
    return deco


def _stream():
    """hipStream_t of the current device's current stream (torch.cuda.current_stream().cuda_stream without the
    Stream object around it: 0.3 instead of 2.7 us of a decode step's host time)."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _p(t):
    return None if t is None else t.data_ptr()


def _need(t, dtype, name, cuda=True):
    if t.dtype != dtype:
        raise TypeError(f"{name}: expected {dtype}, got {t.dtype}")
    if cuda and not t.is_cuda:
        raise ValueError(f"{name}: expected a device tensor")
    if not t.is_contiguous():
        raise ValueError(f"{name}: expected a contiguous tensor")


def _need_all(tensors, dtype, names):
    """_need for device tensors of one type: one look at each while nothing is wrong."""
    for t in tensors:
        if t.dtype is not dtype or not t.is_cuda or not t.is_contiguous():
            for x, nm in zip(tensors, names):
                _need(x, dtype, nm)


_scratches = weakref.WeakSet()   # every Scratch there is
_scratches_lock = threading.Lock()


class Scratch:
    """Scratch tensors by device and purpose, grown on demand and reused from call to call.  They start zeroed: the
    attention kernels keep arrival counters in them that they leave at zero, so calls that may overlap on the device
    (different streams) must not share one.  A cache has one of its own; calls that name none take the process's.
    A tensor that is outgrown is kept as long as its owner: a HIP graph captured earlier replays with its address, so
    handing the block back to the allocator would let that replay write into someone else's memory.  Growing (or first
    use) during a capture is refused: the allocation would land in the graph's private pool and its zero fill would
    become a memset node of the graph."""

    def __init__(self):
        self.areas, self.retired = {}, []
        self.generation = 0   # moves on whenever a tensor is replaced: holders of an address look again
        with _scratches_lock:
            _scratches.add(self)

    def area(self, nbytes, device, tag):
        key = (device, tag)
        w = self.areas.get(key)
        if w is None or w.numel() < nbytes:
            if torch.cuda.is_current_stream_capturing():
                raise RuntimeError(f"scratch area '{tag}' must grow to {nbytes} bytes during a stream capture: run the "
                                   "same call once before capturing")
            if w is not None:
                self.retired.append(w)
                nbytes = max(nbytes, w.numel() * 3 // 2)
            w = torch.zeros(max(nbytes, 256), dtype=torch.uint8, device=device)
            self.areas[key] = w
            self.generation += 1
        return w

    def decoding(self, BG, gs, nc, device):
        """The areas of a decode step of BG groups of gs query heads over nc clusters: of the selection, of the attention."""
        return (self.area(lib().ri_score_select_workspace_bytes(BG, gs, nc), device, "score0"),
                self.area(lib().ri_wave_attention_workspace_bytes(BG, gs), device, "attn0"))


shared_scratch = Scratch()   # the process's


def _workspace(nbytes, device, tag, scratch=None):
    return (shared_scratch if scratch is None else scratch).area(nbytes, device, tag)


def _all_scratch():
    with _scratches_lock:
        return list(_scratches)


def reset_attention_workspaces():
    """Clears the arrival counters of every attention scratch tensor (on the current stream of its device).
    The attention launches leave them at zero; call this after a launch that did not run to its end."""
    for scratch in _all_scratch():
        for (dev, tag), w in list(scratch.areas.items()):
            if tag.startswith("attn"):
                with torch.cuda.device(w.device):
                    check(lib().ri_attention_workspace_reset(_p(w), w.numel(), _stream()), "attention_workspace_reset")


def release_cached_graphs(retired_workspaces=True):
    """Drops what the library keeps alive for replays: the captured clusterings of segment_k_means_csr (only the
    library replays those, so this is always safe) and, with retired_workspaces, the scratch tensors that were
    outgrown.  A graph that a caller captured while such a tensor was current still holds its address: drop the
    retired tensors only when every graph captured before the last growth of a scratch area is gone, or a replay
    would write into memory that has been handed back.  Refused during a stream capture."""
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("release_cached_graphs during a stream capture")
    from .cache_hub import kmeans as _km
    _km._GRAPHS.clear()
    _km._SEEN.clear()
    if retired_workspaces:
        for scratch in _all_scratch():
            scratch.retired.clear()


# limits of the fused decode path (checked by the entry points; callers can check them up front)
MAX_PROBES = 4096          # ri_score_select / ri_wave_attention / ri_lru_access_update: retrieval zone per group
MAX_CLUSTERS = 65536       # ri_score_select / ri_lru_access_update: clusters per group (16-bit ids in the selection)
MAX_GROUP_SIZE = 16        # query heads per KV head
MAX_GROUPS = 4096          # ri_wave_attention / ri_weighted_flash_decoding: batch x KV heads of one launch


# ----------------------------------------------------------------------------------------
# retroinfer_kernels-compatible surface
# ----------------------------------------------------------------------------------------
def batch_gemm_softmax(A, B, D, Norm, Sum, Softmax, batch_count, m, n, k, alpha=1.0, beta=0.0):
    """batch_gemm_softmax.cu:201-209.  A [bc, m, k], B [bc, n, k]; D/Softmax [bc, m, n]."""
    status = step_calls().gemm_softmax(A, B, D, Softmax, Norm, Sum, batch_count, m, n, k, alpha, beta)
    if status is not None:
        return check(status, "batch_gemm_softmax") if status else None
    if A.dtype not in _DT:
        raise RuntimeError("Only Half and BFloat16 are supported")      # batch_gemm_softmax.cu:196
    _need_all((A, B, D, Softmax), A.dtype, ("A", "B", "D", "Softmax"))
    _need_all((Norm, Sum), torch.float32, ("Norm", "Sum"))
    ntiles = (n + 255) // 256
    if A.numel() < batch_count * m * k or B.numel() < batch_count * n * k or \
            D.numel() < batch_count * m * n or Softmax.numel() < batch_count * m * n or \
            Norm.numel() < batch_count * ntiles * m or Sum.numel() < batch_count * ntiles * m:
        raise ValueError("batch_gemm_softmax: a buffer is smaller than its shape arguments")
    fn = lib().ri_batch_gemm_softmax_f16 if A.dtype == torch.float16 else lib().ri_batch_gemm_softmax
    check(fn(_p(A), _p(B), _p(D), _p(Norm), _p(Sum), _p(Softmax), batch_count, m, n, k, float(alpha), float(beta),
             _stream()), "batch_gemm_softmax")


def gather_copy_vectors(key_data, key_buffer, value_data, value_buffer, src_metadata, dst_metadata,
                        data_offsets, groups, data_length, buffer_length, index_size, copy_start, copy_num):
    """gather_copy.cu:288-292.  The rows are moved as 16-bit elements: Half or BFloat16 (gather_copy.cu:63-67)."""
    status = step_calls().gather_vectors(key_data, key_buffer, value_data, value_buffer, src_metadata, dst_metadata, data_offsets,
                                         groups, data_length, buffer_length, index_size, copy_start, copy_num)
    if status is not None:
        return check(status, "gather_copy_vectors") if status else None
    if key_data.dtype not in _DT:
        raise RuntimeError("Only Half and BFloat16 are supported")
    _need_all((key_data, key_buffer, value_data, value_buffer, src_metadata, dst_metadata), key_data.dtype,
              ("key_data", "key_buffer", "value_data", "value_buffer", "src_metadata", "dst_metadata"))
    _need(data_offsets, torch.int64, "data_offsets")
    if key_data.numel() < groups * data_length * 128 or key_buffer.numel() < groups * buffer_length * 128 or \
            value_data.numel() < groups * data_length * 128 or value_buffer.numel() < groups * buffer_length * 128 or \
            data_offsets.numel() < groups * index_size or src_metadata.numel() < groups * data_length or \
            dst_metadata.numel() < groups * buffer_length:
        raise ValueError("gather_copy_vectors: a buffer is smaller than its shape arguments")
    check(lib().ri_gather_copy_vectors(_p(key_data), _p(key_buffer), _p(value_data), _p(value_buffer),
                                       _p(src_metadata), _p(dst_metadata), _p(data_offsets), groups, data_length,
                                       buffer_length, index_size, copy_start, copy_num, _stream()),
          "gather_copy_vectors")


@_ranged("gather_copy_and_concat")
def gather_copy_and_concat(key_data1, key_data2, key_data3, key_buffer, value_data1, value_data2, value_data3,
                           value_buffer, data_offsets2, data_copy_sizes2, buffer_offsets2, copy_chunks2,
                           data_offsets3, data_copy_sizes3, buffer_offsets3, copy_chunks3, valid_lengths,
                           groups, data_length1, data_length2, data_length3, buffer_length, offset_length,
                           copy_vectors1):
    """gather_copy.cu:294-300.  key_data2/value_data2 and the index tensors may be pinned host
    tensors (read in place by the kernel), everything else lives on the device."""
    for t in (data_offsets2, data_copy_sizes2, buffer_offsets2, copy_chunks2, data_offsets3, data_copy_sizes3,
              buffer_offsets3, copy_chunks3, valid_lengths):
        _need(t, torch.int32, "index tensor", cuda=False)
        if not (t.is_cuda or t.is_pinned()):
            raise ValueError("index tensors must be device or pinned host tensors")
    for t in (key_data2, value_data2):
        if not (t.is_cuda or t.is_pinned()):
            raise ValueError("key_data2/value_data2 must be device or pinned host tensors")
    check(lib().ri_gather_copy_and_concat(
        _p(key_data1), _p(key_data2), _p(key_data3), _p(key_buffer), _p(value_data1), _p(value_data2),
        _p(value_data3), _p(value_buffer), _p(data_offsets2), _p(data_copy_sizes2), _p(buffer_offsets2),
        _p(copy_chunks2), _p(data_offsets3), _p(data_copy_sizes3), _p(buffer_offsets3), _p(copy_chunks3),
        _p(valid_lengths), groups, data_length1, data_length2, data_length3, buffer_length, offset_length,
        copy_vectors1, _stream()), "gather_copy_and_concat")


def gather_copy_and_scatter(key_data, key_buffer, value_data, value_buffer, s_offsets, copy_sizes, d_offsets,
                            copy_chunks, groups, data_length, buffer_length, offset_length, s_copy_start):
    """gather_copy.cu:302-305."""
    for t in (s_offsets, copy_sizes, d_offsets, copy_chunks):
        _need(t, torch.int32, "index tensor", cuda=False)
        if not (t.is_cuda or t.is_pinned()):
            raise ValueError("index tensors must be device or pinned host tensors")
    check(lib().ri_gather_copy_and_scatter(_p(key_data), _p(key_buffer), _p(value_data), _p(value_buffer),
                                           _p(s_offsets), _p(copy_sizes), _p(d_offsets), _p(copy_chunks), groups,
                                           data_length, buffer_length, offset_length, s_copy_start, _stream()),
          "gather_copy_and_scatter")


@functools.lru_cache(maxsize=64)
def _flash_workspace_bytes(BG, gs):
    return lib().ri_flash_decoding_workspace_bytes(BG, gs)


@_ranged("flash_attention")
def weighted_flash_decoding(q, k, v, weight=None, previous_out=None, previous_lse=None, cache_seqlens=None,
                            return_softmax_lse=False, scratch=None):
    """Signature of the calls at cache_hub/retroinfer_cache.py:611-617 and :666-674.
    q [BG, 1, gs, D]; k, v [BG, S, 1, D]; weight [BG, 1, 1, S]; previous_out [BG, 1, gs, D];
    previous_lse [BG, gs] (any shape with BG*gs elements); cache_seqlens [BG] int32.
    `scratch`: the caller's own Scratch, where calls may overlap others."""
    BG, one, gs, D = q.shape
    if q.__class__ is torch.Tensor and q.is_cuda and one == 1 and D == 128 and q.dtype in _DT:
        ws = _workspace(_flash_workspace_bytes(BG, gs), q.device, "attn", scratch)
        out = step_calls().flash(q, k, v, weight, previous_out, previous_lse, cache_seqlens, ws, 1.0 / math.sqrt(D),
                                 return_softmax_lse)
        if out is not None:
            return check(out, "weighted_flash_decoding") if out.__class__ is int else out
    S = k.shape[1]
    if one != 1 or D != 128 or k.shape[2] != 1:
        raise ValueError("weighted_flash_decoding: expected q [BG,1,gs,128], k/v [BG,S,1,128]")
    dt = q.dtype
    if weight is not None:
        _need_all((q, k, v, weight), dt, ("q", "k", "v", "weight"))
    else:
        _need_all((q, k, v), dt, ("q", "k", "v"))
    if previous_out is not None:
        _need(previous_out, dt, "previous_out")
        _need(previous_lse, torch.float32, "previous_lse")
    if cache_seqlens is not None:
        _need(cache_seqlens, torch.int32, "cache_seqlens")
    if k.numel() < BG * S * D or v.numel() < BG * S * D or (weight is not None and weight.numel() < BG * S) or \
            (previous_out is not None and (previous_out.numel() < q.numel() or previous_lse.numel() < BG * gs)) or \
            (cache_seqlens is not None and cache_seqlens.numel() < BG):
        raise ValueError("weighted_flash_decoding: a tensor is smaller than the shapes of q and k ask for")
    out = torch.empty_like(q)
    lse = torch.empty((BG, gs), dtype=torch.float32, device=q.device) if return_softmax_lse else None
    ws = _workspace(_flash_workspace_bytes(BG, gs), q.device, "attn", scratch)
    check(_fn("ri_weighted_flash_decoding", dt)(_p(q), _p(k), _p(v), _p(weight), _p(cache_seqlens), _p(previous_out),
                                           _p(previous_lse), _p(out), _p(lse), BG, gs, S, S,
                                           1.0 / math.sqrt(D), _p(ws), ws.numel(), _stream()),
          "weighted_flash_decoding")
    return (out, lse) if return_softmax_lse else out


class ThreadPool:
    """wave_buffer_cpu.cpp:17-35.  first_core (None: workers run where the scheduler puts them): worker i is
    bound to core first_core + i, which is what the reference does with first_core = 0
    (thread_pool.hpp:18-23, 65-66); pinned_workers tells how many the system accepted."""

    def __init__(self, num_threads, first_core=None):
        self._destroy = lib().ri_threadpool_destroy   # bound now: module globals may be gone at interpreter exit
        if first_core is None:
            self._h = lib().ri_threadpool_create(int(num_threads))
        else:
            self._h = lib().ri_threadpool_create_pinned(int(num_threads), int(first_core))
        if not self._h:
            raise RuntimeError("ri_threadpool_create failed")
        self.pinned_workers = lib().ri_threadpool_pinned_workers(self._h)

    def get(self):
        return self

    def __del__(self):
        h, self._h = getattr(self, "_h", None), None
        if h:
            self._destroy(h)


class WaveBufferCPU:
    """wave_buffer_cpu.cpp:822-841.  Keeps references to every registered tensor, because the
    native object stores their addresses."""

    def __init__(self, batch_size, group_num, dim, nprobe, block_size, n_centroids, final_n_centroids,
                 buffer_size, capacity, threads, pool):
        self._pool = pool
        self._keep = {}
        self._destroy = lib().ri_wavebuf_destroy
        self._h = lib().ri_wavebuf_create(batch_size, group_num, dim, nprobe, block_size, n_centroids,
                                          final_n_centroids, buffer_size, capacity, threads, pool._h)
        if not self._h:
            raise ValueError("WaveBufferCPU: invalid construction arguments")

    def __del__(self):
        h, self._h = getattr(self, "_h", None), None
        if h:
            self._destroy(h)

    def set_indices(self, hit_block_ids, hit_block_sizes, hit_block_sizes_cumsum, hit_block_nums,
                    miss_block_ids, miss_block_sizes, miss_block_sizes_cumsum, miss_block_nums,
                    update_buffer_indices, update_block_sizes, update_cache_indices, update_block_nums,
                    searched_clusters):
        ts = [hit_block_ids, hit_block_sizes, hit_block_sizes_cumsum, hit_block_nums, miss_block_ids,
              miss_block_sizes, miss_block_sizes_cumsum, miss_block_nums, update_buffer_indices,
              update_block_sizes, update_cache_indices, update_block_nums]
        for t in ts:
            _need(t, torch.int32, "index tensor", cuda=False)
        _need(searched_clusters, torch.int64, "searched_clusters", cuda=False)
        self._keep["indices"] = ts + [searched_clusters]
        check(lib().ri_wavebuf_set_indices(self._h, *[_p(t) for t in ts], _p(searched_clusters)), "set_indices")

    def set_kv(self, ivf_key, ivf_value, input_keys, input_values):
        self._keep["kv"] = [ivf_key, ivf_value, input_keys, input_values]
        check(lib().ri_wavebuf_set_kv(self._h, _p(ivf_key), _p(ivf_value), ivf_key.size(2), _p(input_keys),
                                      _p(input_values), input_keys.size(1)), "set_kv")

    def async_construction(self, clusters, cluster_size, batch_idx):
        _need(clusters, torch.int32, "clusters", cuda=False)
        _need(cluster_size, torch.int32, "cluster_size", cuda=False)
        self._keep["construction"] = [clusters, cluster_size]
        check(lib().ri_wavebuf_async_construction(self._h, _p(clusters), _p(cluster_size), clusters.size(2),
                                                  int(batch_idx)), "async_construction")

    def construction_sync(self):
        check(lib().ri_wavebuf_construction_sync(self._h), "construction_sync")

    def update_kv(self, update_keys, update_values, clusters, cluster_size):
        _need(clusters, torch.int32, "clusters", cuda=False)
        _need(cluster_size, torch.int32, "cluster_size", cuda=False)
        check(lib().ri_wavebuf_update_kv(self._h, _p(update_keys), _p(update_values), update_keys.size(1),
                                         _p(clusters), _p(cluster_size), clusters.size(1), clusters.size(2)),
              "update_kv")

    def batch_access(self):
        check(lib().ri_wavebuf_batch_access(self._h), "batch_access")

    def sync(self):
        check(lib().ri_wavebuf_sync(self._h), "sync")

    def overflow_events(self):
        return int(lib().ri_wavebuf_overflow_events(self._h))


# ----------------------------------------------------------------------------------------
# fused MI355X entry points
# ----------------------------------------------------------------------------------------
@_ranged("search_topk_clusters")
def score_select(q, centroids, mask, cluster_size_i32, cluster_start, logits, dist, cI, ret_ids, est_ids,
                 ret_tok_off, row_src, meta, nprobe, es, page, max_pages, scale, slot=0, ret_start=None, scratch=None):
    """Centroid scoring + retrieval/estimation selection + token layout.  `slot` names the
    scratch area in `scratch` (None: the process's): calls that may run concurrently (different streams) must use
    different ones.
    The layout goes out as a row table (row_src), as rank tables (ret_tok_off + ret_start), or both."""
    BG, gs, D = q.shape
    nc = centroids.shape[1]
    nb = lib().ri_score_select_workspace_bytes(BG, gs, nc)
    ws = _workspace(nb, q.device, f"score{slot}", scratch)
    _need(centroids, q.dtype, "centroids")
    check(_fn("ri_score_select", q.dtype)(_p(q), _p(centroids), _p(mask), _p(cluster_size_i32), _p(cluster_start),
                                _p(logits), _p(dist), _p(cI), _p(ret_ids), _p(est_ids), _p(ret_tok_off),
                                _p(ret_start), _p(row_src), 0 if row_src is None else row_src.shape[1], _p(meta),
                                BG, gs, nc,
                                nprobe, es, page, max_pages, float(scale), _p(ws), ws.numel(), _stream()),
          "score_select")


def score_logits(q, centroids, logits, scale, slot=0, scratch=None):
    """logits [BG, gs, nc] fp32 = scale * q . centroids^T, no selection."""
    BG, gs, D = q.shape
    nc = centroids.shape[1]
    ws = _workspace(lib().ri_score_select_workspace_bytes(BG, gs, nc), q.device, f"score{slot}", scratch)
    _need(centroids, q.dtype, "centroids")
    check(_fn("ri_score_logits", q.dtype)(_p(q), _p(centroids), _p(logits), BG, gs, nc, float(scale), _p(ws), ws.numel(),
                                _stream()), "score_logits")


@_ranged("flash_attention")
def wave_attention(q, steady_k, steady_v, static_len, store_k, store_v, row_src, meta, est_ids, logits,
                   value_sum, cluster_size_bf16, out, valid_lengths, es, scale, slot=0, ret_tok_off=None,
                   ret_start=None, est_centroids=None, static_len_dev=None, scratch=None):
    """Attention over steady zone + retrieved clusters (read in place) + estimation zone.
    The retrieved rows come from a row table (row_src) or, with row_src None, from the rank tables
    ret_tok_off [BG, np+1] and ret_start [BG, np].  The estimation zone's scores are read from `logits`
    or, with logits None, computed in the launch from the rows of `est_centroids` [BG, nc, 128].
    With static_len_dev (int32 tensor of one element on the device) the number of steady rows is read
    from it when the kernel runs; static_len then only sizes the split.
    `slot`: scratch area in `scratch` (None: the process's), one per concurrent call."""
    BG, gs, D = q.shape
    nc = value_sum.shape[1]
    nb = lib().ri_wave_attention_workspace_bytes(BG, gs)
    ws = _workspace(nb, q.device, f"attn{slot}", scratch)
    for t, nm in ((steady_k, "steady_k"), (store_k, "store_k"), (value_sum, "value_sum"), (out, "out")):
        _need(t, q.dtype, nm)
    check(_fn("ri_wave_attention", q.dtype)(_p(q), _p(steady_k), _p(steady_v), steady_k.shape[-2], static_len,
                                  _p(static_len_dev), _p(store_k),
                                  _p(store_v), store_k.shape[-2], _p(row_src),
                                  0 if row_src is None else row_src.shape[1], _p(ret_tok_off), _p(ret_start),
                                  0 if ret_start is None else ret_start.shape[1], _p(meta), _p(est_ids), _p(logits),
                                  _p(est_centroids), _p(value_sum), _p(cluster_size_bf16), _p(out),
                                  _p(valid_lengths), BG, gs, nc, es, float(scale), _p(ws), ws.numel(), _stream()),
          "wave_attention")


class DecodeStepPlan:
    """score_select + wave_attention of one layer over a device-resident store as one call (ri_decode_step): the
    addresses and sizes, which stay the same from token to token, are checked and laid down once.  `tensors`: the
    fields of ri_decode_step_t that are addresses (None: not given); `key` is what the holder compares to see whether
    they still are what it would hand over now.  `scratch`: whose areas the step works in (None: the process's).  Every
    step may use the attention's arrival counters and partials, also of the shortest contexts: steps that may overlap
    on the device need plans over different Scratch objects."""

    def __init__(self, key, dtype, tensors, nprobe, es, page, max_pages, scale, scratch=None):
        c = tensors["centroids"]
        BG, nc, _ = c.shape
        gs = tensors["logits"].shape[1]
        for nm in ("centroids", "steady_k", "steady_v", "store_k", "store_v", "value_sum", "cluster_size"):
            _need(tensors[nm], dtype, nm)
        self._scratch = shared_scratch if scratch is None else scratch
        score, attn = self._scratch.decoding(BG, gs, nc, c.device)
        tensors = dict(tensors, score_workspace=score, attn_workspace=attn)
        self.key, self.generation = key, self._scratch.generation
        self._tensors = tensors
        self._step = DecodeStep(
            steady_stride=tensors["steady_k"].shape[-2], store_stride=tensors["store_k"].shape[-2],
            score_workspace_bytes=tensors["score_workspace"].numel(),
            attn_workspace_bytes=tensors["attn_workspace"].numel(), BG=BG, gs=gs, nc=nc, np=nprobe, es=es, page=page,
            max_pages=max_pages, half=int(dtype == torch.float16), scale=scale,
            **{nm: _p(t) for nm, t in tensors.items()})
        self._address = ctypes.addressof(self._step)
        self._lru_address = 0
        self._call = lib().ri_decode_step
        self._native = None

    def valid(self, key):
        return self.key == key and self.generation == self._scratch.generation

    def prepare(self, buffers, numbers):
        """Behind the first call: what `step` compares.  buffers, numbers: tuples of everything that this was prepared from."""
        if self._native is None and all(t is None or type(t) is torch.Tensor for t in buffers):
            self._native = step_calls().Step(self._address, self._lru_address, self._tensors["centroids"], buffers,
                                             (*numbers, self.generation))

    def step(self, q, static_len, out_shape, buffers, numbers):
        """The call with a new output of out_shape, in native code; None, and nothing launched, where q is not what a prepared
        call reads or anything of buffers and numbers is not what it was prepared from."""
        if self._native is None or PROFILER_RANGES:
            return None
        out = self._native.run(q, static_len, out_shape, buffers, (*numbers, self._scratch.generation))
        if out.__class__ is int:
            check(out, "step")
        return out

    def run(self, q, static_len, out):
        status = self._call(self._address, q.data_ptr(), static_len, out.data_ptr(), _stream())
        if status:
            check(status, "decode_step")


class HostStepPlan(DecodeStepPlan):
    """The same over a host-resident store with the device-side block cache (ri_host_step).  `tensors` as above with the
    cache tensors as store_k / store_v; lru: DeviceLru of the layer; lists: as for its access_update; host_k, host_v
    [.., rows, 128] pinned; stage_row0: first staging row of the cache tensors."""

    def __init__(self, key, dtype, tensors, nprobe, es, page, max_pages, scale, lru, sizes, starts, lists, row_src, host_k,
                 host_v, stage_row0, scratch=None):
        rows = tensors["store_k"].numel() // (lru.BG * 128)
        tensors = dict(tensors, store_k=tensors["store_k"].view(lru.BG, rows, 128),
                       store_v=tensors["store_v"].view(lru.BG, rows, 128))
        super().__init__(key, dtype, tensors, nprobe, es, page, max_pages, scale, scratch)
        self._lru = lru.prepared(tensors["ret_ids"], sizes, starts, lists, row_src, stage_row0, tensors["meta"], host_k,
                                 host_v, tensors["store_k"], tensors["store_v"])
        self._lru_address = ctypes.addressof(self._lru)
        self._call = lib().ri_host_step

    def run(self, q, static_len, out):
        status = self._call(self._address, self._lru_address, q.data_ptr(), static_len, out.data_ptr(), _stream())
        if status:
            check(status, "host_step")


def append_row(key, value, steady_k, steady_v, pos, pos_dev, row_shape):
    """append_kv in native code where rows of row_shape and zones [batch, heads, rows, 128] are plain contiguous tensors of one
    type and device, with room for pos; else False, and nothing launched."""
    status = step_calls().append(key, value, steady_k, steady_v, pos, pos_dev, row_shape)
    if status:
        check(status, "append_kv")
    return status is not None


def append_kv(key, value, steady_k, steady_v, pos, pos_dev=None):
    """steady[g, pos] = row g of key / value [BG, 128] (any shape of BG * 128 elements), one launch for both."""
    stride = steady_k.shape[-2]
    status = lib().ri_append_kv(key.data_ptr(), value.data_ptr(), steady_k.data_ptr(), steady_v.data_ptr(), stride, pos,
                                _p(pos_dev), steady_k.numel() // (stride * 128), _stream())
    if status:
        check(status, "append_kv")


@_ranged("flash_attention")
def wave_attention_part(q, steady_k, steady_v, static_len, store_k, store_v, row_src, src_row_lo, src_row_hi, meta,
                        est_ids, logits, value_sum, cluster_size_bf16, out, lse_out, es, scale, prev_out=None,
                        prev_lse=None, valid_lengths=None, slot=0, scratch=None):
    """wave_attention over the rows of the row table whose source row lies in [src_row_lo, src_row_hi), merging an
    earlier part's (prev_out, prev_lse) and returning this part's log-sum-exp in lse_out [BG, gs] fp32."""
    BG, gs, D = q.shape
    nc = value_sum.shape[1]
    ws = _workspace(lib().ri_wave_attention_workspace_bytes(BG, gs), q.device, f"attn{slot}", scratch)
    check(_fn("ri_wave_attention_part", q.dtype)(
        _p(q), _p(steady_k), _p(steady_v), steady_k.shape[-2], static_len, None, _p(store_k), _p(store_v),
        store_k.shape[-2], _p(row_src), row_src.shape[1], int(src_row_lo), int(src_row_hi), _p(meta), _p(est_ids),
        _p(logits), _p(value_sum), _p(cluster_size_bf16), _p(prev_out), _p(prev_lse), _p(out), _p(lse_out),
        _p(valid_lengths), BG, gs, nc, es, float(scale), _p(ws), ws.numel(), _stream()), "wave_attention_part")


@_ranged("flash_attention")
def wave_attention_static(q, steady_k, steady_v, static_len, store_k, store_v, row_src, meta, est_ids, logits,
                          value_sum, cluster_size_bf16, out, valid_lengths, es, scale, ret_tok_off=None,
                          ret_start=None, est_centroids=None, static_len_dev=None):
    """wave_attention without a scratch tensor: the library keeps the scratch in a static device array
    (ri_wave_attention_static), so the call allocates nothing.  Calls on one GPU must not overlap."""
    BG, gs, D = q.shape
    nc = value_sum.shape[1]
    check(_fn("ri_wave_attention_static", q.dtype)(
        _p(q), _p(steady_k), _p(steady_v), steady_k.shape[-2], static_len, _p(static_len_dev), _p(store_k),
        _p(store_v), store_k.shape[-2], _p(row_src), 0 if row_src is None else row_src.shape[1], _p(ret_tok_off),
        _p(ret_start), 0 if ret_start is None else ret_start.shape[1], _p(meta), _p(est_ids), _p(logits),
        _p(est_centroids), _p(value_sum), _p(cluster_size_bf16), _p(out), _p(valid_lengths), BG, gs, nc, es,
        float(scale), _stream()), "wave_attention_static")


def buffer_attention(q, buf_k, buf_v, cache_seqlens, est_ids, logits, value_sum, cluster_size_bf16, out, es, scale,
                     slot=0, scratch=None):
    """Attention over the rows [0, cache_seqlens[g]) of an execution buffer [BG, stride, 128] with the
    estimation zone (ids and logits from score_select) merged in the same launch."""
    BG, gs, D = q.shape
    nc = value_sum.shape[1]
    stride = buf_k.shape[-3] if buf_k.dim() == 4 else buf_k.shape[-2]
    ws = _workspace(lib().ri_wave_attention_workspace_bytes(BG, gs), q.device, f"attn{slot}", scratch)
    check(_fn("ri_buffer_attention", q.dtype)(_p(q), _p(buf_k), _p(buf_v), stride, _p(cache_seqlens), stride, _p(est_ids),
                                    _p(logits), _p(value_sum), _p(cluster_size_bf16), _p(out), BG, gs, nc, es,
                                    float(scale), _p(ws), ws.numel(), _stream()), "buffer_attention")


class DeviceLru:
    """State of the device-side block cache manager of one layer (ri_lru_access_update)."""

    def __init__(self, BG, max_clusters, max_blocks, capacity, buffer_size, block, device):
        i32 = lambda *s: torch.zeros(s, dtype=torch.int32, device=device)
        self.BG, self.capacity, self.buffer_size, self.block = BG, capacity, buffer_size, block
        self.stamp = i32(BG, max_clusters)     # step that last touched a resident cluster (0: not resident)
        self.order = i32(BG, max_clusters)     # ... and the cluster's position inside that step
        self.blk_off = i32(BG, max_clusters + 1)
        self.blk_ids = i32(BG, max_blocks)
        self.free_list = torch.arange(capacity, dtype=torch.int32, device=device).repeat(BG, 1).contiguous()
        self.free_count = torch.full((BG,), capacity, dtype=torch.int32, device=device)
        self.epoch = i32(BG)

    def state(self):
        """The tensors whose addresses a prepared call holds."""
        return self.blk_off, self.stamp, self.order, self.blk_ids, self.free_list, self.free_count, self.epoch

    def set_sizes(self, sizes_i32):
        """sizes_i32 [BG, ncl]: recompute the block offsets (offsets of existing clusters do not move
        when clusters are appended)."""
        nb = (sizes_i32.to(torch.int64) + self.block - 1) // self.block
        ncl = sizes_i32.shape[1]
        self.blk_off[:, 1:ncl + 1] = torch.cumsum(nb, 1).to(torch.int32)
        assert int(self.blk_off[:, ncl].max()) <= self.blk_ids.shape[1]

    def access_update(self, ret_ids, sizes, starts, lists, row_src=None, stage_row0=0, meta=None):
        """lists: the 12 tensors hit (ids, sizes, cumsum, num), miss (...), update (buf, sizes, cache, num).
        row_src / meta: row table for attention in place (hits are then not listed for copying)."""
        BG, np_ = ret_ids.shape
        ncl = sizes.shape[1]
        check(lib().ri_lru_access_update(
            _p(ret_ids), _p(sizes), _p(starts), sizes.stride(0), _p(self.blk_off), self.blk_off.shape[1],
            _p(self.stamp), _p(self.order), self.stamp.shape[1], _p(self.blk_ids), self.blk_ids.shape[1], _p(self.free_list),
            _p(self.free_count), _p(self.epoch), *[_p(t) for t in lists], _p(row_src),
            0 if row_src is None else row_src.shape[1], stage_row0, _p(meta), BG, np_, ncl, self.buffer_size,
            self.capacity, self.block, _stream()), "lru_access_update")


    def prepared(self, ret_ids, sizes, starts, lists, row_src, stage_row0, meta, host_k, host_v, cache_k, cache_v):
        """The arguments of access_update and of the copy of the misses, host_k/v [.., rows, 128] to the staging rows of
        cache_k/v [BG, rows, 128], for ri_lru_access and ri_lru_stage_update."""
        names = [f"{a}_{b}" for a in ("hit", "miss") for b in ("ids", "sizes", "cumsum", "num")] + [
            "upd_buf", "upd_sizes", "upd_cache", "upd_num"]
        tensors = dict(zip(names, lists), ret_ids=ret_ids, sizes=sizes, starts=starts, blk_off=self.blk_off,
                       stamp=self.stamp, order=self.order, blk_ids=self.blk_ids, free_list=self.free_list,
                       free_count=self.free_count, epoch=self.epoch, row_src=row_src, meta=meta, host_k=host_k,
                       host_v=host_v, cache_k=cache_k, cache_v=cache_v)
        s = Lru(host_stride=host_k.shape[-2], cache_stride=cache_k.shape[-2], row_src_stride=row_src.shape[1],
                stage_row0=stage_row0, np=ret_ids.shape[1], ncl=sizes.shape[1], meta_stride=sizes.stride(0),
                blk_off_stride=self.blk_off.shape[1], stamp_stride=self.stamp.shape[1],
                blk_ids_stride=self.blk_ids.shape[1], buffer_size=self.buffer_size, capacity=self.capacity,
                block=self.block, BG=self.BG, **{nm: _p(t) for nm, t in tensors.items()})
        s.tensors = tensors   # (alive as long as their addresses are)
        return s


def kmeans_assign(data, centroids, assign, P, N, nc, seg, head_rows):
    check(_fn("ri_kmeans_assign", data.dtype)(_p(data), _p(centroids), _p(assign), P, N, nc, seg, head_rows, _stream()),
          "kmeans_assign")


def kmeans_build_lists(assign, counts, offsets, members, P, N, nc, slot=0):
    """`slot` names the scratch area: calls that may run concurrently (different streams) use different slots."""
    nb = lib().ri_kmeans_workspace_bytes(P, N, nc)
    ws = _workspace(nb, assign.device, f"kmeans{slot}")
    check(lib().ri_kmeans_build_lists(_p(assign), _p(counts), _p(offsets), _p(members), P, N, nc, _p(ws),
                                      ws.numel(), _stream()), "kmeans_build_lists")


def kmeans_update(data, counts, offsets, members, centroids, P, N, nc, seg, head_rows, normalize, slot=0):
    ws = _workspace(lib().ri_kmeans_reduce_workspace_bytes(P, N, nc), data.device, f"kmeans_reduce{slot}")
    check(_fn("ri_kmeans_update", data.dtype)(_p(data), _p(counts), _p(offsets), _p(members), _p(centroids), P, N, nc, seg,
                                 head_rows, int(bool(normalize)), _p(ws), ws.numel(), _stream()), "kmeans_update")


KMEANS_DIRECT_MAX_TOKENS = 16384   # ri_kmeans_update_direct: tokens per problem


def kmeans_update_direct(data, assign, centroids, P, N, nc, seg, head_rows, normalize, lists=None):
    """Lists and means in one launch; lists: (counts, offsets, members) to be written as well."""
    counts, offsets, members = lists or (None, None, None)
    check(_fn("ri_kmeans_update_direct", data.dtype)(_p(data), _p(assign), _p(centroids), _p(counts), _p(offsets),
                                                     _p(members), P, N, nc, seg, head_rows, int(bool(normalize)),
                                                     _stream()), "kmeans_update_direct")


def kmeans_lists_direct(assign, counts, offsets, members, P, N, nc):
    """The lists alone, for at most KMEANS_DIRECT_MAX_TOKENS tokens per problem."""
    check(lib().ri_kmeans_lists_direct(_p(assign), _p(counts), _p(offsets), _p(members), P, N, nc, _stream()),
          "kmeans_lists_direct")


def kmeans_iterate(data, centroids, assign, P, N, nc, seg, head_rows, updates, last):
    """`updates` rounds of kmeans_assign and a normalised update, then one more assignment if `last`."""
    nbytes = lib().ri_kmeans_iterate_workspace_bytes(P, N, nc)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=data.device)
    check(_fn("ri_kmeans_iterate", data.dtype)(_p(data), _p(centroids), _p(assign), P, N, nc, seg, head_rows, updates,
                                               int(bool(last)), _p(ws), nbytes, _stream()), "kmeans_iterate")


def _rows_ok(t):
    return t.stride(-1) == 1 and t.stride(-2) % 8 == 0 and t.stride(-3) % 8 == 0 and t.data_ptr() % 16 == 0


def aligned_rows(t):
    """t if its 128-element rows can be read 16 bytes at a time where they lie, else a contiguous copy."""
    return t if _rows_ok(t) else t.clone(memory_format=torch.contiguous_format)


def _row_strides(t, what):
    """Strides in elements of the two outer dimensions of [., ., 128] rows read 16 bytes at a time."""
    if not _rows_ok(t):
        raise ValueError(f"{what}: rows must be contiguous and 16-byte aligned")
    return t.stride(0), t.stride(1)


def kmeans_init(data, centroids, P, N, nc):
    check(lib().ri_kmeans_init(_p(data), _p(centroids), P, N, nc, _stream()), "kmeans_init")


def kmeans_value_sum(values, counts, offsets, members, value_sum, P, N, nc, slot=0, store=None, store_stride=0):
    """values [P, N, 128], strided or not; store: the cluster-contiguous value rows are written there as well."""
    ws = _workspace(lib().ri_kmeans_reduce_workspace_bytes(P, N, nc), values.device, f"kmeans_reduce{slot}")
    head, row = _row_strides(values, "kmeans_value_sum")
    check(_fn("ri_kmeans_value_rows", values.dtype)(_p(values), head, row, _p(counts), _p(offsets), _p(members),
                                                    _p(value_sum), _p(store), store_stride, P, N, nc, _p(ws), ws.numel(),
                                                    _stream()), "kmeans_value_sum")


def kmeans_store_makes_lists(P, N, nc):
    """Whether the stores are made from the assignment, with the lists, in one launch: short problems whose workgroups of eight
    clusters are resident at once, two to each of 256 compute units up to 12288 tokens, whose lists take 74 KB of LDS, and one to a
    unit past them (figures at km_store_direct_kernel)."""
    return N <= KMEANS_DIRECT_MAX_TOKENS and P * ((nc + 7) // 8) <= (512 if N <= 12288 else 256)


def kmeans_store_rows(values, keys, mean, counts, offsets, members, value_sum, centroids, value_store, key_store, P, N, nc,
                      store_stride, index=None, assign=None):
    """Value sums and means of the centred keys, with both stores; values/keys [P, N, 128], strided or not.
    index: (out, mask, size16, size, start) of prefill_index, filled as well.  assign (up to KMEANS_DIRECT_MAX_TOKENS tokens): the
    lists are made from it and written on the way."""
    vh, vr = _row_strides(values, "kmeans_store_rows")
    kh, kr = _row_strides(keys, "kmeans_store_rows")
    if not values.dtype == keys.dtype == mean.dtype == value_store.dtype == key_store.dtype:
        raise TypeError("kmeans_store_rows: values, keys and the stores must have the same element type")
    if assign is not None:
        check(_fn("ri_kmeans_store_direct", values.dtype)(
            _p(values), vh, vr, _p(keys), kh, kr, _p(mean), _p(assign), _p(counts), _p(offsets), _p(members), _p(value_sum),
            _p(centroids), _p(value_store), _p(key_store), store_stride, *(_p(t) for t in index or (None,) * 5), P, N, nc,
            _stream()), "kmeans_store_rows")
        return
    ws = _workspace(2 * lib().ri_kmeans_reduce_workspace_bytes(P, N, nc), values.device, "kmeans_store")
    fn = _fn("ri_kmeans_store_rows" if index is None else "ri_kmeans_store_index", values.dtype)
    check(fn(_p(values), vh, vr, _p(keys), kh, kr, _p(mean), _p(counts), _p(offsets), _p(members), _p(value_sum),
             _p(centroids), _p(value_store), _p(key_store), store_stride, *(_p(t) for t in index or ()), P, N, nc, _p(ws),
             ws.numel(), _stream()), "kmeans_store_rows")


def permute_rows_strided(src, members, dst, P, N, out_stride_rows):
    """permute_rows from [P, N, 128] rows with strides of their own."""
    head, row = _row_strides(src, "permute_rows")
    check(lib().ri_permute_rows_strided(_p(src), head, row, _p(members), _p(dst), P, N, out_stride_rows, _stream()),
          "permute_rows")


def prefill_mean(keys, first, N):
    """Mean [H, 1, 128] of keys[first:first + N] ([T, H, 128]) per head, the bits of torch.mean over the heads' own rows;
    None for shapes the kernel does not take."""
    H = keys.shape[1]
    nbytes = lib().ri_prefill_mean_workspace_bytes(H, N)
    if nbytes == 0:
        return None
    kr, kh = _row_strides(keys, "prefill_mean")
    if first + N > keys.shape[0]:
        raise ValueError("prefill_mean: rows outside the sequence")
    mean = torch.empty((H, 1, 128), dtype=keys.dtype, device=keys.device)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=keys.device)
    check(_fn("ri_prefill_mean", keys.dtype)(_p(keys), kr, kh, first, N, H, _p(mean), _p(ws), nbytes, _stream()),
          "prefill_mean")
    return mean


def prefill_split(keys, values, first, N, start0, n_start, end0, n_end, out, steady_k, steady_v, mean=None, centroids=None):
    """keys/values [T, H, 128]; out [H, N, 128], less mean [H, 1, 128] where given; steady_k/v [H, rows, 128].  centroids (with
    mean): [H, nc, 128], which kmeans_init of out would fill."""
    kr, kh = _row_strides(keys, "prefill_split")
    vr, vh = _row_strides(values, "prefill_split")
    T, H = keys.shape[0], keys.shape[1]
    if first + N > T or start0 + n_start > T or end0 + n_end > T or n_start + n_end > steady_k.shape[1]:
        raise ValueError("prefill_split: rows outside the sequence")
    if not keys.dtype == values.dtype == out.dtype == steady_k.dtype == steady_v.dtype:
        raise TypeError("prefill_split: keys, values and the cache must have the same element type")
    lead = (_p(keys), _p(values), kr, kh, vr, vh, first, N, start0, n_start, end0, n_end, H)
    tail = (_p(out), _p(steady_k), _p(steady_v), steady_k.stride(0) // 128, _stream())
    if mean is None:
        check(lib().ri_prefill_split(*lead, *tail), "prefill_split")
    elif centroids is not None:
        _need(centroids, keys.dtype, "centroids")
        check(_fn("ri_prefill_split_init", keys.dtype)(*lead, _p(mean), *tail[:-1], _p(centroids), centroids.shape[1], tail[-1]),
              "prefill_split")
    else:
        check(_fn("ri_prefill_split_centred", keys.dtype)(*lead, _p(mean), *tail), "prefill_split")


def prefill_center(keys, mean):
    H, N, _ = keys.shape
    check(_fn("ri_prefill_center", keys.dtype)(_p(keys), _p(mean), H, N, _stream()), "prefill_center")


def prefill_index(centroids, mean, counts, offsets, out, mask, size16, size, start):
    H, nc, _ = centroids.shape
    check(_fn("ri_prefill_index", centroids.dtype)(_p(centroids), _p(mean), _p(counts), _p(offsets), _p(out), _p(mask),
                                                   _p(size16), _p(size), _p(start), H, nc, _stream()), "prefill_index")


def permute_rows(src, members, dst, P, N, in_stride_rows, out_stride_rows):
    check(lib().ri_permute_rows(_p(src), _p(members), _p(dst), P, N, in_stride_rows, out_stride_rows, _stream()),
          "permute_rows")

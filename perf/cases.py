"""What a user of this package has it do, as measurable cases: decoded tokens over a wave-index cache (launched
call by call or replayed as a graph, K/V in device or in host memory), the prefill that builds the index, the
clustering by itself, and the operator surface that code written against `retroinfer_kernels` calls.

`listed()` gives the named cases, `draw(rng)` one more of the same ranges.  Index parameters follow from the context
length as in `synth.derive_config` (16 tokens per cluster, a segment per 8192 tokens, a retrieval zone of 1.8 % and an
estimation zone of 23.2 % of the clusters); shapes are those of the benchmark's configurations or generic."""
import math

import torch

from retrievalattention_amd import kernels, synth
from retrievalattention_amd.attn_hub import retroinfer_decode_attn
from retrievalattention_amd.cache_hub import retroinfer_cache
from retrievalattention_amd.cache_hub.kmeans import segment_k_means_csr

DIM = 128
STEADY = synth.STEADY_START + synth.STEADY_END
ESTIMATE = 0.232
DEVICE = "cuda:0"
TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one layer of one short sequence: the interactive single user, nothing to stream, launches and host work count
        dict(name="decode_small", kind="decode", dtype="bf16", batch=1, kv_heads=8, group=4, tokens=8192, budget=0.018,
             pad=0, generated=0),
        # the benchmark's headline shape: four long-context sequences, one layer of a decoded token
        dict(name="decode_batch", kind="decode", dtype="bf16", batch=4, kv_heads=8, group=4, tokens=131072,
             budget=0.018, pad=0, generated=0),
        # the largest decode: eight sequences of 256K tokens, eight query heads per KV head
        dict(name="decode_wide", kind="decode", dtype="bf16", batch=8, kv_heads=8, group=8, tokens=262144,
             budget=0.018, pad=0, generated=0),
        # sequences of unequal length (left padding), odd sizes, IEEE half, the 10 % retrieval budget of the throughput
        # harness, some tokens already generated
        dict(name="decode_ragged", kind="decode", dtype="fp16", batch=3, kv_heads=4, group=7, tokens=30011, budget=0.1,
             pad=4567, generated=37),
        # serving loops replay a captured token: layers of the headline shape ...
        dict(name="replay_batch", kind="replay", dtype="bf16", batch=4, kv_heads=8, group=4, tokens=131072,
             budget=0.018, layers=4),
        # ... and many layers over short contexts
        dict(name="replay_short", kind="replay", dtype="bf16", batch=2, kv_heads=8, group=4, tokens=16384, budget=0.018,
             layers=8),
        # clustered K/V in host memory behind the block cache: consecutive tokens whose queries drift, so that part of
        # each step's clusters has to cross the host link
        dict(name="host_drift", kind="host", dtype="bf16", batch=8, kv_heads=4, group=7, tokens=61440, budget=0.018,
             steps=6),
        # building the index of one sequence of one layer at the end of its prefill: short, long, ragged
        dict(name="prefill_short", kind="prefill", dtype="bf16", kv_heads=8, tokens=8192, pad=0),
        dict(name="prefill_long", kind="prefill", dtype="bf16", kv_heads=8, tokens=131072, pad=0),
        dict(name="prefill_ragged", kind="prefill", dtype="fp16", kv_heads=4, tokens=50021, pad=1234),
        # the clustering alone, every iteration over all centroids
        dict(name="kmeans_unsegmented", kind="kmeans", dtype="bf16", heads=8, tokens=131072, centroids=8192, segments=1),
        # the reference's operators in the order its own cache calls them, over an assembled execution buffer
        dict(name="operators", kind="operators", dtype="bf16", groups=32, group=4, clusters=8192, probes=147,
             estimated=1900, rows=4773),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "replay", "host", "prefill", "prefill", "kmeans", "operators"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    heads, group = rng.choice((1, 2, 4, 8)), rng.choice((1, 3, 4, 4, 7, 8, 12, 16))
    budget = rng.choice((0.018, 0.018, 0.1))
    if kind == "decode":
        tokens = _log(rng, 1500, 262144)
        batch = min(_log(rng, 1, 16), max(1, 64 * 262144 // (heads * tokens)))
        return dict(kind=kind, dtype=dtype, batch=batch, kv_heads=heads, group=group, tokens=tokens, budget=budget,
                    pad=rng.randrange(tokens // 8) if batch > 1 else 0, generated=rng.randrange(200))
    if kind == "replay":
        tokens = _log(rng, 1500, 131072)
        layers = rng.randrange(2, 9)
        batch = min(_log(rng, 1, 16), max(1, 128 * 131072 // (heads * tokens * layers)))
        return dict(kind=kind, dtype=dtype, batch=batch, kv_heads=heads, group=group, tokens=tokens, budget=budget,
                    layers=layers)
    if kind == "host":
        tokens = _log(rng, 4096, 65536)
        return dict(kind=kind, dtype=dtype, batch=_log(rng, 1, 8), kv_heads=rng.choice((1, 2, 4)), group=group,
                    tokens=tokens, budget=0.018, steps=rng.randrange(3, 8))
    if kind == "prefill":
        tokens = _log(rng, 1500, 131072)
        return dict(kind=kind, dtype=dtype, kv_heads=heads, tokens=tokens, pad=rng.randrange(tokens // 8))
    if kind == "kmeans":
        tokens = _log(rng, 2048, 131072)
        segments = rng.choice((1, 1, max(1, tokens // 8192)))
        per = max(1, int(tokens / rng.uniform(16, 48) / segments / 32))
        return dict(kind=kind, dtype=dtype, heads=heads, tokens=tokens, centroids=32 * per * segments,
                    segments=segments)
    clusters = 8 * _log(rng, 16, 2048)
    return dict(kind=kind, dtype=dtype, groups=_log(rng, 1, 64), group=group, clusters=clusters,
                probes=max(1, int(clusters * budget)), estimated=max(1, int(clusters * ESTIMATE)),
                rows=_log(rng, 80, 16384))


# ------------------------------------------------------------------------------------------------ inputs
def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEVICE)


def _sequence(gen, tokens, heads, dtype):
    """K and V [1, tokens, heads, 128] of one sequence: keys from a Gaussian mixture with one centre per 16 tokens and
    four outlier channels per head, as keys after rotary embedding show them; normal values."""
    centres = _normal(gen, heads, max(1, tokens // 16), DIM)
    noise = torch.full((heads, 1, DIM), 0.3, device=DEVICE)
    for h in range(heads):
        channels = torch.randperm(DIM, generator=gen, device=DEVICE)[:4]
        centres[h, :, channels] *= 8
        noise[h, :, channels] *= 8
    keys = torch.empty((1, tokens, heads, DIM), dtype=dtype, device=DEVICE)
    for h in range(heads):
        label = torch.randint(centres.shape[1], (tokens,), generator=gen, device=DEVICE)
        keys[0, :, h] = (centres[h, label] + noise[h] * _normal(gen, tokens, DIM)).to(dtype)
    return keys, _normal(gen, 1, tokens, heads, DIM).to(dtype)


def _cache(case, batch, layers, **options):
    """An empty cache for prompts of case["tokens"] clustered tokens (and the steady zone's) and up to 256 new ones."""
    index = synth.derive_config(case["tokens"], budget_ratio=case.get("budget", 0.018), estimate_ratio=ESTIMATE)
    context, new = case["tokens"] + STEADY, 256
    pads = [0] * (batch - 1) + [case.get("pad", 0)]
    return retroinfer_cache(
        pads, layers, batch, context + new, case["kv_heads"], case["kv_heads"] * case.get("group", 4), DIM,
        TYPES[case["dtype"]], {str(layer): DEVICE for layer in range(layers)}, new, index["static_pattern_start"],
        index["static_pattern_end"], 4, index["n_centroids"], index["n_segment"], index["nprobe"],
        index["max_compute_cluster_num"], index["cache_unit_size"], index["cache_cluster_num"], 1, 0, **options)


def _decoding(case, gen, layers, **options):
    """A cache of `layers` prefilled layers and the new token's inputs for each of them.  The cache has one layer more:
    the last layer's call is what moves a sequence on to its next token, so passes over the layers before it repeat
    the same token, as a measurement has to."""
    batch, heads, group = case["batch"], case["kv_heads"], case["group"]
    dtype = TYPES[case["dtype"]]
    cache = _cache(case, batch, layers + 1, **options)
    for layer in range(layers):
        for b in range(batch):
            k, v = _sequence(gen, case["tokens"] + STEADY, heads, dtype)
            cache.prefill_update_kv_cache(None, k, v, layer, b)
            cache.sync(layer, b)
    cache.prepare_cache()
    for _ in range(case.get("generated", 0)):
        row = _normal(gen, 2, batch, 1, heads, DIM).to(dtype)
        for layer in range(layers + 1):
            cache.decode_update_kv_cache(row[0], row[1], layer)
    q = [_normal(gen, batch, 1, heads * group, DIM).to(dtype) for _ in range(layers)]
    k = [_normal(gen, batch, 1, heads, DIM).to(dtype) for _ in range(layers)]
    v = [_normal(gen, batch, 1, heads, DIM).to(dtype) for _ in range(layers)]
    return cache, q, k, v


def _step(cache, q, k, v, layer):
    """One layer of one decoded token, as a model's layer calls it: append the token's K/V, attend."""
    cache.decode_update_kv_cache(k, v, layer)
    return retroinfer_decode_attn(q, None, None, layer, cache)


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    state = {"kind": kind, "case": case}
    if kind == "decode":
        state["cache"], state["q"], state["k"], state["v"] = _decoding(case, gen, 1, kv_residency="device")
    elif kind == "replay":
        # the captured token: one eager pass first (scratch areas reach their size), then the capture
        layers = case["layers"]
        cache, q, k, v = _decoding(case, gen, layers, kv_residency="device", device_positions=True)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for layer in range(layers):
                _step(cache, q[layer], k[layer], v[layer], layer)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["out"] = [_step(cache, q[layer], k[layer], v[layer], layer) for layer in range(layers)]
        state.update(cache=cache, q=q, k=k, v=v, graph=graph)
    elif kind == "host":
        cache, q, k, v = _decoding(case, gen, 1, kv_residency="host")
        drift = [q[0] + 0.75 * _normal(gen, *q[0].shape) for _ in range(case["steps"])]
        state.update(cache=cache, q=[x.to(q[0].dtype) for x in drift], k=k, v=v)
    elif kind == "prefill":
        state["cache"] = _cache(case, 1, 1, kv_residency="device")
        state["k"], state["v"] = _sequence(gen, case["tokens"] + STEADY, case["kv_heads"], TYPES[case["dtype"]])
    elif kind == "kmeans":
        k, v = _sequence(gen, case["tokens"], case["heads"], TYPES[case["dtype"]])
        k = k[0].transpose(0, 1)
        state["k"] = (k - k.float().mean(dim=1, keepdim=True).to(k.dtype)).contiguous()
        state["v"] = v[0].transpose(0, 1).contiguous()
    else:
        state.update(_operator_inputs(case, gen))
    return state


def _operator_inputs(case, gen):
    groups, group, n, rows = case["groups"], case["group"], case["clusters"], case["rows"]
    dtype = TYPES[case["dtype"]]
    probes, estimated = case["probes"], case["estimated"]
    size = torch.randint(1, 33, (groups, n), generator=gen, device=DEVICE)
    empty = lambda *shape, dt=dtype: torch.empty(shape, dtype=dt, device=DEVICE)  # noqa: E731
    tiles = (n + 255) // 256
    return dict(
        q=_normal(gen, groups, 1, group, DIM).to(dtype), centroids=_normal(gen, groups, n, DIM).to(dtype),
        value_sum=(_normal(gen, groups, n, DIM) * size[..., None].sqrt()).to(dtype), size=size.to(dtype),
        ids=torch.rand((groups, n), generator=gen, device=DEVICE).argsort(dim=1)[:, :probes + estimated].contiguous(),
        keys=_normal(gen, groups, rows, 1, DIM).to(dtype), values=_normal(gen, groups, rows, 1, DIM).to(dtype),
        lengths=torch.randint(rows // 2, rows + 1, (groups,), generator=gen, device=DEVICE, dtype=torch.int32),
        product=empty(groups, group, n), softmax=empty(groups, group, n),
        norm=empty(groups, tiles, group, dt=torch.float32), sum=empty(groups, tiles, group, dt=torch.float32),
        es_keys=empty(groups, estimated, 1, DIM), es_values=empty(groups, estimated, 1, DIM),
        es_size=empty(groups, 1, 1, estimated))


# ------------------------------------------------------------------------------------------------ passes
def run(state):
    kind = state["kind"]
    if kind == "replay":
        state["graph"].replay()
        layers = slice(0, state["case"]["layers"])
        return {"out": state["out"], "steady_keys": state["cache"].steady_zone_keys[layers],
                "steady_values": state["cache"].steady_zone_values[layers]}
    if kind in ("decode", "host"):
        cache = state["cache"]
        out = [_step(cache, q, state["k"][0], state["v"][0], 0) for q in state["q"]]
        return {"out": out, "steady_keys": cache.steady_zone_keys[0], "steady_values": cache.steady_zone_values[0]}
    if kind == "prefill":
        cache = state["cache"]
        k, v = cache.prefill_update_kv_cache(None, state["k"], state["v"], 0, 0)
        cache.sync(0, 0)
        return {"k": k, "v": v, "centroids": cache.centroids[0], "value_sum": cache.value_sum[0],
                "size": cache.cluster_size[0], "size_i32": cache.cluster_size_i32[0], "start": cache.cluster_start[0],
                "mask": cache.centroids_mask[0], "steady_keys": cache.steady_zone_keys[0],
                "steady_values": cache.steady_zone_values[0], "store_keys": cache.list_keys[0],
                "store_values": cache.list_values[0]}
    if kind == "kmeans":
        r = segment_k_means_csr(state["k"], state["v"], state["case"]["centroids"], 10, state["case"]["segments"])
        return {"centroids": r.centroids, "value_sum": r.value_sum, "assign": r.assign, "counts": r.counts,
                "offsets": r.offsets, "members": r.members}
    return _operators(state)


def _operators(s):
    case = s["case"]
    groups, group, n, estimated = case["groups"], case["group"], case["clusters"], case["estimated"]
    kernels.batch_gemm_softmax(s["q"], s["centroids"], s["product"], s["norm"], s["sum"], s["softmax"], groups, group, n,
                               DIM, 1.0 / math.sqrt(DIM))
    kernels.gather_copy_vectors(s["centroids"], s["es_keys"], s["value_sum"], s["es_values"], s["size"], s["es_size"],
                                s["ids"], groups, n, estimated, s["ids"].shape[1], case["probes"], estimated)
    es_out, es_lse = kernels.weighted_flash_decoding(s["q"], s["es_keys"], s["es_values"], s["es_size"],
                                                     return_softmax_lse=True)
    out = kernels.weighted_flash_decoding(s["q"], s["keys"], s["values"], previous_out=es_out, previous_lse=es_lse,
                                          cache_seqlens=s["lengths"])
    return {"product": s["product"], "softmax": s["softmax"], "es_keys": s["es_keys"], "es_values": s["es_values"],
            "es_size": s["es_size"], "es_out": es_out, "es_lse": es_lse, "out": out}


# ------------------------------------------------------------------------------------------------ accounting
def work(case):
    kind, row = case["kind"], DIM * 2
    if kind in ("decode", "replay", "host"):
        index = synth.derive_config(case["tokens"], budget_ratio=case["budget"], estimate_ratio=ESTIMATE)
        n, probes = index["n_centroids"], index["nprobe"]
        estimated = index["max_compute_cluster_num"] - probes
        groups, group = case["batch"] * case["kv_heads"], case["group"]
        clustered = case["tokens"] - case.get("pad", 0) / case["batch"]
        attended = probes * clustered / n + STEADY + case.get("generated", 0) + 1
        # centroids, mask and query; value sums and sizes of the estimation zone; K and V of the attended tokens;
        # the appended rows; the output
        bytes_ = groups * (n * (row + 1) + group * row + estimated * (row + 2) + attended * 2 * row + 2 * 2 * row +
                           group * row)
        flops = groups * group * 2 * DIM * (n + estimated + 2 * attended)
        times = case.get("layers", 1) * case.get("steps", 1)
        return {"bytes": bytes_ * times, "flops": flops * times}
    if kind == "prefill":
        index = synth.derive_config(case["tokens"])
        heads, n = case["kv_heads"], index["n_centroids"]
        clustered = case["tokens"] - case["pad"]
        # K and V in, the same rows out in cluster order; per cluster two vectors, two sizes, a start and a flag
        return {"bytes": heads * (4 * (clustered + STEADY) * row + n * (2 * row + 11)),
                "flops": heads * 2 * DIM * clustered * (9 * n / index["n_segment"] + n)}
    if kind == "kmeans":
        heads, tokens, n = case["heads"], case["tokens"], case["centroids"]
        return {"bytes": heads * (2 * tokens * row + n * (2 * row + 8) + tokens * 8),
                "flops": heads * 2 * DIM * tokens * (9 * n / case["segments"] + n)}
    groups, group, n, estimated = case["groups"], case["group"], case["clusters"], case["estimated"]
    attended = 0.75 * case["rows"]
    # scores and their softmax out; estimation rows gathered (in, out) and attended; the execution buffer attended
    return {"bytes": groups * (n * row + 2 * group * n * 2 + estimated * (4 * row + 12) + attended * 2 * row +
                               3 * group * row),
            "flops": groups * group * 2 * DIM * (n + 2 * estimated + 2 * attended)}


def tolerance(case):
    # the clustering is defined to the bit (fixed summation order, ascending lists, ties to the lower id), and the store
    # is a copy of the inputs' rows; attention outputs are 16-bit values of sums with 16-bit probabilities
    return "exact" if case["kind"] in ("prefill", "kmeans") else {"rel": 1e-2}

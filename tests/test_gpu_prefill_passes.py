"""The passes around the prefill clustering against torch, bit for bit: heads taken apart, keys centred, initial
centroids, value rows summed and stored, index entries (GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,N,nc,fused", [(1, 1, 32, False), (2, 63, 32, True), (3, 65, 64, False), (8, 1000, 96, True),
                                          (2, 20001, 1088, False)])
def test_prefill_passes(dev, dtype, H, N, nc, fused):
    from retrievalattention_amd import kernels
    from retrievalattention_amd.cache_hub.kmeans import init_centroid_indices
    g = torch.Generator().manual_seed(H * N + nc)
    vs, sps, spe = 5, 3, 17
    T = vs + sps + N + spe
    if fused:      # keys and values as slices of one projection: rows further apart than their heads fill
        kv = torch.randn(T, 2, H, 128, generator=g).to(dtype).to(dev)
        K, V = kv[:, 0], kv[:, 1]
    else:
        K, V = (torch.randn(T, H, 128, generator=g).to(dtype).to(dev) for _ in range(2))
    lo = vs + sps
    hk, hv = K[lo:lo + N].transpose(0, 1), V[lo:lo + N].transpose(0, 1)
    ck = torch.empty((H, N, 128), dtype=dtype, device=dev)
    zk, zv = (torch.zeros((H, sps + spe + 2, 128), dtype=dtype, device=dev) for _ in range(2))
    kernels.prefill_split(K, V, lo, N, vs, sps, lo + N, spe, ck, zk, zv)
    assert torch.equal(ck, hk)
    for z, src in ((zk, K), (zv, V)):
        ref = torch.cat((src[vs:lo], src[lo + N:], torch.zeros_like(src[:2])))
        assert torch.equal(z, ref.transpose(0, 1))

    mean = torch.mean(ck, dim=1, keepdim=True)
    centred = ck - mean
    kernels.prefill_center(ck, mean)
    assert torch.equal(ck, centred)

    cent = torch.empty((H, nc, 128), dtype=dtype, device=dev)
    kernels.kmeans_init(ck, cent, H, N, nc)
    assert torch.equal(cent, ck[:, init_centroid_indices(N, nc, dev)])

    assign = torch.randint(0, nc - 1, (H, N), generator=g, dtype=torch.int32)      # the last cluster stays empty
    assign[:, : N // 2] = 3                                                        # one list beyond a block of sums
    assign = assign.to(dev)
    counts, offsets, members = (torch.empty(s, dtype=torch.int32, device=dev) for s in ((H, nc), (H, nc + 1), (H, N)))
    kernels.kmeans_build_lists(assign, counts, offsets, members, H, N, nc)
    if N <= kernels.KMEANS_DIRECT_MAX_TOKENS:
        lists = [torch.full_like(t, -1) for t in (counts, offsets, members)]
        kernels.kmeans_lists_direct(assign, *lists, H, N, nc)
        assert all(torch.equal(a, b) for a, b in zip(lists, (counts, offsets, members)))
    sums, ref_sums = (torch.empty((H, nc, 128), dtype=dtype, device=dev) for _ in range(2))
    store, store_k = (torch.zeros((H, N + 7, 128), dtype=dtype, device=dev) for _ in range(2))
    kernels.kmeans_value_sum(hv.contiguous(), counts, offsets, members, ref_sums, H, N, nc)
    kernels.kmeans_value_sum(hv, counts, offsets, members, sums, H, N, nc, store=store, store_stride=N + 7)
    kernels.permute_rows_strided(hk, members, store_k, H, N, N + 7)
    at = members.long()[:, :, None].expand(-1, -1, 128)
    assert torch.equal(sums, ref_sums)
    for st, src in ((store, hv), (store_k, hk)):
        assert torch.equal(st[:, :N], torch.gather(src, 1, at)) and not st[:, N:].any()

    # sums, means and both stores in one pass against the passes by themselves
    means, both = cent.clone(), cent.clone()
    kernels.kmeans_update(ck, counts, offsets, members, means, H, N, nc, 1, N, False)
    sums.zero_()
    stores = [torch.zeros_like(store) for _ in range(2)]
    kernels.kmeans_store_rows(hv, hk, mean, counts, offsets, members, sums, both, *stores, H, N, nc, N + 7)
    assert torch.equal(both, means) and torch.equal(sums, ref_sums)
    assert torch.equal(stores[0], store) and torch.equal(stores[1], store_k)

    out, mask = torch.empty_like(cent), torch.empty((H, nc), dtype=torch.bool, device=dev)
    size16, size, start = torch.empty((H, nc), dtype=dtype, device=dev), torch.empty_like(counts), torch.empty_like(counts)
    kernels.prefill_index(cent, mean, counts, offsets, out, mask, size16, size, start)
    assert torch.equal(out, cent + mean) and torch.equal(mask, counts == 0) and torch.equal(size16, counts.to(dtype))
    assert torch.equal(size, counts) and torch.equal(start, offsets[:, :nc])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,N,nc", [(1, 1, 32), (3, 257, 64), (8, 1000, 96), (2, 20001, 1088)])
def test_index_entries_on_the_way_to_the_stores(dev, dtype, H, N, nc):
    """The entries that the stores' launches fill are those of the finished means: of short lists, of long ones, whose
    means are folded later, and of empty clusters, which keep their centroids."""
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(H * N + nc)
    rows = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)
    K, V, mean, cent = rows(N, H, 128), rows(N, H, 128), rows(H, 1, 128), rows(H, nc, 128)
    hk, hv = K.transpose(0, 1), V.transpose(0, 1)
    assign = torch.randint(0, nc - 1, (H, N), generator=g, dtype=torch.int32)
    assign[:, : N // 2] = 3
    assign = assign.to(dev)
    counts, offsets, members = (torch.empty(s, dtype=torch.int32, device=dev) for s in ((H, nc), (H, nc + 1), (H, N)))
    kernels.kmeans_build_lists(assign, counts, offsets, members, H, N, nc)

    def stored(**options):
        means, sums = cent.clone(), torch.zeros_like(cent)
        stores = [torch.zeros((H, N + 7, 128), dtype=dtype, device=dev) for _ in range(2)]
        kernels.kmeans_store_rows(hv, hk, mean, counts, offsets, members, sums, means, *stores, H, N, nc, N + 7, **options)
        return means, sums, *stores

    def entries():
        return (torch.zeros_like(cent), torch.zeros((H, nc), dtype=torch.bool, device=dev),
                torch.zeros((H, nc), dtype=dtype, device=dev), torch.zeros_like(counts), torch.zeros_like(counts))

    apart, filled = entries(), entries()
    plain = stored()
    kernels.prefill_index(plain[0], mean, counts, offsets, *apart)
    assert all(torch.equal(a, b) for a, b in zip(stored(index=filled), plain))
    assert all(torch.equal(a, b) for a, b in zip(filled, apart))
    assert torch.equal(filled[0], plain[0] + mean) and torch.equal(filled[1], counts == 0)


# Lists made in the launch that stores their rows: problems of fewer tokens than a load takes, lists of one block, of just more and
# of a whole problem, last workgroups of few clusters, the most tokens; rows with strides of their own.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,N,nc", [(1, 1, 32), (3, 3, 32), (2, 255, 32), (8, 1000, 96), (3, 2051, 128), (8, 8191, 512), (16, 8192, 512),
                                    (5, 16383, 1024), (33, 2000, 540), (2, 16384, 32)])
@pytest.mark.parametrize("kind", ["even", "blocks", "one"])
def test_stores_that_make_the_lists(dev, dtype, H, N, nc, kind):
    """The lists of ri_kmeans_lists_direct, and over them what the launches that take lists write, bit for bit."""
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(H * N + nc)
    rows = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)
    kv, mean, cent = rows(N, 2, H, 128), rows(H, 1, 128), rows(H, nc, 128)
    hk, hv = kv[:, 0].transpose(0, 1), kv[:, 1].transpose(0, 1)
    assign = torch.randint(0, nc - 1, (H, N), generator=g, dtype=torch.int32)
    if kind == "blocks":   # lists of 256 and 257 tokens, and one of several blocks in the same workgroup's clusters
        for first, last, c in ((0, 256, nc - 1), (256, 513, 2), (513, 1400, 5), (1400, 2800, 6)):
            assign[:, first:last] = c
    elif kind == "one":
        assign[:] = nc - 2
    assign = assign[:, torch.randperm(N, generator=g)].contiguous().to(dev)

    def stored(index, made):
        lists = [torch.full(s, -1, dtype=torch.int32, device=dev) for s in ((H, nc), (H, nc + 1), (H, N))]
        if not made:
            kernels.kmeans_lists_direct(assign, *lists, H, N, nc)
        means, sums = cent.clone(), torch.full_like(cent, 7)
        stores = [torch.zeros((H, N + 7, 128), dtype=dtype, device=dev) for _ in range(2)]
        entries = (torch.zeros_like(cent), torch.zeros((H, nc), dtype=torch.bool, device=dev),
                   torch.zeros((H, nc), dtype=dtype, device=dev), torch.zeros_like(lists[0]), torch.zeros_like(lists[0]))
        kernels.kmeans_store_rows(hv, hk, mean, *lists, sums, means, *stores, H, N, nc, N + 7, entries if index else None,
                                  assign if made else None)
        return (*lists, means, sums, *stores, *entries)

    for index in (True, False):
        assert all(torch.equal(a, b) for a, b in zip(stored(index, True), stored(index, False)))


@pytest.mark.parametrize("N,nc", [(2000, 128), (20000, 128)])
def test_clustering_fills_the_index_with_stores_or_without(dev, N, nc):
    """The index entries that a clustering is handed hold the same, whether it writes the stores as well or not."""
    from retrievalattention_amd.cache_hub.kmeans import segment_k_means_csr
    H, dtype = 2, torch.bfloat16
    g = torch.Generator().manual_seed(N)
    rows = [torch.randn(H, N, 128, generator=g).to(dtype).to(dev) for _ in range(2)]
    mean = rows[0].float().mean(dim=1, keepdim=True).to(dtype)
    got = []
    for stores in (True, False):
        entries = (torch.full((H, nc, 128), 7, dtype=dtype, device=dev), torch.ones((H, nc), dtype=torch.bool, device=dev),
                   *(torch.full((H, nc), -1, dtype=t, device=dev) for t in (dtype, torch.int32, torch.int32)))
        more = dict(key_rows=rows[0], key_store=torch.empty_like(rows[0]), value_store=torch.empty_like(rows[1]),
                    store_stride=N) if stores else {}
        r = segment_k_means_csr(rows[0] - mean, rows[1], nc, 3, key_mean=mean, index=entries, **more)
        assert torch.equal(entries[0], r.centroids + mean) and torch.equal(entries[3], r.counts)
        assert torch.equal(entries[4], r.offsets[:, :-1])
        got.append(entries)
    assert all(torch.equal(a, b) for a, b in zip(*got))


# where the order of the sum changes (one part, four, eight, sixteen ...; one head has a rule of its own), and around it
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,N", [(1, 1), (1, 1020), (1, 1021), (1, 8193), (1, 16384), (1, 16385), (1, 40007), (2, 3),
                                 (2, 510), (3, 511), (8, 4094), (5, 4095), (4, 32752), (2, 32753), (8, 65504), (2, 65505),
                                 (32, 2049), (1, 262144), (2, 131009), (2, 262144)])
def test_prefill_mean(dev, dtype, H, N):
    from retrievalattention_amd import kernels
    g = torch.Generator(device=dev).manual_seed(H + N)
    vs, sps, spe = 5, 3, 17
    T = vs + sps + N + spe
    kv = torch.randn(T, 2, H, 128, generator=g, device=dev)
    kv = (kv + 0.1) * torch.where(torch.arange(128, device=dev) < 4, 8.0, 1.0)
    kv = (kv * (2.0 ** -15 if N % 3 == 0 else 1.0)).to(dtype)      # (halves below the smallest normal one)
    K, V = (kv[:, 0], kv[:, 1]) if N % 2 else (kv[:, 0].contiguous(), kv[:, 1].contiguous())
    lo = vs + sps
    ck, ref = (torch.empty((H, N, 128), dtype=dtype, device=dev) for _ in range(2))
    zones = [torch.zeros((H, sps + spe, 128), dtype=dtype, device=dev) for _ in range(4)]
    kernels.prefill_split(K, V, lo, N, vs, sps, lo + N, spe, ref, *zones[:2])
    mean = kernels.prefill_mean(K, lo, N)
    assert torch.equal(mean, torch.mean(ref, dim=1, keepdim=True))
    kernels.prefill_center(ref, mean)
    kernels.prefill_split(K, V, lo, N, vs, sps, lo + N, spe, ck, *zones[2:], mean)
    assert torch.equal(ck, ref) and torch.equal(zones[0], zones[2]) and torch.equal(zones[1], zones[3])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,N,nc", [(1, 32, 32), (3, 100, 32), (2, 1000, 41), (8, 4099, 256), (1, 7, 33), (4, 50021, 3072)])
def test_initial_centroids_come_with_the_split(dev, dtype, H, N, nc):
    """What the split writes for the centroids are the rows that kmeans_init takes of the centred keys, and everything else is as
    without them: whole and partial workgroups of centroids, more centroids than rows."""
    from retrievalattention_amd import kernels
    g = torch.Generator(device=dev).manual_seed(N)
    vs, sps, spe = 3, 4, 20
    K, V = torch.randn(2, vs + sps + N + spe, H, 128, generator=g, device=dev).to(dtype)
    lo, mean = vs + sps, torch.randn(H, 1, 128, generator=g, device=dev).to(dtype)
    keys = [torch.empty((H, N, 128), dtype=dtype, device=dev) for _ in range(2)]
    zones = [torch.zeros((H, sps + spe, 128), dtype=dtype, device=dev) for _ in range(4)]
    cent = [torch.zeros((H, nc + 1, 128), dtype=dtype, device=dev)[:, :nc].contiguous() for _ in range(2)]
    kernels.prefill_split(K, V, lo, N, vs, sps, lo + N, spe, keys[0], *zones[:2], mean)
    kernels.kmeans_init(keys[0], cent[0], H, N, nc)
    kernels.prefill_split(K, V, lo, N, vs, sps, lo + N, spe, keys[1], *zones[2:], mean, cent[1])
    assert torch.equal(keys[0], keys[1]) and torch.equal(zones[0], zones[2]) and torch.equal(zones[1], zones[3])
    assert torch.equal(cent[0], cent[1])


def test_prefill_mean_leaves_other_shapes(dev):
    from retrievalattention_amd import kernels
    assert kernels.prefill_mean(torch.empty((40, 33, 128), dtype=torch.bfloat16, device=dev), 0, 40) is None
    assert kernels.prefill_mean(torch.empty((262145, 1, 128), dtype=torch.bfloat16, device=dev), 0, 262145) is None


@pytest.mark.parametrize("residency", ["device", "host-cpu"])
def test_captured_clusterings_serve_the_caches_that_follow(dev, residency):
    """Layers of two caches in a row, launched, captured and replayed, with initial centroids in the captured clustering's own
    tensor, against prefills of which each is launched kernel by kernel."""
    from retrievalattention_amd.cache_hub import kmeans
    from tests.test_gpu_cache import _gen, _make_cache
    layers, ctx = 3, 2500 + 68
    K, V = _gen(layers, 2, 2, 4, ctx, 64, dev, 3)

    def prefilled(b, captured):
        cache = _make_cache(dev, residency, layers, 1, 2, 4, ctx, 96, 1, 8, 16)
        for layer in range(layers):
            if not captured:
                kmeans._GRAPHS.clear(), kmeans._SEEN.clear()
            cache.prefill_update_kv_cache(None, K[layer][b], V[layer][b], layer, 0)
            cache.sync(layer, 0)
        torch.cuda.synchronize()
        if residency != "device":
            cache.prepare_cache()
        return [[x[layer].clone() for x in (cache.centroids, cache.value_sum, cache.cluster_size_i32, cache.cluster_start,
                                            cache.list_keys, cache.list_values)] for layer in range(layers)]
    kmeans._GRAPHS.clear(), kmeans._SEEN.clear()
    for b in range(2):
        for got, want in zip(prefilled(b, True), prefilled(b, False)):
            rows = int(want[2][0].sum())
            for x, y in zip(got, want):
                x, y = (t[..., :rows, :] if t.dim() == 4 else t for t in (x, y))
                assert torch.equal(x, y)

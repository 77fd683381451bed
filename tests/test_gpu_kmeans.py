"""K-means kernels against the oracle (GPU).

Assignment scores come out of the matrix cores, whose accumulation order differs from any CPU
sum, so a token may legitimately land on the runner-up centroid when the two best scores are
closer than fp32 rounding noise; the test accepts exactly that and nothing else.  Everything
downstream of the assignment (lists, sums, means, normalisation, value sums) is bit-exact."""
import numpy as np
import pytest
import torch

from oracle import kmeans as okm

pytestmark = pytest.mark.gpu


def _mixture(G, N, K, seed, sigma=0.3, dt=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    centers = torch.randn(G, K, 128, generator=g)
    a = torch.randint(K, (G, N), generator=g)
    keys = torch.gather(centers, 1, a[..., None].expand(G, N, 128)) + sigma * torch.randn(G, N, 128, generator=g)
    vals = torch.randn(G, N, 128, generator=g)
    return keys.to(dt), vals.to(dt)


def _check_assign(data, cent, got):
    """got must be the oracle's argmax, or a centroid whose fp64 score is within fp32 noise of it."""
    a, best, _ = okm.assign(data, cent)
    got = got.astype(np.int64)
    diff = np.nonzero(a != got)[0]
    if diff.size:
        s = (data[diff].double().numpy() * cent[got[diff]].double().numpy()).sum(1)
        scale = np.abs(data[diff].double().numpy()).sum(1) * np.abs(cent.double().numpy()).max()
        assert np.all(best[diff] - s <= 1e-6 * np.maximum(scale, 1.0)), "assignment differs beyond a near-tie"
    return diff.size


@pytest.mark.parametrize("P,N,nc,seed", [(3, 1000, 64, 0), (2, 8192, 512, 1), (1, 4100, 1024, 2), (4, 37, 32, 3)])
def test_assign_update_valuesum(dev, P, N, nc, seed, dt=torch.bfloat16):
    from retrievalattention_amd import kernels
    keys, vals = _mixture(P, N, nc, seed, dt=dt)
    idx = okm.init_indices(N, nc)
    cent = keys[:, idx].contiguous()
    kd, vd, cd = keys.to(dev), vals.to(dev), cent.to(dev).clone()
    assign = torch.empty(P, N, dtype=torch.int32, device=dev)
    counts = torch.empty(P, nc, dtype=torch.int32, device=dev)
    offsets = torch.empty(P, nc + 1, dtype=torch.int32, device=dev)
    members = torch.empty(P, N, dtype=torch.int32, device=dev)
    vsum = torch.empty(P, nc, 128, dtype=dt, device=dev)
    kernels.kmeans_assign(kd, cd, assign, P, N, nc, 1, N)
    kernels.kmeans_build_lists(assign, counts, offsets, members, P, N, nc)
    cn = cd.clone()
    kernels.kmeans_update(kd, counts, offsets, members, cn, P, N, nc, 1, N, True)
    cu = cd.clone()
    kernels.kmeans_update(kd, counts, offsets, members, cu, P, N, nc, 1, N, False)
    kernels.kmeans_value_sum(vd, counts, offsets, members, vsum, P, N, nc)
    torch.cuda.synchronize()
    A = assign.cpu().numpy()
    for p in range(P):
        _check_assign(keys[p], cent[p], A[p])
        # lists: counts, offsets and ascending members of the kernel's own assignment
        lists, cnt = okm.reverse_index(A[p].astype(np.int64), nc)
        assert np.array_equal(counts[p].cpu().numpy(), cnt)
        off = offsets[p].cpu().numpy()
        assert off[0] == 0 and np.array_equal(np.diff(off), cnt)
        mem = members[p].cpu().numpy()
        for c in range(nc):
            assert np.array_equal(mem[off[c]:off[c + 1]], lists[c, :cnt[c]])
        # sums / means / normalisation given that assignment: bit-exact
        s, cnt2 = okm.cluster_sums(keys[p], A[p].astype(np.int64), nc)
        assert torch.equal(cn[p].cpu(), okm.update(cent[p], s, cnt2, True))
        assert torch.equal(cu[p].cpu(), okm.update(cent[p], s, cnt2, False))
        assert torch.equal(vsum[p].cpu(), okm.value_sum(vals[p], A[p].astype(np.int64), nc))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("P,N,nc", [(5, 1001, 32), (8, 8193, 544), (16, 8200, 544), (20, 9757, 608), (33, 8200, 512),
                                    (3, 100000, 1056), (4, 65500, 1056)])
def test_assign_tilings(dev, P, N, nc, dt):
    """One size for every tiling of the assignment, with a remainder of tokens and of centroids."""
    from retrievalattention_amd import kernels
    g = torch.Generator(device=dev).manual_seed(N)
    data = torch.randn(P, N, 128, generator=g, device=dev).to(dt)
    cent = torch.nn.functional.normalize(torch.randn(P, nc, 128, generator=g, device=dev), dim=-1).to(dt)
    assign = torch.full((P, N), -1, dtype=torch.int32, device=dev)
    kernels.kmeans_assign(data, cent, assign, P, N, nc, 1, N)
    for p in range(P):
        s = data[p].double() @ cent[p].double().T
        best, at = s.max(dim=1)
        mine = s.gather(1, assign[p].long()[:, None])[:, 0]
        assert bool((best - mine <= 1e-5).all())            # (fp32 sums of products may swap near-ties)
        assert float((at != assign[p]).float().mean()) < 1e-3


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("P,N,nc", [(5, 1001, 32), (8, 8193, 544), (16, 8200, 544), (20, 9757, 608), (33, 8200, 512),
                                    (3, 100000, 1056)])
def test_assign_ties_go_to_the_lowest_id(dev, P, N, nc, dt):
    """Small whole numbers: every score is exact in fp32, and every centroid appears again four rows on (the other half
    of the wave), 32 rows on (the next sub-tile) or in place of one before it, so that most maxima are tied."""
    from retrievalattention_amd import kernels
    g = torch.Generator(device=dev).manual_seed(N)
    data = torch.randint(-2, 3, (P, N, 128), generator=g, device=dev).to(dt)
    cent = torch.randint(-2, 3, (P, nc, 128), generator=g, device=dev).to(dt)
    cent[:, 4:nc:8] = cent[:, 0:nc - 4:8]
    cent[:, 33:nc:64] = cent[:, 1:nc - 32:64]
    cent[:, nc - 1] = cent[:, 2]
    cent[:, nc // 2 + 1] = float("nan")      # scores that are no number never win, and a token without others gets 0
    data[0, N // 2] = float("nan")
    assign = torch.full((P, N), -1, dtype=torch.int32, device=dev)
    kernels.kmeans_assign(data, cent, assign, P, N, nc, 1, N)
    ids = torch.arange(nc, device=dev)
    for p in range(P):
        s = (data[p].double() @ cent[p].double().T).nan_to_num(nan=-1e9)
        first = torch.where(s == s.max(dim=1, keepdim=True)[0], ids, nc).amin(dim=1)
        assert torch.equal(assign[p].long(), first)


# Loops over more than two thousand centroids, and launches a little past two and three rounds of workgroups.
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("P,N,nc", [(3, 66001, 2080), (8, 17001, 544), (8, 18001, 544), (24, 8001, 1056)])
def test_assign_long_loops_and_short_last_rounds(dev, P, N, nc, dt):
    test_assign_tilings(dev, P, N, nc, dt)
    test_assign_ties_go_to_the_lowest_id(dev, P, N, nc, dt)


# Which tiling serves a launch follows its 256-token pieces: both sides of every line.
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("pieces,nc", [(128, 96), (129, 96), (256, 96), (257, 96), (384, 96), (385, 96), (512, 96), (513, 96),
                                       (640, 96), (641, 96), (768, 96), (769, 96), (1024, 96), (1024, 288), (1152, 96),
                                       (1153, 96)])
def test_assign_at_the_lines_between_tilings(dev, pieces, nc, dt):
    test_assign_tilings(dev, 1, pieces * 256 - 3, nc, dt)
    test_assign_ties_go_to_the_lowest_id(dev, 1, pieces * 256 - 3, nc, dt)


# Launches with a piece for 129 to about 200 compute units, by pieces and centroids, and the lines of the longest ones.
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("pieces,nc", [(129, 224), (129, 256), (220, 256), (221, 256), (129, 288), (208, 1024), (209, 1024),
                                       (192, 2048), (193, 2048), (130, 6016), (130, 6048), (1280, 96), (1281, 96), (1280, 288),
                                       (1281, 288)])
def test_assign_with_work_for_half_the_units(dev, pieces, nc, dt):
    test_assign_tilings(dev, 1, pieces * 256 - 3, nc, dt)
    test_assign_ties_go_to_the_lowest_id(dev, 1, pieces * 256 - 3, nc, dt)
    if pieces < 256:
        test_assign_finds_every_row(dev, 2, (pieces + 1) // 2 * 256 - 255, nc, dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("P,N,nc", [(5, 1001, 32), (8, 8193, 544), (16, 8200, 544), (20, 9757, 608), (33, 8200, 512),
                                    (2, 32768, 2048)])
def test_assign_finds_every_row(dev, P, N, nc, dt):
    """Scores that are exact (tokens that pick out one dimension of the centroids), with the maximum in every row of a
    sub-tile, with ties, with centroids that are no numbers (never chosen) and infinities: the first of the largest."""
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(nc + N)
    cent = torch.randint(-9, 10, (P, nc, 128), generator=g).float()
    dim = torch.randint(0, 128, (P, N), generator=g)
    cent[:, :, 64:] = torch.randint(-2, 1, (P, nc, 64), generator=g).float()     # ties everywhere
    cent[:, torch.arange(64) % nc, torch.arange(64)] = 20.                       # row c is the best of dimension c
    cent[1, 7] = float("nan")
    cent[0, :, 100] = -float("inf")      # (0 * inf is no number either: every other token of the problem has none)
    keys = torch.zeros(P, N, 128).scatter_(2, dim[..., None], 1.0)
    got = torch.full((P, N), -1, dtype=torch.int32, device=dev)
    kernels.kmeans_assign(keys.to(dt).to(dev), cent.to(dt).to(dev), got, P, N, nc, 1, N)
    score = torch.gather(cent.transpose(1, 2), 1, dim[..., None].expand(P, N, nc))
    score[0] = -float("inf")
    score = torch.nan_to_num(score, nan=-float("inf"), neginf=-float("inf"))
    assert np.array_equal(got.cpu().numpy(), score.numpy().argmax(axis=2))


@pytest.mark.parametrize("P,N,nc,seed", [(3, 1000, 64, 10), (2, 8192, 512, 11), (1, 4100, 1024, 12), (4, 37, 32, 13)])
def test_assign_update_valuesum_float16(dev, P, N, nc, seed):
    """IEEE half keys, values and centroids (the reference's harnesses default to fp16, simple_test.py:29):
    the same fixed-order fp32 sums, rounded to fp16 on store."""
    test_assign_update_valuesum(dev, P, N, nc, seed, dt=torch.float16)


def test_big_and_empty_clusters(dev):
    """All tokens identical: one cluster takes everything (list longer than a wave and than
    the LDS sort), the others stay empty and keep their centroid."""
    from retrievalattention_amd import kernels
    P, N, nc = 1, 20000, 64
    g = torch.Generator().manual_seed(5)
    row = torch.randn(128, generator=g).to(torch.bfloat16)
    keys = row.expand(P, N, 128).contiguous()
    cent = torch.randn(P, nc, 128, generator=g).to(torch.bfloat16)
    kd, cd = keys.to(dev), cent.to(dev).clone()
    assign = torch.empty(P, N, dtype=torch.int32, device=dev)
    counts = torch.empty(P, nc, dtype=torch.int32, device=dev)
    offsets = torch.empty(P, nc + 1, dtype=torch.int32, device=dev)
    members = torch.empty(P, N, dtype=torch.int32, device=dev)
    kernels.kmeans_assign(kd, cd, assign, P, N, nc, 1, N)
    kernels.kmeans_build_lists(assign, counts, offsets, members, P, N, nc)
    kernels.kmeans_update(kd, counts, offsets, members, cd, P, N, nc, 1, N, True)
    torch.cuda.synchronize()
    a, _, _ = okm.assign(keys[0, :1], cent[0])
    assert int(counts.cpu()[0, a[0]]) == N and int(counts.cpu().sum()) == N
    assert torch.equal(members.cpu()[0], torch.arange(N, dtype=torch.int32))
    keep = torch.ones(nc, dtype=torch.bool); keep[a[0]] = False
    assert torch.equal(cd.cpu()[0, keep], cent[0, keep])
    s, cnt = okm.cluster_sums(keys[0], np.full(N, a[0]), nc)
    assert torch.equal(cd.cpu()[0], okm.update(cent[0], s, cnt, True))


def test_medium_clusters_sorted(dev):
    """Clusters of a few hundred to a few thousand tokens exercise the workgroup sort."""
    from retrievalattention_amd import kernels
    P, N, nc = 2, 30000, 32
    g = torch.Generator().manual_seed(6)
    assign = torch.randint(0, 8, (P, N), generator=g, dtype=torch.int32)
    assign[0, ::3] = 31
    ad = assign.to(dev)
    counts = torch.empty(P, nc, dtype=torch.int32, device=dev)
    offsets = torch.empty(P, nc + 1, dtype=torch.int32, device=dev)
    members = torch.empty(P, N, dtype=torch.int32, device=dev)
    kernels.kmeans_build_lists(ad, counts, offsets, members, P, N, nc)
    torch.cuda.synchronize()
    for p in range(P):
        order = np.argsort(assign[p].numpy(), kind="stable")
        assert np.array_equal(members[p].cpu().numpy(), order.astype(np.int32))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_long_lists_blocked_sums(dev, dt):
    """Lists of 1 to several thousand random rows: update and value sums equal the oracle's
    blocked fixed-order sums bit for bit (lists over 256 rows take the block-item path, several
    of them per problem, next to short lists and empty clusters)."""
    from retrievalattention_amd import kernels
    P, N, nc = 3, 20011, 96
    g = torch.Generator().manual_seed(16)
    keys = torch.randn(P, N, 128, generator=g).to(dt)
    vals = torch.randn(P, N, 128, generator=g).to(dt)
    assign = torch.randint(0, 5, (P, N), generator=g, dtype=torch.int32)       # five lists of ~4000
    small = torch.randint(8, 90, (P, N), generator=g, dtype=torch.int32)       # the rest: ~100 each, 90..95 empty
    pick = torch.rand(P, N, generator=g) < 0.4
    assign[pick] = small[pick]
    assign[1, :700] = 7                                                        # 700+: three blocks, last one ragged
    assign[2, 5] = 95                                                          # a single-row list
    cent = torch.randn(P, nc, 128, generator=g).to(dt)
    ad, kd, vd = assign.to(dev), keys.to(dev), vals.to(dev)
    counts = torch.empty(P, nc, dtype=torch.int32, device=dev)
    offsets = torch.empty(P, nc + 1, dtype=torch.int32, device=dev)
    members = torch.empty(P, N, dtype=torch.int32, device=dev)
    kernels.kmeans_build_lists(ad, counts, offsets, members, P, N, nc)
    for normalize in (True, False):
        cd = cent.to(dev).clone()
        kernels.kmeans_update(kd, counts, offsets, members, cd, P, N, nc, 1, N, normalize)
        vs = torch.full((P, nc, 128), 7.0, dtype=dt, device=dev)
        kernels.kmeans_value_sum(vd, counts, offsets, members, vs, P, N, nc)
        torch.cuda.synchronize()
        for p in range(P):
            a = assign[p].numpy().astype(np.int64)
            s, cnt = okm.cluster_sums(keys[p], a, nc)
            assert np.array_equal(counts[p].cpu().numpy(), cnt)
            assert torch.equal(cd[p].cpu(), okm.update(cent[p], s, cnt, normalize))
            assert torch.equal(vs[p].cpu(), okm.value_sum(vals[p], a, nc))


def test_long_lists_back_to_back(dev):
    """Long lists placed so that their blocks sit as close together as the layout allows (lengths
    just above one, two and three blocks, at offsets just below and at block boundaries, with empty
    and one-row clusters between and after them): every block is summed exactly once, in order."""
    from retrievalattention_amd import kernels
    sizes = [[255, 257, 0, 257, 1, 511, 0, 0, 512, 513, 255, 769, 3, 0, 300, 0],
             [0, 0, 1025, 1, 257, 257, 257, 0, 2, 256, 256, 258, 254, 768, 0, 0],
             [4000, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 257]]
    P, nc = len(sizes), 32
    N = max(sum(r) for r in sizes)
    g = torch.Generator().manual_seed(21)
    assign = torch.empty(P, N, dtype=torch.int32)
    for p, row in enumerate(sizes):
        row = row + [0] * (nc - len(row))
        row[nc - 2] += N - sum(row)                      # the remainder goes to one late cluster
        ids = torch.repeat_interleave(torch.arange(nc, dtype=torch.int32), torch.tensor(row))
        assign[p] = ids[torch.randperm(N, generator=g)]
    keys = torch.randn(P, N, 128, generator=g).to(torch.bfloat16)
    cent = torch.randn(P, nc, 128, generator=g).to(torch.bfloat16)
    ad, kd, cd = assign.to(dev), keys.to(dev), cent.to(dev).clone()
    counts = torch.empty(P, nc, dtype=torch.int32, device=dev)
    offsets = torch.empty(P, nc + 1, dtype=torch.int32, device=dev)
    members = torch.empty(P, N, dtype=torch.int32, device=dev)
    kernels.kmeans_build_lists(ad, counts, offsets, members, P, N, nc)
    kernels.kmeans_update(kd, counts, offsets, members, cd, P, N, nc, 1, N, True)
    vs = torch.full((P, nc, 128), 7.0, dtype=torch.bfloat16, device=dev)
    kernels.kmeans_value_sum(kd, counts, offsets, members, vs, P, N, nc)
    torch.cuda.synchronize()
    for p in range(P):
        a = assign[p].numpy().astype(np.int64)
        s, cnt = okm.cluster_sums(keys[p], a, nc)
        assert np.array_equal(counts[p].cpu().numpy(), cnt)
        assert torch.equal(cd[p].cpu(), okm.update(cent[p], s, cnt, True))
        assert torch.equal(vs[p].cpu(), okm.value_sum(keys[p], a, nc))


@pytest.mark.parametrize("P,N,nc,seed", [(3, 1000, 64, 0), (2, 16384, 512, 1), (2, 16385, 512, 2), (5, 37, 32, 3),
                                         (2, 8192, 512, 4), (1, 4100, 1024, 5), (2, 1023, 96, 6), (1, 1, 32, 7)])
def test_build_lists_is_a_stable_sort(dev, P, N, nc, seed):
    """Inverted lists over the sizes on either side of the single-workgroup path (problems of at most
    16384 tokens with at most 512 clusters) and of the one- and two-pass paths: members are the stable
    argsort of the assignment, offsets and counts its CSR bounds; some clusters are empty."""
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(seed)
    assign = torch.randint(0, max(nc - 3, 1), (P, N), generator=g, dtype=torch.int32)
    assign[0, N // 2:] = nc - 1                     # one long run, and the highest id in use
    ad = assign.to(dev)
    counts = torch.full((P, nc), -1, dtype=torch.int32, device=dev)
    offsets = torch.full((P, nc + 1), -1, dtype=torch.int32, device=dev)
    members = torch.full((P, N), -1, dtype=torch.int32, device=dev)
    kernels.kmeans_build_lists(ad, counts, offsets, members, P, N, nc)
    torch.cuda.synchronize()
    for p in range(P):
        a = assign[p].numpy()
        cnt = np.bincount(a, minlength=nc)
        assert np.array_equal(members[p].cpu().numpy(), np.argsort(a, kind="stable"))
        assert np.array_equal(counts[p].cpu().numpy(), cnt)
        assert np.array_equal(offsets[p].cpu().numpy(), np.concatenate([[0], np.cumsum(cnt)]))


@pytest.mark.parametrize("P,N,nc", [(3, 1000, 544), (2, 40001, 1056), (1, 300000, 8192), (2, 70000, 40000), (1, 3000, 262144)])
def test_build_lists_by_buckets(dev, P, N, nc):
    """Ids of two digits: the least and the most clusters, a scan of several rounds, buckets whose counters need several,
    one bucket with most of the tokens and buckets without any."""
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(N)
    assign = torch.randint(0, max(nc - 700, 1), (P, N), generator=g, dtype=torch.int32)
    assign[0, N // 3:] = nc - 1
    counts, offsets, members = (torch.full(s, -1, dtype=torch.int32, device=dev) for s in ((P, nc), (P, nc + 1), (P, N)))
    kernels.kmeans_build_lists(assign.to(dev), counts, offsets, members, P, N, nc)
    for p in range(P):
        cnt = torch.bincount(assign[p], minlength=nc)
        assert torch.equal(members[p].cpu().long(), torch.argsort(assign[p], stable=True))
        assert torch.equal(counts[p].cpu().long(), cnt)
        assert torch.equal(offsets[p].cpu().long(), torch.cat((torch.zeros(1, dtype=torch.int64), torch.cumsum(cnt, 0))))


@pytest.mark.parametrize("G,N,nc,S,seed", [(2, 4096, 256, 4, 0), (1, 8192, 512, 1, 1), (2, 3001, 192, 3, 2)])
def test_segment_k_means_teacher_forced(dev, G, N, nc, S, seed, dt=torch.bfloat16):
    """Whole driver against the oracle, iteration by iteration: every step is checked on the
    state the kernels actually produced (the trajectory itself is chaotic under near-ties)."""
    from retrievalattention_amd import kernels
    from retrievalattention_amd.cache_hub.kmeans import segment_k_means, segment_k_means_csr, csr_to_dense
    keys, vals = _mixture(G, N, nc, seed, dt=dt)
    kd, vd = keys.to(dev), vals.to(dev)
    cent, vsum, clusters, csize = segment_k_means(kd, vd, nc, 10, S)
    torch.cuda.synchronize()
    # replay with the kernels step by step, comparing each step with the oracle
    idx = okm.init_indices(N, nc)
    c_dev = kd[:, idx.to(dev)].contiguous()
    nseg, ncs, P = N // S, nc // S, G * S
    a = torch.empty(P, nseg, dtype=torch.int32, device=dev)
    cnt = torch.empty(P, ncs, dtype=torch.int32, device=dev)
    off = torch.empty(P, ncs + 1, dtype=torch.int32, device=dev)
    mem = torch.empty(P, nseg, dtype=torch.int32, device=dev)
    for it in range(9):
        before = c_dev.cpu().view(P, ncs, 128).clone()
        kernels.kmeans_assign(kd, c_dev, a, P, nseg, ncs, S, N)
        kernels.kmeans_build_lists(a, cnt, off, mem, P, nseg, ncs)
        kernels.kmeans_update(kd, cnt, off, mem, c_dev, P, nseg, ncs, S, N, True)
        torch.cuda.synchronize()
        A = a.cpu().numpy()
        after = c_dev.cpu().view(P, ncs, 128)
        for p in range(P):
            gi, si = p // S, p % S
            d = keys[gi, si * nseg:(si + 1) * nseg]
            _check_assign(d, before[p], A[p])
            s, c2 = okm.cluster_sums(d, A[p].astype(np.int64), ncs)
            assert torch.equal(after[p], okm.update(before[p], s, c2, True)), f"iteration {it} problem {p}"
    # final pass and outputs of the driver equal the replayed state
    r = segment_k_means_csr(kd, vd, nc, 10, S)
    torch.cuda.synchronize()
    assert torch.equal(r.centroids.cpu(), cent.cpu())
    before = c_dev.cpu()
    A = r.assign.cpu().numpy()
    for gi in range(G):
        _check_assign(keys[gi], before[gi], A[gi])
        s, c2 = okm.cluster_sums(keys[gi], A[gi].astype(np.int64), nc)
        assert torch.equal(cent.cpu()[gi], okm.update(before[gi], s, c2, False))
        assert torch.equal(vsum.cpu()[gi], okm.value_sum(vals[gi], A[gi].astype(np.int64), nc))
        lists, sz = okm.reverse_index(A[gi].astype(np.int64), nc)
        assert np.array_equal(csize.cpu().numpy()[gi], sz)
        assert np.array_equal(clusters.cpu().numpy()[gi][:, :lists.shape[1]], lists)
    # invariants: every token in exactly one list, sizes add up
    assert int(csize.sum()) == G * N


@pytest.mark.parametrize("G,N,nc,S,seed", [(2, 4096, 256, 4, 10), (2, 3001, 192, 3, 12)])
def test_segment_k_means_teacher_forced_float16(dev, G, N, nc, S, seed):
    test_segment_k_means_teacher_forced(dev, G, N, nc, S, seed, dt=torch.float16)


@pytest.mark.parametrize("P,N,nc,kind", [
    (3, 1, 32, "even"), (2, 63, 32, "even"), (4, 64, 64, "one"), (2, 513, 96, "even"), (1, 8192, 512, "skew"),
    (130, 700, 512, "even"), (2, 4100, 1024, "even"), (1, 16384, 512, "one"), (1, 16384, 1024, "skew"), (1, 16383, 32, "even"),
    (16, 8192, 512, "skew"), (64, 1000, 512, "skew"), (100, 2000, 512, "one"),
])
def test_update_direct_equals_lists_and_update(dev, P, N, nc, kind):
    """Lists and means in one launch against the separate launches, bit for bit: every number of clusters per workgroup,
    lists longer than a block, a single list, problems that do not fill a round of the waves."""
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(N + nc)
    a = torch.randint(0, nc, (P, N), generator=g, dtype=torch.int32)
    if kind == "one":
        a[:] = nc // 3
    elif kind == "skew":
        big = torch.rand(P, N, generator=g)
        a[big < 0.5] = 7
        a[big > 0.8] = nc - 1
    a = a.to(dev)
    for dt in (torch.bfloat16, torch.float16):
        rows = torch.randn(P, N, 128, generator=g).to(dt).to(dev)
        cent = torch.randn(P, nc, 128, generator=g).to(dt).to(dev)
        i32 = lambda *s: torch.full(s, -1, dtype=torch.int32, device=dev)
        lists, got = (i32(P, nc), i32(P, nc + 1), i32(P, N)), (i32(P, nc), i32(P, nc + 1), i32(P, N))
        kernels.kmeans_build_lists(a, *lists, P, N, nc)
        for normalize in (True, False):
            want, direct = cent.clone(), cent.clone()
            kernels.kmeans_update(rows, *lists, want, P, N, nc, 1, N, normalize)
            kernels.kmeans_update_direct(rows, a, direct, P, N, nc, 1, N, normalize, got if normalize else None)
            assert torch.equal(want.view(torch.int16), direct.view(torch.int16))
        for x, y in zip(lists, got):
            assert torch.equal(x, y)
    with pytest.raises(RuntimeError):
        kernels.kmeans_update_direct(rows, a, cent, P, kernels.KMEANS_DIRECT_MAX_TOKENS + 1, nc, 1, N, True)


# Ends of the runs that the eight waves read four tokens to a lane (256, 512 and 1024 at a time, run lengths in 256s), rows
# of assignments that begin on four bytes only, and the three widths of a workgroup (by the number of problems).
@pytest.mark.parametrize("P", [1, 20, 70])
@pytest.mark.parametrize("N", [3, 255, 257, 511, 1025, 2047, 2049, 4095, 4099, 6145, 8193])
def test_update_direct_at_the_ends_of_runs(dev, P, N):
    for kind in ("even", "skew"):
        test_update_direct_equals_lists_and_update(dev, P, N, 512, kind)


def _passes_one_by_one(keys, cent, seg, updates, last):
    """What ri_kmeans_iterate stands for: plain assignments and updates."""
    from retrievalattention_amd import kernels
    G, N, _ = keys.shape
    n, nc, P = N // seg, cent.shape[1] // seg, G * seg
    assign, members = (torch.empty(P, n, dtype=torch.int32, device=keys.device) for _ in range(2))
    counts = torch.empty(P, nc, dtype=torch.int32, device=keys.device)
    offsets = torch.empty(P, nc + 1, dtype=torch.int32, device=keys.device)
    for i in range(updates + last):
        kernels.kmeans_assign(keys, cent, assign, P, n, nc, seg, N)
        if i < updates:
            kernels.kmeans_build_lists(assign, counts, offsets, members, P, n, nc)
            kernels.kmeans_update(keys, counts, offsets, members, cent, P, n, nc, seg, N, True)
    return assign, cent


# The smallest problems whose passes know of each other, with remainders of tokens and of the list's last sub-tile; the most
# centroids, the most problems, segments with tokens left over; and shapes on the other side of the line.
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("kind", ["mixture", "normal", "ties", "odd"])
@pytest.mark.parametrize("G,N,nc,seg", [(6, 45001, 2080, 1), (2, 17001, 16384, 1), (64, 16385, 544, 1), (2, 70003, 8192, 2),
                                        (1, 20001, 64, 1), (2, 3001, 192, 3)])
def test_iterate_equals_its_passes(dev, G, N, nc, seg, kind, dt):
    """Bit for bit the centroids and the assignment of the passes run one by one."""
    from retrievalattention_amd import kernels
    g = torch.Generator(device=dev).manual_seed(N + nc)
    keys = torch.randn(G, N, 128, generator=g, device=dev)
    if kind == "mixture":      # clusters of keys with a few large dimensions: the largest keys take every token at first
        centres = torch.randn(G, max(N // 16, 1), 128, generator=g, device=dev)
        centres[:, :, :4] *= 8
        label = torch.randint(centres.shape[1], (G, N), generator=g, device=dev)
        keys = torch.gather(centres, 1, label[..., None].expand(G, N, 128)) + 0.3 * keys
    elif kind == "ties":       # small whole numbers in few dimensions: keys and scores come many times over
        keys = torch.randint(-2, 3, (G, N, 128), generator=g, device=dev).float()
        keys[:, :, 6:] = 0
    elif kind == "odd":        # keys without a norm of any size (their mean's is no number), infinities, and no numbers
        keys[:, ::3] *= 1e-30 if dt == torch.bfloat16 else 0
        keys[:, 5::4001] = float("inf")
        keys[:, 9::5003, 7] = float("nan")
    keys = keys.to(dt).contiguous()
    start = torch.empty(G, nc, 128, dtype=dt, device=dev)
    kernels.kmeans_init(keys, start, G, N, nc)
    for updates, last in ((9, True), (4, False), (0, True)):
        want, cent = _passes_one_by_one(keys, start.clone(), seg, updates, last)
        mine = start.clone()
        got = torch.full_like(want, -1)
        kernels.kmeans_iterate(keys, mine, got, G * seg, N // seg, nc // seg, seg, N, updates, last)
        assert torch.equal(got, want)
        assert torch.equal(mine.view(torch.int16), cent.view(torch.int16))


@pytest.mark.parametrize("G,N,nc,seg", [(3, 102400, 2048, 1), (3, 102401, 2048, 1)])
def test_iterate_on_both_sides_of_fifty_tokens_a_centroid(dev, G, N, nc, seg):
    test_iterate_equals_its_passes(dev, G, N, nc, seg, "mixture", torch.bfloat16)


def test_iterate_refuses(dev):
    from retrievalattention_amd import _lib
    lib = _lib.lib()
    keys = torch.zeros(1, 64, 128, dtype=torch.bfloat16, device=dev)
    cent = torch.zeros(1, 32, 128, dtype=torch.bfloat16, device=dev)
    assign = torch.empty(1, 64, dtype=torch.int32, device=dev)
    nbytes = lib.ri_kmeans_iterate_workspace_bytes(1, 64, 32)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    call = lambda nc=32, updates=1, room=nbytes, p=ws.data_ptr(): lib.ri_kmeans_iterate(
        keys.data_ptr(), cent.data_ptr(), assign.data_ptr(), 1, 64, nc, 1, 64, updates, 1, p, room, 0)
    assert call() == 0
    assert call(nc=33) != 0 and call(updates=-1) != 0 and call(room=nbytes - 1) != 0 and call(p=None) != 0


# The assignments that passes hand over in 16 bits, eight to a lane: problems of fewer than eight tokens, runs of a wave that
# end inside a lane's eight or that no token is left for, second rounds, odd starts of a problem's row, 8, 16 and 32 clusters to
# a workgroup, and the most centroids whose ids leave a word over.
@pytest.mark.parametrize("G,N,nc,seg", [(1, 7, 32, 1), (3, 8, 32, 1), (5, 9, 64, 1), (1, 255, 64, 1), (3, 1025, 96, 3),
                                        (2, 2049, 96, 1), (8, 8191, 512, 1), (3, 15 * 1001, 480, 15), (130, 4099, 256, 1),
                                        (2, 16384, 1024, 1), (1, 16383, 65504, 1), (1, 300, 65536, 1)])
@pytest.mark.parametrize("kind", ["mixture", "ties"])
def test_iterate_hands_assignments_over(dev, G, N, nc, seg, kind):
    test_iterate_equals_its_passes(dev, G, N, nc, seg, kind, torch.bfloat16)


# Tables of digit counts that the scatter adds up itself and the smallest that a launch scans: whole ids of 6, 7 and 9 bits and
# ids of two digits on both sides of 16384 counts, fewer than 64 digits, 512 buckets, last chunks of one token.
@pytest.mark.parametrize("P,N,nc", [(2, 262144, 64), (2, 262145, 64), (1, 131073, 100), (3, 32768, 512), (3, 32769, 512), (2, 131072, 8192),
                                    (2, 131073, 8192), (5, 16385, 33), (2, 20000, 32), (3, 17409, 544), (1, 33793, 16384), (2, 32768, 16384)])
def test_build_lists_on_both_sides_of_the_table(dev, P, N, nc):
    test_build_lists_is_a_stable_sort(dev, P, N, nc, N % 97)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("wide", [False, True])
def test_sums_of_lists_of_every_length(dev, dt, wide):
    """Lists whose lengths lie around the eights, the rounds of 64 rows and the blocks of 256 of a wave's sum, in rows that are
    next to each other and in rows too far apart for offsets of 31 bits: the sums that the oracle defines."""
    from retrievalattention_amd import kernels
    lengths = [0, 1, 2, 7, 8, 9, 15, 31, 56, 57, 63, 64, 65, 71, 72, 127, 128, 129, 136, 191, 192, 193, 200, 255, 256, 257, 264, 319,
               320, 321, 511, 512, 513, 576, 777, 1024, 1100, 3000, 5000, 6, 64, 16]
    nc = len(lengths) + (-len(lengths)) % 32
    g = torch.Generator().manual_seed(7)
    a = torch.cat([torch.full((n,), c) for c, n in enumerate(lengths)])[torch.randperm(sum(lengths), generator=g)].int()
    N = a.numel()
    rows = torch.randn(N, 128, generator=g).to(dt)
    counts, offsets, members = (torch.empty(1, n, dtype=torch.int32, device=dev) for n in (nc, nc + 1, N))
    kernels.kmeans_build_lists(a[None].to(dev), counts, offsets, members, 1, N, nc)
    assert counts[0, :len(lengths)].tolist() == lengths
    if wide:
        pitch = (1 << 30) // N // 8 * 8 + 128   # elements: N rows of it are past 2 GiB
        values = torch.zeros(N * pitch, dtype=dt, device=dev).view(N, pitch)[:, :128]
        values.copy_(rows)
    else:
        values = rows.to(dev)
    sums = torch.empty(1, nc, 128, dtype=dt, device=dev)
    kernels.kmeans_value_sum(values[None], counts, offsets, members, sums, 1, N, nc)
    s, _ = okm.cluster_sums(rows, a.numpy().astype(np.int64), nc)
    assert torch.equal(sums[0].cpu(), torch.from_numpy(s).to(dt))


@pytest.mark.parametrize("G,N,nc,seg", [(3, 40001, 96, 1), (1, 65600, 640, 1), (5, 17001, 32, 1), (2, 50003, 1024, 3), (1, 16640, 32, 1)])
@pytest.mark.parametrize("kind", ["mixture", "ties", "odd"])
def test_iterate_folds_long_lists_where_they_are_summed(dev, G, N, nc, seg, kind):
    """Longer problems whose passes know nothing of each other: lists of two blocks, of hundreds, and one of all tokens."""
    nc = nc if seg == 1 else nc // 32 // seg * 32 * seg
    test_iterate_equals_its_passes(dev, G, N, nc, seg, kind, torch.bfloat16)

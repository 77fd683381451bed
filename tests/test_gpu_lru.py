"""Device-side block cache manager against its Python restatement (oracle.wavebuf.DeviceLruModel), and
against the restatement of the reference's manager (oracle.wavebuf.LruModel) where the two policies coincide."""
import random

import pytest
import torch

from oracle.wavebuf import DeviceLruModel, LruModel
from tests.parity import BlockIdMap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncl,nprobe,capacity,buffer_size,steps,seed", [
    (200, 12, 60, 48, 40, 0),        # constant eviction pressure
    (3840, 69, 600, 552, 25, 1),     # config-4 sizes: 5 % cache
    (300, 20, 40, 30, 30, 2),        # buffer cut-off and admissions cut short
    (2500, 40, 4000, 400, 12, 3),    # cache larger than everything requested: no eviction
    (300, 20, 0, 160, 6, 4),         # a cache without blocks (throughput_eval/test.py:77): all misses, none admitted
    (20000, 1500, 9000, 12000, 6, 5),   # probe lists past 1023 ranks (four ranks per thread)
    (40000, 3000, 2000, 20000, 5, 6),   #   with the buffer cut-off and admissions cut short
])
def test_lists_match_the_model_step_by_step(dev, ncl, nprobe, capacity, buffer_size, steps, seed):
    from retrievalattention_amd import kernels
    BG, block = 3, 8
    rnd = random.Random(seed)
    sizes = [[rnd.choice([0, 1, 7, 8, 9, 16, 23, 40]) if rnd.random() < 0.3 else rnd.randint(1, 30) for _ in range(ncl)]
             for _ in range(BG)]
    models = [DeviceLruModel(s, block, capacity, buffer_size) for s in sizes]
    sz = torch.tensor(sizes, dtype=torch.int32, device=dev)
    st = (torch.cumsum(sz.long(), 1) - sz.long()).to(torch.int32)
    lru = kernels.DeviceLru(BG, ncl + 7, int(((sz + block - 1) // block).sum(1).max()) + 5, capacity, buffer_size, block,
                            dev)
    lru.set_sizes(sz)
    lists = [torch.full((BG, buffer_size), -7, dtype=torch.int32, device=dev) if i % 4 != 3
             else torch.zeros(BG, dtype=torch.int32, device=dev) for i in range(12)]
    hot = [rnd.sample(range(ncl), min(ncl, 3 * nprobe)) for _ in range(BG)]
    for step in range(steps):
        ids = []
        for g in range(BG):   # mostly a hot set (hits), some fresh ids (misses), now and then an invalid id
            pool = hot[g] if rnd.random() < 0.8 else list(range(ncl))
            row = rnd.sample(pool, nprobe)
            if rnd.random() < 0.2:
                row[rnd.randrange(nprobe)] = ncl + 3
            ids.append(row)
        t = torch.tensor(ids, dtype=torch.int32, device=dev)
        lru.access_update(t, sz, st, lists)
        torch.cuda.synchronize()
        host = [x.cpu() for x in lists]
        for g in range(BG):
            hit, miss, upd = models[g].step(ids[g])
            for k, ref in enumerate((hit, miss, upd)):
                a, b, c, n = host[4 * k:4 * k + 4]
                assert int(n[g]) == len(ref), (step, g, k)
                got = list(zip(a[g, :len(ref)].tolist(), b[g, :len(ref)].tolist(), c[g, :len(ref)].tolist()))
                if k == 2:   # update lists are (buffer offset, size, cache block id); the model gives (id, size, offset)
                    got = [(z, y, x) for x, y, z in got]
                assert got == ref, (step, g, k)
            assert int(lru.free_count[g]) == len(models[g].free)
            assert lru.free_list[g, :len(models[g].free)].tolist() == models[g].free
            stamp = lru.stamp[g, :ncl].cpu()
            assert [int(x) for x in stamp] == models[g].stamp
            order = lru.order[g, :ncl].cpu()
            assert all(int(order[c]) == models[g].sub[c] for c in models[g].blocks)
    assert capacity == 0 or any(len(m.blocks) > 0 for m in models)


@pytest.mark.parametrize("ncl,nprobe,capacity,steps,seed", [(40, 1, 24, 250, 0), (300, 1, 64, 250, 1), (200, 12, 60, 80, 2),
                                                           (60, 8, 10, 120, 3), (3000, 150, 900, 40, 4)])
def test_lists_equal_the_reference_policy(dev, ncl, nprobe, capacity, steps, seed):
    """The kernel's hit / miss / admission lists and its evictions equal those of the reference's manager
    (LruModel, itself checked against the reference's own BufferManager build) over random probe traces: one
    probe per step, several probes with eviction pressure, a cache smaller than one step's hits (hits of the
    current step are evicted), a config-4-like size.  Block id values aside: an id map is kept and must stay
    a bijection."""
    from retrievalattention_amd import kernels
    BG, block, buffer_size = 2, 8, max(16, 4 * nprobe)
    rnd = random.Random(seed)
    sizes = [[rnd.randint(0, 30) for _ in range(ncl)] for _ in range(BG)]
    refs = [LruModel(s, block, capacity, buffer_size) for s in sizes]
    maps = [BlockIdMap() for _ in range(BG)]
    sz = torch.tensor(sizes, dtype=torch.int32, device=dev)
    st = (torch.cumsum(sz.long(), 1) - sz.long()).to(torch.int32)
    lru = kernels.DeviceLru(BG, ncl, int(((sz + block - 1) // block).sum(1).max()) + 1, capacity, buffer_size, block, dev)
    lru.set_sizes(sz)
    lists = [torch.full((BG, buffer_size), -7, dtype=torch.int32, device=dev) if i % 4 != 3
             else torch.zeros(BG, dtype=torch.int32, device=dev) for i in range(12)]
    hot = [rnd.sample(range(ncl), max(2, min(ncl, 3 * nprobe), ncl // 3 if nprobe == 1 else 0)) for _ in range(BG)]
    evictions = 0
    for step in range(steps):
        ids = [rnd.sample(hot[g] if rnd.random() < 0.6 else range(ncl), nprobe) for g in range(BG)]
        lru.access_update(torch.tensor(ids, dtype=torch.int32, device=dev), sz, st, lists)
        torch.cuda.synchronize()
        host = [x.cpu() for x in lists]
        for g in range(BG):
            before = set(refs[g].resident)
            hit, miss = refs[g].access(ids[g])
            upd = refs[g].update()
            evictions += len(before - set(refs[g].resident))
            lists_g = []
            for k, ref in enumerate((hit, miss, upd)):
                a, b, c, n = host[4 * k:4 * k + 4]
                assert int(n[g]) == len(ref), (step, g, k)
                got = list(zip(a[g, :len(ref)].tolist(), b[g, :len(ref)].tolist(), c[g, :len(ref)].tolist()))
                lists_g.append([(z, y, x) for x, y, z in got] if k == 2 else got)
            # hits: block ids through the map (a hit of this step may be evicted by the same step's admission)
            assert [(maps[g].to_ref(x), y, z) for x, y, z in lists_g[0]] == hit, (step, g, 0)
            assert lists_g[1] == miss, (step, g, 1)      # misses: host rows, no block ids involved
            # blocks of clusters evicted in this step go back to the free list and may be handed out again at once
            maps[g].retain({b for ids_c in refs[g].resident.values() for b in ids_c} - {b for b, _, _ in upd})
            for (bg, _, _), (br, _, _) in zip(lists_g[2], upd):     # admission hands out ids: the map learns them
                maps[g].bind(bg, br)
            assert [(maps[g].to_ref(x), y, z) for x, y, z in lists_g[2]] == upd, (step, g, 2)
            # the same clusters are resident: evictions happened in the same order
            resident = set(torch.nonzero(lru.stamp[g, :ncl]).flatten().tolist())
            assert resident == set(refs[g].resident), (step, g)
    assert evictions > 0


def test_row_table_for_attention_in_place(dev):
    """With a row table the manager lists no hits for copying and writes, for every retrieved token in
    rank order, its row in a tensor that holds the cache blocks followed by the staged misses."""
    from retrievalattention_amd import kernels
    BG, block, ncl, nprobe, capacity, buffer_size = 2, 8, 500, 30, 150, 120
    rnd = random.Random(9)
    sizes = [[rnd.randint(0, 45) for _ in range(ncl)] for _ in range(BG)]
    stage0 = capacity * block
    models = [DeviceLruModel(s, block, capacity, buffer_size, stage_row0=stage0) for s in sizes]
    sz = torch.tensor(sizes, dtype=torch.int32, device=dev)
    st = (torch.cumsum(sz.long(), 1) - sz.long()).to(torch.int32)
    lru = kernels.DeviceLru(BG, ncl, int(((sz + block - 1) // block).sum(1).max()), capacity, buffer_size, block, dev)
    lru.set_sizes(sz)
    lists = [torch.zeros((BG, buffer_size), dtype=torch.int32, device=dev) if i % 4 != 3
             else torch.zeros(BG, dtype=torch.int32, device=dev) for i in range(12)]
    row_src = torch.full((BG, buffer_size * block), -1, dtype=torch.int32, device=dev)
    meta = torch.zeros(BG, 4, dtype=torch.int32, device=dev)
    hot = [rnd.sample(range(ncl), 60) for _ in range(BG)]
    for step in range(25):
        ids = [rnd.sample(hot[g] if rnd.random() < 0.7 else range(ncl), nprobe) for g in range(BG)]
        lru.access_update(torch.tensor(ids, dtype=torch.int32, device=dev), sz, st, lists, row_src=row_src,
                          stage_row0=stage0, meta=meta)
        torch.cuda.synchronize()
        for g in range(BG):
            hit, miss, upd = models[g].step(ids[g])
            rows = models[g].rows
            assert int(meta[g, 1]) == len(rows) and int(meta[g, 2]) == len(hit) + len(miss)
            assert row_src[g, :len(rows)].tolist() == rows
            assert int(lists[3][g]) == 0 and int(lists[7][g]) == len(miss) and int(lists[11][g]) == len(upd)
            assert lru.free_list[g, :len(models[g].free)].tolist() == models[g].free
    assert any(any(r < stage0 for r in m.rows) for m in models) and any(any(r >= stage0 for r in m.rows) for m in models)


def test_bad_arguments(dev):
    from retrievalattention_amd import _lib
    l = _lib.lib()
    z = torch.zeros(64, dtype=torch.int32, device=dev)
    p = z.data_ptr()
    ptrs = [p] * 12
    assert l.ri_lru_access_update(p, p, p, 8, p, 9, p, p, 8, p, 8, p, p, p, *ptrs, None, 0, 0, None, 1, 4097, 8, 4, 4, 8, None) == -1   # np too large
    assert l.ri_lru_access_update(p, p, p, 4, p, 9, p, p, 8, p, 8, p, p, p, *ptrs, None, 0, 0, None, 1, 2, 8, 4, 4, 8, None) == -1      # stride < ncl
    assert l.ri_lru_access_update(None, p, p, 8, p, 9, p, p, 8, p, 8, p, p, p, *ptrs, None, 0, 0, None, 1, 2, 8, 4, 4, 8, None) == -1


@pytest.mark.parametrize("ncl,nprobe,capacity,buffer_size", [(300, 20, 60, 48), (4097, 60, 500, 400), (9000, 1100, 3000, 5000),
                                                             (200, 10, 0, 64)])
def test_access_and_stage_update_equal_the_one_launch(dev, ncl, nprobe, capacity, buffer_size):
    """Access and update apart: same lists, row table and books as in one launch, with ages of one to three bytes, and the
    missed rows in the staging rows."""
    import ctypes
    from retrievalattention_amd import kernels
    from retrievalattention_amd._lib import lib
    BG, block = 2, 8
    g = torch.Generator().manual_seed(ncl)
    sz = torch.randint(0, 30, (BG, ncl), generator=g, dtype=torch.int32).to(dev)
    st = (torch.cumsum(sz.long(), 1) - sz.long()).to(torch.int32)
    n = int(sz.sum(1).max())
    max_blocks = int(((sz + block - 1) // block).sum(1).max()) + 1
    host = [torch.randn(BG, n, 128, generator=g).to(torch.bfloat16).pin_memory() for _ in range(2)]
    stage0 = capacity * block
    cache = [torch.zeros(BG, stage0 + buffer_size * block, 128, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    sides = []
    for _ in range(2):
        lru = kernels.DeviceLru(BG, ncl, max_blocks, capacity, buffer_size, block, dev)
        lru.set_sizes(sz)
        lists = [torch.zeros((BG,) if i % 4 == 3 else (BG, buffer_size), dtype=torch.int32, device=dev) for i in range(12)]
        row_src = torch.zeros(BG, buffer_size * block, dtype=torch.int32, device=dev)
        sides.append((lru, lists, row_src, torch.zeros(BG, 4, dtype=torch.int32, device=dev)))
    hot = torch.randperm(ncl, generator=g)[:4 * nprobe]
    ids = torch.zeros(BG, nprobe, dtype=torch.int32, device=dev)
    lru, lists, row_src, meta = sides[1]
    s = lru.prepared(ids, sz, st, lists, row_src, stage0, meta, *host, *cache)
    for step in range(12):
        for b in range(BG):
            ids[b] = hot[torch.randperm(hot.numel(), generator=g)[:nprobe]]
        if step in (4, 8):
            for side in sides:
                side[0].epoch += 300 if step == 4 else 70000
        sides[0][0].access_update(ids, sz, st, sides[0][1], row_src=sides[0][2], stage_row0=stage0, meta=sides[0][3])
        for fn in (lib().ri_lru_access, lib().ri_lru_stage_update):
            assert fn(ctypes.addressof(s), kernels._stream()) == 0
        for x, y in zip(sides[0][1] + list(sides[0][2:]), lists + [row_src, meta]):
            assert torch.equal(x, y), step
        for name in ("stamp", "blk_ids", "free_list", "free_count", "epoch"):
            assert torch.equal(getattr(sides[0][0], name), getattr(lru, name)), (step, name)
        resident = lru.stamp > 0
        assert torch.equal(sides[0][0].order[resident], lru.order[resident])
        for b in range(BG):
            for j in range(int(lists[7][b])):
                row, k, at = (int(lists[4 + x][b, j]) for x in range(3))
                for h, c in zip(host, cache):
                    assert torch.equal(c[b, stage0 + at:stage0 + at + k].cpu(), h[b, row:row + k])


@pytest.mark.parametrize("BG,block", [(1, 8), (3, 1), (63, 3), (65, 8), (130, 16)])
def test_missed_rows_are_staged_in_rank_order(dev, BG, block, most=39):
    """Items numbered through all groups, sixty-four groups at a time: groups without misses, partial blocks, blocks shorter and
    longer than the eight rows a wave copies at a time; nothing is written behind the rows."""
    import ctypes
    from retrievalattention_amd import kernels
    from retrievalattention_amd._lib import lib
    g = torch.Generator().manual_seed(BG)
    ncl, nprobe = 24, 7
    sz = torch.randint(0, most + 1, (BG, ncl), generator=g, dtype=torch.int32)
    sz[1::5] = 0
    st = (torch.cumsum(sz.long(), 1) - sz.long()).to(torch.int32)
    n = max(1, int(sz.sum(1).max()))
    buffer_size = nprobe * ((most + block - 1) // block)
    host = [torch.randn(BG, n, 128, generator=g).to(torch.bfloat16).pin_memory() for _ in range(2)]
    cache = [torch.zeros(BG, buffer_size * block + 1, 128, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    lru = kernels.DeviceLru(BG, ncl, int(((sz + block - 1) // block).sum(1).max()) + 1, 0, buffer_size, block, dev)
    lru.set_sizes(sz.to(dev))
    lists = [torch.zeros((BG,) if i % 4 == 3 else (BG, buffer_size), dtype=torch.int32, device=dev) for i in range(12)]
    row_src = torch.zeros(BG, buffer_size * block, dtype=torch.int32, device=dev)
    ids = torch.stack([torch.randperm(ncl, generator=g)[:nprobe] for _ in range(BG)]).to(torch.int32)
    s = lru.prepared(ids.to(dev), sz.to(dev), st.to(dev), lists, row_src, 0, torch.zeros(BG, 4, dtype=torch.int32, device=dev),
                     *host, *cache)
    for fn in (lib().ri_lru_access, lib().ri_lru_stage_update):
        assert fn(ctypes.addressof(s), kernels._stream()) == 0
    for h, c in zip(host, cache):
        want = torch.zeros(c.shape, dtype=c.dtype)
        for b in range(BG):
            rows = torch.cat([torch.arange(st[b, i], st[b, i] + sz[b, i]) for i in ids[b].tolist()])
            want[b, :len(rows)] = h[b, rows]
        assert torch.equal(c.cpu(), want)


@pytest.mark.parametrize("BG,block,most", [(1, 8, 1), (40, 8, 1), (40, 8, 2), (64, 8, 3), (70, 8, 5), (40, 2, 7), (200, 8, 1),
                                           (33, 8, 8)])
def test_short_blocks_are_staged_in_rank_order(dev, BG, block, most):
    """Blocks of few rows, which more waves than one of a workgroup copy: from eight down to two of them."""
    test_missed_rows_are_staged_in_rank_order(dev, BG, block, most)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("BG,gs,nc,nprobe,es,buffer_blocks", [
    # selection and look-up in one launch: every number of threads and of clusters to a thread, heads padded and not, no
    # estimation zone, a probe list as long as the threads take, a buffer that cuts the list
    (1, 1, 8, 3, 2, 100), (3, 8, 256, 255, 0, 2000), (2, 12, 256, 9, 100, 12), (2, 4, 264, 20, 60, 200), (5, 7, 512, 511, 1, 4000),
    (2, 3, 520, 511, 9, 4000), (3, 16, 1024, 18, 237, 100), (2, 8, 1032, 30, 300, 40), (1, 9, 2048, 40, 500, 300),
    (1, 4, 2048, 1023, 500, 8000), (2, 7, 2056, 600, 300, 5000), (2, 8, 4096, 74, 950, 400), (70, 4, 64, 5, 10, 30),
    # past it
    (2, 8, 256, 256, 0, 2000), (1, 4, 512, 512, 0, 4000), (2, 9, 2056, 40, 300, 300), (1, 4, 4104, 74, 950, 400),
    (1, 2, 2048, 1024, 300, 8000), (1, 8, 8200, 20, 300, 200)])
def test_host_step_equals_the_operators(dev, dtype, BG, gs, nc, nprobe, es, buffer_blocks):
    """The prepared step against selection and look-up called by themselves: the same ids, lists, row table and books, and the
    output of an attention over the step's own row table."""
    from retrievalattention_amd import kernels
    block, steps = 8, 4
    g = torch.Generator().manual_seed(BG * nc + nprobe)
    rn = lambda *s: torch.randn(*s, generator=g).to(dtype)
    sz = torch.randint(0, 21, (BG, nc), generator=g, dtype=torch.int32)
    st = (torch.cumsum(sz.long(), 1) - sz.long()).to(torch.int32)
    n, max_blocks = int(sz.sum(1).max()) + 1, int(((sz + 7) // 8).sum(1).max()) + 1
    mask, size16 = (sz == 0).to(dev), sz.to(dtype).to(dev)
    sz, st = sz.to(dev), st.to(dev)
    capacity, stage0 = max_blocks, max_blocks * block
    cent, vs, sk, sv = rn(BG, nc, 128).to(dev), rn(BG, nc, 128).to(dev), rn(BG, 70, 128).to(dev), rn(BG, 70, 128).to(dev)
    host = [rn(BG, n, 128).pin_memory() for _ in range(2)]
    scale = 128 ** -0.5
    i32 = lambda *s: torch.full(s, -5, dtype=torch.int32, device=dev)
    sides = []
    for _ in range(2):
        lru = kernels.DeviceLru(BG, nc, max_blocks, capacity, buffer_blocks, block, dev)
        lru.set_sizes(sz)
        lists = [torch.zeros((BG,) if i % 4 == 3 else (BG, buffer_blocks), dtype=torch.int32, device=dev) for i in range(12)]
        sides.append(dict(lru=lru, lists=lists, row_src=i32(BG, buffer_blocks * block), meta=i32(BG, 4), ret=i32(BG, nprobe),
                          est=i32(BG, max(es, 1)), logits=torch.zeros(BG, gs, nc, device=dev), valid=i32(BG)))
    a, b = sides
    cache = [torch.zeros(BG, stage0 + buffer_blocks * block, 128, dtype=dtype, device=dev) for _ in range(2)]
    est = lambda d: d["est"] if es else None
    plan = kernels.HostStepPlan(None, dtype, dict(
        centroids=cent, mask=mask, logits=b["logits"], ret_ids=b["ret"], est_ids=est(b), meta=b["meta"], steady_k=sk, steady_v=sv,
        store_k=cache[0], store_v=cache[1], value_sum=vs, cluster_size=size16, valid_lengths=b["valid"]), nprobe, es, 8,
        buffer_blocks, scale, b["lru"], sz, st, b["lists"], b["row_src"], *host, stage0)
    q0 = rn(BG, gs, 128).to(dev)
    for step in range(steps):
        q = q0 + 0.3 * step * rn(BG, gs, 128).to(dev)
        kernels.score_select(q, cent, mask, None, None, a["logits"], None, None, a["ret"], est(a), None, None, None, nprobe, es, 8,
                             buffer_blocks, scale)
        a["lru"].access_update(a["ret"], sz, st, a["lists"], row_src=a["row_src"], stage_row0=stage0, meta=a["meta"])
        got, want = (torch.empty(BG, gs, 128, dtype=dtype, device=dev) for _ in range(2))
        plan.run(q, 70, got)
        for name in ("ret", "est", "logits", "row_src", "meta"):
            if es or name != "est":
                assert torch.equal(a[name], b[name]), (step, name)
        for x, y in zip(a["lists"], b["lists"]):
            assert torch.equal(x, y), step
        for name in ("stamp", "blk_ids", "free_list", "free_count", "epoch"):
            assert torch.equal(getattr(a["lru"], name), getattr(b["lru"], name)), (step, name)
        kernels.wave_attention(q, sk, sv, 70, *cache, b["row_src"], b["meta"], est(b), b["logits"] if es else None, vs, size16, want,
                               b["valid"], es, scale)
        assert torch.equal(got, want), step

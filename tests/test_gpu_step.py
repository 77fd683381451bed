"""ri_append_kv: the token's rows land at their position and nowhere else."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BG,stride,pos,on_device", [(1, 1, 0, False), (3, 70, 69, False), (16, 69, 0, True),
                                                     (37, 324, 100, True), (37, 324, 324, True), (5, 8, -1, True)])
def test_append_kv(dev, BG, stride, pos, on_device):
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(BG)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(dev)
    k, v, zk, zv = bf(BG, 128), bf(BG, 128), bf(BG, stride, 128), bf(BG, stride, 128)
    want = [zk.clone(), zv.clone()]
    if 0 <= pos < stride:
        want[0][:, pos], want[1][:, pos] = k, v
    at = torch.tensor([pos], dtype=torch.int64, device=dev) if on_device else None
    kernels.append_kv(k, v, zk, zv, 0 if on_device else pos, at)
    assert torch.equal(zk, want[0]) and torch.equal(zv, want[1])
    if not on_device:
        with pytest.raises(RuntimeError):
            kernels.append_kv(k, v, zk, zv, stride)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("BG,gs,nc,np_,es,static,pages,on_device", [
    (1, 1, 8, 1, 0, 0, 100, False), (2, 4, 8, 3, 5, 1, 100, True), (3, 5, 40, 7, 33, 17, 100, False),
    (5, 8, 256, 4, 60, 70, 2, True), (4, 3, 264, 10, 100, 69, 100, False), (8, 4, 512, 9, 118, 98, 100, False),
    (2, 7, 504, 12, 150, 100, 3, True), (256, 2, 16, 2, 3, 5, 100, False), (257, 2, 16, 2, 3, 5, 100, False),
    (2, 4, 512, 13, 118, 98, 100, False), (2, 4, 512, 13, 118, 98, 40, False), (3, 8, 512, 9, 118, 98, 72, False),
    (3, 8, 512, 9, 118, 98, 76, True),
    # one workgroup per group, past 128 groups: heads padded and not, every number of waves that score, no estimation zone, cut
    # pages, the zone's length from the device, and both sides of 448 rows
    (129, 1, 8, 1, 0, 0, 100, False), (129, 5, 40, 7, 33, 17, 100, False), (256, 7, 64, 2, 20, 69, 1, True),
    (200, 8, 256, 4, 0, 70, 100, False), (256, 3, 128, 2, 30, 300, 100, True), (130, 8, 512, 9, 118, 98, 100, True),
    (129, 8, 264, 13, 118, 122, 100, False), (129, 8, 264, 13, 118, 123, 100, False), (160, 4, 104, 18, 0, 160, 3, True),
    (160, 4, 104, 18, 0, 161, 3, True)])
def test_short_step_equals_the_operators(dev, dtype, BG, gs, nc, np_, es, static, pages, on_device):
    """The step in one launch, of several workgroups per group up to 128 groups and of one past them (and, past its limits, the
    launches one by one), against scoring + selection and attention called by themselves: the same lists; outputs differ
    only where the rows of a group are split in another way, by roundings of the 16-bit probabilities and of the output, each at most 2^-8 of a value (2^-11 in half), of which a
    norm over the output sees a fraction."""
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(BG * nc + gs)
    rn = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)
    size = torch.randint(0, 30, (BG, nc), generator=g, dtype=torch.int32)
    size[:, 0] = 0
    start = (size.cumsum(1) - size).int().to(dev)
    rows = int(size.sum(1).max()) + 1
    mask = (size == 0).to(dev)
    size16, size = size.to(dtype).to(dev), size.to(dev)
    q, cent, vs = rn(BG, gs, 128), rn(BG, nc, 128), rn(BG, nc, 128)
    zone = static + 3
    sk, sv, store_k, store_v = rn(BG, zone, 128), rn(BG, zone, 128), rn(BG, rows, 128), rn(BG, rows, 128)
    length = torch.tensor([static], dtype=torch.int32, device=dev) if on_device else None

    def fresh():
        i32 = lambda *s: torch.full(s, -5, dtype=torch.int32, device=dev)
        return dict(logits=torch.zeros(BG, gs, nc, device=dev), ret_ids=i32(BG, np_), est_ids=i32(BG, max(es, 1)),
                    ret_tok_off=i32(BG, np_ + 1), ret_start=i32(BG, np_), meta=i32(BG, 4), valid_lengths=i32(BG))
    a, b = fresh(), fresh()
    scale = 128 ** -0.5
    est = lambda d: d["est_ids"] if es else None
    kernels.score_select(q, cent, mask, size, start, a["logits"], None, None, a["ret_ids"], est(a), a["ret_tok_off"], None,
                         a["meta"], np_, es, 8, pages, scale, ret_start=a["ret_start"])
    want, got = torch.empty(BG, gs, 128, dtype=dtype, device=dev), torch.empty(BG, gs, 128, dtype=dtype, device=dev)
    kernels.wave_attention(q, sk, sv, static, store_k, store_v, None, a["meta"], est(a), a["logits"] if es else None, vs,
                           size16, want, a["valid_lengths"], es, scale, ret_tok_off=a["ret_tok_off"],
                           ret_start=a["ret_start"], static_len_dev=length)
    plan = kernels.DecodeStepPlan(None, dtype, dict(
        b, est_ids=est(b), centroids=cent, mask=mask, cluster_size_i32=size, cluster_start=start, steady_k=sk, steady_v=sv,
        static_len_dev=length, store_k=store_k, store_v=store_v, value_sum=vs, cluster_size=size16), np_, es, 8, pages, scale)
    for _ in range(2):
        plan.run(q, static, got)
    for name in a:
        if es or name != "est_ids":
            assert torch.equal(a[name], b[name]), name
    wf, gf = want.float(), got.float()
    assert (wf - gf).norm() <= (4e-3 if dtype == torch.bfloat16 else 5e-4) * wf.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("BG,gs,nc,np_,es,static,pages,on_device", [
    # several workgroups per group that score for themselves: many rows, few clusters, no estimation zone, cut pages
    (3, 8, 512, 51, 119, 98, 1000, False), (2, 4, 504, 512 - 8, 0, 700, 2000, True), (1, 1, 8, 1, 7, 900, 100, False),
    (5, 7, 384, 38, 100, 300, 20, False), (128, 3, 64, 12, 30, 700, 100, True), (256, 8, 32, 4, 20, 400, 100, False),
    # of which one has all rows where they are few after all: on both sides of the line, and of the one for many groups
    (3, 8, 512, 51, 119, 98, 4, True), (2, 4, 512, 20, 200, 128, 1, False), (2, 4, 512, 20, 200, 137, 1, False),
    (5, 1, 384, 38, 0, 69, 10, True), (80, 4, 256, 40, 60, 69, 10, False), (80, 4, 256, 40, 60, 572, 1, True),
    (80, 4, 256, 40, 60, 581, 1, True),
    # scored before: every number of clusters a thread takes, with remainders; who sums the scores; heads padded and not
    (2, 4, 520, 9, 100, 69, 100, False), (3, 8, 1024, 18, 237, 70, 200, True), (2, 16, 1032, 40, 300, 69, 300, False),
    (1, 12, 2048, 36, 475, 500, 200, False), (2, 9, 2056, 512, 300, 69, 2000, False), (1, 3, 4096, 73, 950, 0, 300, True),
    (2, 7, 4096, 20, 0, 69, 9, False), (1, 8, 3584, 70, 800, 69, 300, False), (1, 4, 4104, 73, 950, 69, 300, False),
    (1, 1, 8192, 147, 1900, 69, 700, True), (2, 5, 8200, 512, 1900, 69, 2000, False), (1, 16, 16384, 300, 7000, 69, 2000, False),
    (1, 8, 16384, 512, 15872, 69, 3000, False), (300, 2, 520, 5, 50, 20, 100, False),
    # 1024 threads that select
    (1, 2, 1024, 513, 300, 69, 3000, False), (2, 8, 4096, 1024, 3000, 69, 5000, True), (1, 4, 4104, 700, 0, 69, 50, False),
    (1, 7, 8192, 1024, 7168, 69, 5000, False), (2, 3, 8200, 9, 2000, 300, 5000, False), (1, 8, 16384, 1024, 15360, 69, 9000, False),
    # past the limits
    (1, 2, 16392, 20, 300, 69, 100, False), (1, 2, 2048, 1025, 300, 69, 6000, False), (1, 9, 2048, 513, 300, 69, 3000, False),
    (1, 16, 16384, 300, 7200, 69, 2000, False)])
def test_joined_step_equals_the_operators(dev, dtype, BG, gs, nc, np_, es, static, pages, on_device):
    """Steps whose attention's workgroups make the selection: the same lists, and outputs as above."""
    test_short_step_equals_the_operators(dev, dtype, BG, gs, nc, np_, es, static, pages, on_device)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("BG,gs,nc,np_,es,static,pages,on_device", [
    # who sums the scores: on both sides of 2048 clusters for seven and eight heads, of 4096 for six, with 1024 selecting threads too
    (2, 7, 2048, 36, 475, 69, 300, False), (2, 7, 2056, 36, 475, 69, 300, True), (3, 8, 2056, 600, 300, 69, 4000, False),
    (2, 6, 2056, 37, 470, 69, 300, False), (2, 6, 4096, 73, 950, 69, 600, False), (2, 6, 4104, 73, 950, 69, 600, True),
    (49, 7, 2432, 36, 475, 69, 300, True), (49, 7, 2440, 36, 475, 69, 300, True), (65, 8, 4096, 73, 950, 69, 600, False),
    # of 2048 for more than eight heads in many groups too, and for eight in up to 64
    (65, 16, 2048, 36, 475, 69, 300, False), (65, 16, 2056, 36, 475, 69, 300, False), (65, 9, 4096, 73, 950, 69, 600, True),
    (49, 12, 2432, 43, 560, 69, 300, False), (130, 10, 2064, 37, 478, 69, 300, True), (64, 8, 2056, 37, 476, 69, 300, False),
    (65, 8, 2056, 37, 476, 69, 300, False)])
def test_joined_step_at_the_line_of_the_sums(dev, dtype, BG, gs, nc, np_, es, static, pages, on_device):
    test_short_step_equals_the_operators(dev, dtype, BG, gs, nc, np_, es, static, pages, on_device)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("BG,gs,nc,np_,es,static,pages,on_device", [
    # more than eight heads over few clusters: one workgroup per group and several, few and many waves that score, no estimation zone,
    # a probe list that is all clusters, cut pages, and past the limits
    (1, 9, 8, 3, 2, 1, 100, False), (2, 16, 8, 8, 0, 0, 100, True), (5, 12, 40, 7, 33, 300, 100, False), (8, 16, 256, 5, 60, 70, 3, True),
    (3, 10, 264, 30, 200, 69, 300, False), (8, 12, 480, 9, 110, 98, 100, False), (2, 16, 512, 512, 0, 69, 2000, False),
    (1, 13, 512, 51, 461, 700, 500, True), (130, 9, 64, 6, 20, 90, 100, False), (256, 16, 32, 4, 8, 20, 100, False),
    (257, 16, 32, 4, 8, 20, 100, False)])
def test_few_clusters_of_many_heads(dev, dtype, BG, gs, nc, np_, es, static, pages, on_device):
    test_short_step_equals_the_operators(dev, dtype, BG, gs, nc, np_, es, static, pages, on_device)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gs,nc,np_,es,static,peak", [(4, 512, 9, 118, 69, 1), (4, 512, 9, 118, 98, 3), (8, 512, 12, 118, 120, 1),
                                                      (1, 496, 8, 115, 200, 1), (7, 384, 15, 100, 90, 3)])
def test_short_steps_of_several_workgroups_are_as_near_to_64_bits(dev, dtype, gs, nc, np_, es, static, peak):
    """Eight groups, which several workgroups each attend, and the same eight seventeen times over, which one workgroup each does:
    the errors of both against 64 bits.  A part rounds its probabilities to 16 bits against its own maximum and hands over 32 bits,
    so it is no further off; 5 % is what a norm over 8 * gs * 128 roundings moves by chance."""
    from retrievalattention_amd import kernels
    g = torch.Generator().manual_seed(gs * nc + static)
    rn = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)
    size = torch.randint(1, 32, (8, nc), generator=g, dtype=torch.int32)
    start, rows = (size.cumsum(1) - size).int().to(dev), int(size.sum(1).max()) + 1
    size16, size = size.to(dtype).to(dev), size.to(dev)
    q, cent = (peak * torch.randn(8, gs, 128, generator=g)).to(dtype).to(dev), rn(8, nc, 128)
    vs = (rn(8, nc, 128).float() * size[..., None].float().sqrt()).to(dtype)
    sk, sv, store_k, store_v = rn(8, static, 128), rn(8, static, 128), rn(8, rows, 128), rn(8, rows, 128)
    scale, outs = 128 ** -0.5, []
    for times in (1, 17):
        of = lambda t: t.repeat(times, *[1] * (t.dim() - 1))
        i32 = lambda *s: torch.zeros(s, dtype=torch.int32, device=dev)
        BG = 8 * times
        kept = dict(logits=torch.zeros(BG, gs, nc, device=dev), ret_ids=i32(BG, np_), est_ids=i32(BG, es),
                    ret_tok_off=i32(BG, np_ + 1), ret_start=i32(BG, np_), meta=i32(BG, 4), valid_lengths=i32(BG))
        outs.append(torch.empty(BG, gs, 128, dtype=dtype, device=dev))
        kernels.DecodeStepPlan(None, dtype, dict(
            kept, centroids=of(cent), mask=of(size == 0), cluster_size_i32=of(size), cluster_start=of(start), steady_k=of(sk),
            steady_v=of(sv), static_len_dev=None, store_k=of(store_k), store_v=of(store_v), value_sum=of(vs),
            cluster_size=of(size16)), np_, es, 8, 1000, scale).run(of(q), static, outs[-1])
        ids = kept["ret_ids"][:8], kept["est_ids"][:8]
    exact = torch.empty(8, gs, 128, dtype=torch.float64, device=dev)
    for x in range(8):
        ret, est = ids[0][x].tolist(), ids[1][x].long()
        at = torch.cat([torch.arange(int(start[x, c]), int(start[x, c] + size[x, c]), device=dev) for c in ret])
        k, v = torch.cat((sk[x], store_k[x, at], cent[x, est])).double(), torch.cat((sv[x], store_v[x, at], vs[x, est])).double()
        w = torch.cat((torch.ones(static + len(at), device=dev), size16[x, est].float())).double()
        p = torch.softmax(q[x].double() @ k.T * scale, dim=1)
        exact[x] = (p @ v) / (p @ w)[:, None]
    several, one = ((o[:8].double() - exact).norm() / exact.norm() for o in outs)
    assert several <= 1.05 * one and one <= (4e-3 if dtype == torch.bfloat16 else 5e-4), (float(several), float(one))

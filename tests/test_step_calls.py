"""The native calls of a decode step and of the operators (csrc/step_calls.cpp): what they leave to the general way, and that
both ways do the same."""
import math

import pytest
import torch

from retrievalattention_amd import kernels
from retrievalattention_amd._lib import step_calls

ROW = (2, 1, 3, 128)


def _rows(**change):
    t = dict(k=torch.zeros(ROW, dtype=torch.bfloat16), v=torch.zeros(ROW, dtype=torch.bfloat16),
             zk=torch.zeros(2, 3, 5, 128, dtype=torch.bfloat16), zv=torch.zeros(2, 3, 5, 128, dtype=torch.bfloat16), pos=1,
             at=None, shape=ROW)
    t.update(change)
    return t.values()


class _Sub(torch.Tensor):
    pass


def test_what_is_no_plain_device_tensor_is_left_to_the_general_way():
    """Host tensors, subclasses and other objects: nothing is launched, and nothing is raised."""
    native = step_calls()
    assert native.append(*_rows()) is None
    assert native.append(*_rows(k=torch.zeros(ROW, dtype=torch.bfloat16).as_subclass(_Sub))) is None
    assert native.append(*_rows(k=object())) is None and native.append(*_rows(at=3)) is None
    x = torch.zeros(8, dtype=torch.bfloat16)
    assert native.gemm_softmax(x, x, x, x, x, x, 1, 1, 1, 128, 1.0, 0.0) is None
    assert native.gather_vectors(x, x, x, x, x, x, x, 1, 1, 1, 1, 0, 1) is None
    assert native.flash(x, x, x, None, None, None, None, x, 1.0, False) is None
    with pytest.raises(TypeError):
        native.append(x)


def _gather_args(device="cpu", short=None):
    """Two groups, 24 rows each, 5 of them gathered; `short`: the argument that has an element too few."""
    e = lambda n, name, dt=torch.bfloat16: torch.zeros(n - (name == short), dtype=dt, device=device)  # noqa: E731
    return (e(2 * 24 * 128, "key_data"), e(2 * 8 * 128, "key_buffer"), e(2 * 24 * 128, "value_data"),
            e(2 * 8 * 128, "value_buffer"), e(2 * 24, "src_metadata"), e(2 * 8, "dst_metadata"),
            e(2 * 10, "data_offsets", torch.int64), 2, 24, 8, 10, 3, 5)


def _flash_args(device="cpu", short=None):
    """q, k, v, weight, previous_out, previous_lse, cache_seqlens of two groups of three heads over 24 rows; `short`: the one that
    has rows (k) or elements too few."""
    z = lambda *s, dt=torch.bfloat16: torch.zeros(s, dtype=dt, device=device)  # noqa: E731
    e = lambda n, name, dt=torch.bfloat16: z(n - (name == short), dt=dt)  # noqa: E731
    return (z(2, 1, 3, 128), z(2 - (short == "k"), 24, 1, 128), e(2 * 24 * 128, "v"), e(2 * 24, "weight"),
            e(2 * 3 * 128, "previous_out"), e(2 * 3, "previous_lse", torch.float32), e(2, "cache_seqlens", torch.int32))


GATHERED = ("key_data", "key_buffer", "value_data", "value_buffer", "src_metadata", "dst_metadata", "data_offsets")
ATTENDED = ("k", "v", "weight", "previous_out", "previous_lse", "cache_seqlens")


@pytest.mark.parametrize("short", (None,) + GATHERED + ATTENDED)
def test_short_buffers_are_refused_before_a_launch(monkeypatch, short):
    """The wrappers' general way, on host tensors that it is told to take: nothing is called with a buffer that is smaller than
    the other arguments say."""
    calls = []

    class Library:
        def __getattr__(self, name):
            return lambda *a: calls.append(name) or 0
    for name in ("_need", "_need_all"):
        monkeypatch.setattr(kernels, name, lambda *a, **k: None)
    monkeypatch.setattr(kernels, "lib", Library)
    monkeypatch.setattr(kernels, "_stream", lambda: 0)
    monkeypatch.setattr(kernels, "_workspace", lambda *a: torch.zeros(1))
    monkeypatch.setattr(kernels, "_flash_workspace_bytes", lambda *a: 256)   # (it keeps what the library says)
    for names, call in ((GATHERED, lambda: kernels.gather_copy_vectors(*_gather_args(short=short))),
                        (ATTENDED, lambda: kernels.weighted_flash_decoding(*_flash_args(short=short)))):
        calls.clear()
        if short in names:
            with pytest.raises(ValueError, match="smaller"):
                call()
            assert not calls
        else:
            call()
            assert len(calls) == 1


@pytest.mark.gpu
def test_short_buffers_are_left_to_the_general_way(dev):
    """The native calls launch nothing then, and the general way raises."""
    native = step_calls()
    assert native.gather_vectors(*_gather_args(dev)) == 0
    ws = kernels._workspace(kernels._flash_workspace_bytes(2, 3), dev, "attn")
    assert isinstance(native.flash(*_flash_args(dev), ws, 1.0, False), torch.Tensor)
    for short in GATHERED:
        assert native.gather_vectors(*_gather_args(dev, short)) is None, short
        with pytest.raises(ValueError):
            kernels.gather_copy_vectors(*_gather_args(dev, short))
    for short in ATTENDED:
        assert native.flash(*_flash_args(dev, short), ws, 1.0, False) is None, short
        with pytest.raises(ValueError):
            kernels.weighted_flash_decoding(*_flash_args(dev, short))


@pytest.mark.gpu
@pytest.mark.parametrize("change,takes", [
    (dict(), True), (dict(pos=4), True), (dict(pos=5), False), (dict(shape=(2, 1, 3)), False), (dict(shape=(2, 3, 1, 128)), False),
    (dict(zk=torch.zeros(2, 3, 5, 128)), False), (dict(zk=torch.zeros(2, 5, 3, 128, dtype=torch.bfloat16).transpose(1, 2)), False),
    (dict(k=torch.zeros(2, 3, 1, 128, dtype=torch.bfloat16).transpose(1, 2)), True),
    (dict(k=torch.zeros(2, 1, 128, 3, dtype=torch.bfloat16).transpose(2, 3)), False),
    (dict(v=torch.zeros(2 * 3 * 128 + 4, dtype=torch.bfloat16)[4:].view(ROW)), False),
    (dict(at=torch.tensor([2])), True), (dict(at=torch.tensor([2], dtype=torch.int32)), False),
    (dict(at=torch.tensor([7])), True)])
def test_append_takes_rows_as_a_layer_hands_them_over(dev, change, takes):
    args = [x.to(dev) if isinstance(x, torch.Tensor) else x for x in _rows(**change)]
    if "v" in change:   # (a copy would be aligned)
        args[1] = torch.zeros(2 * 3 * 128 + 4, dtype=torch.bfloat16, device=dev)[4:].view(ROW)
    k, v, zk, zv, pos, at, shape = args
    k.normal_(), v.normal_()
    before = zk.clone(), zv.clone()
    assert kernels.append_row(k, v, zk, zv, pos, at, shape) is takes
    row = pos if at is None else int(at)
    if takes and row < 5:
        before[0][:, :, row], before[1][:, :, row] = k[:, 0], v[:, 0]
    assert torch.equal(zk, before[0]) and torch.equal(zv, before[1])


@pytest.mark.gpu
@pytest.mark.parametrize("residency", ["device", "device-pos", "host"])
def test_step_follows_its_buffers(dev, residency):
    """A prepared step in native code gives what the general way gives, also behind a buffer that was replaced, another number
    of probes, and queries of a subclass."""
    from tests.test_gpu_cache import _gen, _make_cache, _prefill
    ctx = 1024 + 68
    cache = _make_cache(dev, residency, 1, 2, 2, 4, ctx, 64, 1, 8, 16)
    _prefill(cache, *_gen(1, 2, 2, 4, ctx, 64, dev, 5), 1, 2)
    cache.layer_num = 2   # (no layer is the last one: the same token again)
    q = torch.randn(2, 1, 8, 128, device=dev).bfloat16()
    plan = lambda: cache._plans[(0, 0)]
    general, native = cache.compute(q, 0), cache.compute(q, 0)
    assert torch.equal(general, native) and native.shape == general.shape and plan()._native is not None
    first = plan()
    cache.value_sum[0] = cache.value_sum[0].clone() * 2
    moved = cache.compute(q, 0)
    assert plan() is not first and not torch.equal(moved, general)
    assert torch.equal(cache.compute(q, 0), moved)
    assert torch.equal(cache.compute(q.as_subclass(_Sub), 0).as_subclass(torch.Tensor), moved)
    cache.nprobe -= 1
    other = cache.compute(q, 0)
    assert not torch.equal(other, moved) and torch.equal(cache.compute(q, 0), other)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_operators_natively_and_in_general(dev, dtype):
    """The same call with plain tensors and with a subclass, which takes the general way."""
    g = torch.Generator(device=dev).manual_seed(3)
    r = lambda *s, dt=dtype: torch.randn(s, generator=g, device=dev).to(dt)
    BG, gs, n, rows = 3, 5, 264, 40
    q, cent, keys, values, weight = r(BG, 1, gs, 128), r(BG, n, 128), r(BG, rows, 1, 128), r(BG, rows, 1, 128), \
        r(BG, 1, 1, rows).abs()
    lengths = torch.tensor([40, 7, 23], dtype=torch.int32, device=dev)
    ids = torch.stack([torch.randperm(n, generator=g, device=dev) for _ in range(BG)])
    results = []
    for of in (lambda t: t, lambda t: t.as_subclass(_Sub)):
        product, softmax = (torch.zeros(BG, gs, n, dtype=dtype, device=dev) for _ in range(2))
        norm, total = (torch.zeros(BG, 2, gs, device=dev) for _ in range(2))
        kernels.batch_gemm_softmax(of(q), cent, product, norm, total, softmax, BG, gs, n, 128, 1 / math.sqrt(128))
        bk, bv, bs = torch.zeros_like(keys), torch.zeros_like(values), torch.zeros_like(weight)
        kernels.gather_copy_vectors(of(cent), bk, cent, bv, r(BG, n) * 0 + 1, bs, ids, BG, n, rows, n, 3, rows)
        a, lse = kernels.weighted_flash_decoding(of(q), keys, values, weight, return_softmax_lse=True)
        b = kernels.weighted_flash_decoding(of(q), keys, values, previous_out=a.as_subclass(torch.Tensor),
                                            previous_lse=lse.as_subclass(torch.Tensor), cache_seqlens=lengths)
        results.append([x.as_subclass(torch.Tensor) for x in (product, softmax, norm, total, bk, bv, bs, a, lse, b)])
    for x, y in zip(*results):
        assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)
    with pytest.raises(ValueError):
        kernels.batch_gemm_softmax(q, cent, product, norm[:1], total, softmax, BG, gs, n, 128)


@pytest.mark.gpu
def test_numbers_that_the_native_call_does_not_take(dev):
    """What float() takes and PyFloat does not goes the general way; sizes past 64 bits are refused as sizes past the buffers are."""
    z = lambda *s, dt=torch.bfloat16: torch.zeros(s, dtype=dt, device=dev)  # noqa: E731
    a, b = z(1, 2, 128) + 1, z(1, 8, 128) + 1
    out = []
    for alpha, beta in ((0.5, 0.0), ("0.5", "0")):
        out.append(z(1, 2, 8))
        kernels.batch_gemm_softmax(a, b, out[-1], z(1, 1, 2, dt=torch.float32), z(1, 1, 2, dt=torch.float32), z(1, 2, 8), 1, 2, 8,
                                   128, alpha, beta)
    assert torch.equal(*out) and float(out[0][0, 0, 0]) == 64.0
    for m, n in ((1 << 70, 8), (2, 1 << 70), (1 << 40, 8)):
        with pytest.raises(ValueError):
            kernels.batch_gemm_softmax(a, b, out[0], z(1, 1, 2, dt=torch.float32), z(1, 1, 2, dt=torch.float32), z(1, 2, 8), 1, m, n,
                                       128)

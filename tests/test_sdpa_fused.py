"""The one-kernel attention path (bf16 / f16, head size 64 or 128) at the sizes where it can go wrong: ends of the tiles
of 32 / 64 keys and 32 / 128 query rows, both forms around 64 rows, keys split over workgroups, masks whose rows start at
any element or whose keys do not lie side by side, rows without a key, strided and broadcast tensors, and buffers it does
not take (the composition runs then)."""
import ctypes as C

import numpy as np
import pytest

from onednn_amd import cabi, dnnl
from tests.test_sdpa import DT, ideal, make, md4, run, storage, tolerance, values
from onednn_amd.problem import storage_dtype
from tests.test_inner_product import encode

SHAPES = [  # b, h, hk, sq, sk
    (1, 2, 2, 1, 1), (2, 3, 3, 1, 31), (1, 2, 2, 3, 33), (1, 4, 1, 16, 64), (1, 4, 1, 17, 65),   # few rows, 64 and 68
    (1, 2, 2, 64, 63), (1, 2, 2, 65, 64), (1, 1, 1, 128, 65), (1, 3, 1, 129, 191), (2, 2, 2, 257, 40),
    (1, 2, 1, 1, 3000), (1, 1, 1, 200, 2500),                                                        # split keys
]


ONE_KERNEL = "hip:sdpa(hip:mfma_sdpa:gfx950)"


def check(dt, d, shape, **kw):
    b, h, hk, sq, sk = shape
    q, k, v = make(21, b, h, hk, sq, sk, d, d, dt, mag=kw.pop("mag", 1.0))
    sc = np.array([kw.pop("sc", 1.0 / np.sqrt(d))], np.float32)
    mask = kw.pop("mask", None)
    got, impl = run(q, k, v, dt, dt, True, scale=sc, mask=mask, mask_type=kw.get("mask_type", 0))
    want, pabs = ideal(q, k, v, dt, scale=float(sc[0]), mask=None if mask is None else mask.astype(np.float64),
                       mask_type=kw.get("mask_type", 0))
    assert impl == ONE_KERNEL
    err = np.abs(values(dt, got) - want)
    tol = tolerance(dt, dt, sk, pabs, want)
    assert (err <= tol).all(), f"{impl}: worst {np.nanmax(err / tol):.2f} of the bound"


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_edges_of_the_tiles(gpu, dt, d, shape):
    check(dt, d, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 2, 2, 200, 200), (1, 4, 1, 40, 150), (1, 2, 2, 150, 333)])
@pytest.mark.parametrize("mask_type", [1, 2, 3])
def test_masks_and_a_negative_scale(gpu, shape, mask_type):
    b, h, hk, sq, sk = shape
    mask = (np.random.default_rng(5).standard_normal((1, 1, sq, sk)) * 2).astype(np.float32) if mask_type == 1 else None
    check("bf16", 64, shape, mask=mask, mask_type=mask_type, sc=-0.11)


def run_views(q, k, v, dt, mask=None, mdt=None, mask_type=0, alg=dnnl.softmax_accurate, dst_bshd=False):
    """As `run`, every tensor with the strides of its numpy view; dst stored [b][h][s][d] or [b][s][h][d]."""
    eng = dnnl.engine(dnnl.gpu, 0)
    strm = dnnl.stream(eng)
    (b, h, sq, d), hk = q.shape, k.shape[1]
    view_md = lambda x, t: dnnl.memory_desc(list(x.shape), DT[t], strides=[n // x.itemsize for n in x.strides])  # noqa: E731
    d_md = dnnl.memory_desc([b, h, sq, d], DT[dt], strides=[sq * h * d, d, h * d, 1] if dst_bshd else [h * sq * d, sq * d, d, 1])
    m_md = None if mask is None else view_md(mask, mdt)
    pd = dnnl.sdpa_primitive_desc(eng, view_md(q, dt), view_md(k, dt), view_md(v, dt), d_md, mask_md=m_md, kv_head_number=hk,
                                  attn_mask_type=mask_type, softmax_alg=alg)
    assert pd.impl_info_str() == ONE_KERNEL
    dst = dnnl.memory(d_md, eng)
    args = {arg: dnnl.memory(view_md(x, dt), eng, storage(x)) for arg, x in
            ((dnnl.ARG_QUERIES, q), (dnnl.ARG_KEYS, k), (dnnl.ARG_VALUES, v))}
    args[dnnl.ARG_DST] = dst
    if mask is not None:
        args[dnnl.ARG_ATTN_MASK] = dnnl.memory(m_md, eng, storage(mask))
    dnnl.sdpa(pd).execute(strm, args)
    strm.wait()
    got = dst.read(storage_dtype(DT[dt]))
    got = got.reshape(b, sq, h, d).transpose(0, 2, 1, 3) if dst_bshd else got.reshape(b, h, sq, d)
    return values(dt, got)


def within(dt, got, want, pabs, v, rows=slice(None)):
    """`tolerance`, and for f16 half a step of its subnormals (2^-25) for dst and for every probability, which meets |v| and
    a division by a sum of at least 1: without a scale the scores spread over dozens of units of e."""
    tol = tolerance(dt, dt, v.shape[2], pabs, want)
    if dt == "f16":
        tol = tol + 2.0 ** -25 * (1 + np.abs(values(dt, v)).sum(axis=2, keepdims=True))
    return (np.abs(got - want) <= tol)[:, :, rows].all()


@pytest.mark.gpu
@pytest.mark.parametrize("alg", [dnnl.softmax_accurate, dnnl.softmax_accurate_inf_as_zero])
@pytest.mark.parametrize("dt,d", [("bf16", 64), ("f16", 128)])
@pytest.mark.parametrize("mask_type,shape", [(1, (1, 2, 2, 6, 40)), (1, (1, 2, 2, 130, 200)), (1, (1, 1, 1, 130, 2500)),
                                             (1, (1, 2, 1, 3, 3000)), (3, (1, 2, 2, 200, 70)), (3, (1, 1, 1, 600, 500)),
                                             (3, (1, 2, 1, 20, 9))])
def test_rows_without_a_key(gpu, mask_type, shape, dt, d, alg):
    """0 / 0, or zeros if asked for, in both forms and with the keys of one and of several parts; the rows beside them."""
    b, h, hk, sq, sk = shape
    q, k, v = make(26, b, h, hk, sq, sk, d, d, dt)
    mask = None
    if mask_type == 1:
        mask = (np.random.default_rng(7).standard_normal((1, 1, sq, sk)) * 2).astype(np.float32)
        mask[0, 0, [1, sq - 1]] = -np.inf
    got = run_views(q, k, v, dt, mask, "f32", mask_type, alg)
    want, pabs = ideal(q, k, v, dt, mask=None if mask is None else mask.astype(np.float64), mask_type=mask_type)
    none = np.isnan(want).all(axis=(0, 1, 3))
    assert none.sum() == (2 if mask_type == 1 else sq - sk)
    empty = got[:, :, none]
    assert np.isnan(empty).all() if alg == dnnl.softmax_accurate else not empty.any()
    assert within(dt, got, want, pabs, v, ~none)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,d", [("bf16", 128), ("f16", 64)])
@pytest.mark.parametrize("mask_type", [2, 3])
@pytest.mark.parametrize("shape", [(1, 1, 1, 200, 2500), (1, 2, 1, 16, 3000), (1, 1, 1, 1500, 1500), (2, 1, 1, 33, 1000)])
def test_causal_masks_with_split_keys(gpu, shape, mask_type, dt, d):
    check(dt, d, shape, mask_type=mask_type)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 2, 2, 150, 200), (2, 2, 2, 3, 200), (1, 4, 1, 40, 131)])
@pytest.mark.parametrize("mdt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("layout", ["shared", "per head", "per batch", "keys apart", "one key", "one query"])
def test_mask_layouts(gpu, layout, mdt, shape):
    b, h, hk, sq, sk = shape
    dims = {"per head": (1, h, sq, sk), "per batch": (b, 1, sq, sk), "one key": (b, h, sq, 1), "one query": (1, h, 1, sk)}
    dims = dims.get(layout, (1, 1, sq, sk))
    raw = encode((np.random.default_rng(8).standard_normal(dims) * 2).astype(np.float32), mdt)
    if layout == "keys apart":   # [..][keys][queries] in memory
        raw = np.ascontiguousarray(raw.transpose(0, 1, 3, 2)).transpose(0, 1, 3, 2)
    q, k, v = make(27, b, h, hk, sq, sk, 128, 128, "bf16")
    want, pabs = ideal(q, k, v, "bf16", mask=values(mdt, raw))
    assert within("bf16", run_views(q, k, v, "bf16", raw, mdt, 1), want, pabs, v)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 4, 4, 150, 200), (2, 4, 1, 33, 70), (2, 4, 1, 5, 1200)])
def test_heads_inside_the_rows_and_keys_of_one_batch(gpu, shape):
    """q, k, v and dst stored [b][s][h][d]; then keys and values of one batch under two."""
    b, h, hk, sq, sk = shape
    r = np.random.default_rng(28)
    bshd = lambda n, s, heads: encode(r.standard_normal((n, s, heads, 64)).astype(np.float32), "f16").transpose(0, 2, 1, 3)  # noqa: E731
    for kb in (b, 1):
        q, k, v = bshd(b, sq, h), bshd(kb, sk, hk).transpose(0, 1, 3, 2), bshd(kb, sk, hk)
        want, pabs = ideal(q, k, v, "f16")
        assert within("f16", run_views(q, k, v, "f16", dst_bshd=True), want, pabs, v)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 2, 2, 3, 33), (1, 2, 2, 90, 100), (1, 1, 1, 3, 600)])
@pytest.mark.parametrize("sc,mag", [(0.0, 1.0), (-0.0, 1.0), (1e-35, 1e17), (-1e-38, 2e18)])
@pytest.mark.parametrize("mask_type", [0, 3])
def test_scales_at_and_near_zero(gpu, shape, sc, mag, mask_type):
    """Small scales of large scores are used as they are (a subnormal one too); with a scale of zero every key that is
    seen weighs the same and masked ones weigh nothing."""
    check("bf16", 64, shape, sc=sc, mag=mag, mask_type=mask_type)


@pytest.mark.gpu
def test_unaligned_buffers_run_the_composition(gpu):
    """q one element off a 16-byte boundary: the same result within the same bound."""
    b, h, sq, sk, d = 1, 2, 40, 72, 64
    q, k, v = make(22, b, h, h, sq, sk, d, d, "bf16")
    eng = dnnl.engine(dnnl.gpu, 0)
    strm = dnnl.stream(eng)
    mds = [md4(q.shape, "bf16"), md4(k.shape, "bf16", transposed=True), md4(v.shape, "bf16"), md4((b, h, sq, d), "bf16")]
    pd = dnnl.sdpa_primitive_desc(eng, *mds)
    prim = dnnl.sdpa(pd)
    flat = np.zeros(q.size + 1, storage_dtype(DT["bf16"]))
    flat[1:] = storage(q).reshape(-1)
    raw = cabi.DeviceBuffer.from_numpy(flat)
    qm = dnnl.memory.__new__(dnnl.memory)
    qm.md, qm.engine, qm.h = mds[0], eng, C.c_void_p()
    assert dnnl.lib().dnnl_memory_create(C.byref(qm.h), mds[0].h, eng.h, C.c_void_p(raw.ptr + 2)) == dnnl.success
    dst = dnnl.memory(mds[3], eng)
    args = {dnnl.ARG_QUERIES: qm, dnnl.ARG_KEYS: dnnl.memory(mds[1], eng, storage(k)),
            dnnl.ARG_VALUES: dnnl.memory(mds[2], eng, storage(v)), dnnl.ARG_DST: dst}
    want, pabs = ideal(q, k, v, "bf16")

    def matches():
        got = values("bf16", dst.read(storage_dtype(DT["bf16"])).reshape(b, h, sq, d))
        return (np.abs(got - want) <= tolerance("bf16", "bf16", sk, pabs, want)).all()

    for _ in range(2):
        prim.execute(strm, args)
        strm.wait()
        assert matches()
    # a primitive whose first execution is recorded: the composition is set up under the capture
    hs = cabi.Stream()
    strm = dnnl.stream(eng, hip_stream=hs.ptr)
    prim = dnnl.sdpa(pd)
    with cabi.Graph(hs) as g:
        prim.execute(strm, args)
    try:
        for _ in range(3):
            dst.write(np.zeros((b, h, sq, d), storage_dtype(DT["bf16"])))
            assert not matches()
            g.launch()
            hs.sync()
            assert matches()
    finally:
        g.destroy()
        hs.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("what,shape", [("k", (1, 64, 64, 2048, 2048)), ("q", (1, 2, 2, 200, 200)), ("q", (1, 4, 1, 9, 1100)),
                                        ("mask", (1, 1, 1, 300, 400))])
def test_dst_in_the_memory_of_an_input(gpu, what, shape):
    """The keys, the queries and a mask are read before dst is stored, wherever dst lies: what a dst of its own holds."""
    b, h, hk, sq, sk = shape
    d = 64
    eng = dnnl.engine(dnnl.gpu, 0)
    strm = dnnl.stream(eng)
    q, k, v = make(25, b, h, hk, sq, sk, d, d, "bf16")
    mds = [md4(q.shape, "bf16"), md4(k.shape, "bf16", transposed=True), md4(v.shape, "bf16"), md4((b, h, sq, d), "bf16")]
    mask = (np.random.default_rng(6).standard_normal((1, 1, sq, sk)) * 2).astype(np.float32) if what == "mask" else None
    m_md = md4(mask.shape, "f32") if what == "mask" else None
    prim = dnnl.sdpa(dnnl.sdpa_primitive_desc(eng, *mds, mask_md=m_md, kv_head_number=hk, attn_mask_type=int(what == "mask")))

    def result(shared):
        args = {dnnl.ARG_QUERIES: dnnl.memory(mds[0], eng, storage(q)), dnnl.ARG_KEYS: dnnl.memory(mds[1], eng, storage(k)),
                dnnl.ARG_VALUES: dnnl.memory(mds[2], eng, storage(v)), dnnl.ARG_DST: dnnl.memory(mds[3], eng)}
        if what == "mask":
            args[dnnl.ARG_ATTN_MASK] = dnnl.memory(m_md, eng, mask)
        if shared:
            dst = dnnl.memory.__new__(dnnl.memory)
            dst.md, dst.engine, dst.h = mds[3], eng, C.c_void_p()
            at = args[{"k": dnnl.ARG_KEYS, "q": dnnl.ARG_QUERIES, "mask": dnnl.ARG_ATTN_MASK}[what]].get_data_handle()
            assert dnnl.lib().dnnl_memory_create(C.byref(dst.h), mds[3].h, eng.h, C.c_void_p(at)) == dnnl.success
            args[dnnl.ARG_DST] = dst
        prim.execute(strm, args)
        strm.wait()
        return values("bf16", args[dnnl.ARG_DST].read(storage_dtype(DT["bf16"])))

    own, inside = result(False), result(True)
    if what == "q":   # in place, element for element: the same kernel
        assert np.array_equal(own, inside)
    else:             # both paths round the probabilities and dst once, 2^-8 of a value each
        assert np.linalg.norm(own - inside) <= 2 * 2.0 ** -8 * np.linalg.norm(own)


@pytest.mark.gpu
@pytest.mark.parametrize("mdt,lowest", [("f32", np.finfo(np.float32).min), ("bf16", -3.3895313892515355e38), ("f16", -65504.0)])
@pytest.mark.parametrize("shape", [(1, 2, 2, 150, 333), (1, 2, 2, 3, 1200)])
def test_mask_of_the_types_lowest_value(gpu, shape, mdt, lowest):
    """Not -inf: a query all of whose keys are masked so weighs them alike in f32 (the scores vanish beside the mask;
    65504 in f16 leaves them), the others see what is left."""
    b, h, hk, sq, sk = shape
    q, k, v = make(23, b, h, hk, sq, sk, 64, 64, "bf16")
    mask = np.zeros((1, 1, sq, sk), np.float32)
    mask[..., : sk // 2] = lowest
    mask[:, :, 1, :] = lowest
    stored = {"f32": mask, "bf16": (mask.view(np.uint32) >> 16).astype(np.uint16), "f16": mask.astype(np.float16).view(np.uint16)}[mdt]
    sc = np.array([0.125], np.float32)
    got, impl = run(q, k, v, "bf16", "bf16", True, scale=sc, mask=stored, mdt=mdt, mask_type=1)
    assert impl == ONE_KERNEL
    want, pabs = ideal(q, k, v, "bf16", scale=0.125, mask=mask.astype(np.float64))
    if mdt != "f16":
        want[:, :, 1, :] = values("bf16", v).astype(np.float64).mean(axis=2)
        pabs[:, :, 1, :] = np.abs(values("bf16", v)).astype(np.float64).mean(axis=2)
    else:   # a score beside 65504 is rounded to 2^-8, so a weight and their sum move by 2^-9 each: twice bf16's 2^-8
        pabs = 2 * pabs
    assert (np.abs(values("bf16", got) - want) <= tolerance("bf16", "bf16", sk, pabs, want)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 2, 2, 129, 65), (1, 2, 2, 3, 33)])
def test_an_infinite_last_value_stays_infinite(gpu, shape):
    """The tile's rows beyond the last key must not turn it into NaN."""
    b, h, hk, sq, sk = shape
    q, k, v = make(24, b, h, hk, sq, sk, 64, 64, "bf16")
    v[:, :, sk - 1, 5] = 0x7f80
    got, impl = run(q, k, v, "bf16", "bf16", True)
    got = values("bf16", got)
    assert impl == ONE_KERNEL and np.isposinf(got[..., 5]).all()
    assert np.isfinite(np.delete(got, 5, axis=3)).all()

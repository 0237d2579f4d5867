"""The decode kernels with f16 activations: against the oracle under the bound of the factored sum (the f16 form keeps
64 + w where the bf16 form keeps 128 + w, so tests/helpers.py decode_bound covers it), one-hot rows bit for bit, and
infinite activations, whose factored sums are NaN where the terms' sum is an infinity.
"""
import numpy as np
import pytest

from onednn_amd import cabi, configs
from onednn_amd import dtypes as dtp
from onednn_amd.problem import GpuRun, run_gpu
from tests.helpers import assert_bit_exact, assert_decode_close, decode

IMPLS = {"plain": (cabi.IMPL_WOQ_GEMV, "hip:woq_gemv"), "packed": (cabi.IMPL_WOQ_PACKED, "hip:woq_packed")}


def f16_problem(M, N, K, group, layout, wdt="u4", sdt="f16", zdt="u4", zkind="grouped", ddt="f16", relu_bias=False):
    p = configs.woq_variant(M, N, K, group, wei_dt=wdt, sc_dt=sdt, zp_dt=zdt, zp_kind=zkind, dst_dt=ddt, relu_bias=relu_bias)
    src = decode(p.src_dt, p.src, M * K).astype(np.float32).reshape(M, K)
    p.src, p.src_dt = src.astype(np.float16).view(np.uint16), cabi.DT_F16
    if layout == "packed":
        p.wei_packing = cabi.WEI_PACK_WOQ64
    return p


def test_f16_activations_take_the_decode_kernels():
    for layout, (_, name) in IMPLS.items():
        for M, N, K, group in [(1, 128, 128, 128), (32, 192, 8320, 64)]:
            st, impl = cabi.query(f16_problem(M, N, K, group, layout).desc())
            assert st == cabi.SUCCESS and cabi.impl_name(impl).startswith(name)
    assert cabi.impl_name(cabi.query(f16_problem(33, 128, 128, 128, "plain").desc())[1]).startswith("hip:mfma_h16")


CASES = [
    # M, N, K, group, weights, scales, zero points, dst, bias + relu
    (1, 64, 32, 32, "u4", "f16", "u4", "grouped", "f16", False),
    (1, 1280, 7680, 64, "s4", "f16", "u4", "none", "f16", False),
    (4, 320, 8320, 128, "u4", "f16", "u4", "grouped", "f32", False),
    (8, 192, 1056, 1056, "u4", "f32", "u8", "common", "f32", True),
    (13, 256, 2048, 512, "s4", "f16", "s8", "grouped", "f16", True),
    (16, 4160, 384, 128, "u4", "f32", "s32", "grouped", "f32", False),
    (17, 256, 2048, 128, "s4", "bf16", "s4", "column", "f16", False),
    (32, 128, 3072, 64, "u4", "f16", "u4", "grouped", "f16", False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("layout", IMPLS)
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c))
def test_f16_attribute_variants(gpu, oracle, case, layout):
    M, N, K, group, wdt, sdt, zdt, zkind, ddt, relu_bias = case
    p = f16_problem(M, N, K, group, layout, wdt, sdt, zdt, zkind, ddt, relu_bias)
    got, name = run_gpu(p, cabi.IMPL_AUTO)
    assert name.startswith(IMPLS[layout][1])
    _, ideal, asum = oracle.run_oracle(p, want_ideal=True)
    assert_decode_close(p, got, ideal, asum, what=name)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", IMPLS)
@pytest.mark.parametrize("K,group", [(32, 32), (256, 64), (512, 128), (2048, 2048)])
def test_f16_one_hot_rows_are_exact(gpu, oracle, layout, K, group):
    M = 32
    p = f16_problem(M, 128, K, group, layout, ddt="f32")
    hot = np.zeros((M, K), np.float16)
    r = np.random.default_rng(K)
    hot[np.arange(M), r.choice(K, size=M, replace=K < M)] = 1.0
    p.src = hot.view(np.uint16)
    got, name = run_gpu(p, IMPLS[layout][0])
    assert_bit_exact(p, got, oracle.run_oracle(p), name)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", IMPLS)
@pytest.mark.parametrize("M,K,wdt,zkind,ddt,relu_bias", [(3, 512, "u4", "grouped", "f32", False), (20, 512, "s4", "none", "f16", True),
                                                         (12, 4096, "s4", "common", "f16", False)])
def test_f16_infinite_activations(gpu, oracle, layout, M, K, wdt, zkind, ddt, relu_bias):
    # weights and zero points that never meet (w - zp is not 0), infinities of one sign per row: no term is NaN
    p = f16_problem(M, 192, K, 128, layout, wdt=wdt, zkind=zkind, zdt="u4" if wdt == "u4" else "s8", ddt=ddt, relu_bias=relu_bias)
    r = np.random.default_rng(5)
    p.wei = dtp.pack_nibbles(r.integers(1, 8, size=(K, 192), dtype=np.uint8))
    if "wei_zp" in p.quant:
        z = p.quant["wei_zp"].data
        z[...] = 0x99 if wdt == "u4" else -3
    src = np.asarray(p.src).view(np.float16).reshape(M, K)
    src[0, K - 1] = np.inf
    src[1, 0] = -np.inf
    src[2, K // 2] = np.nan
    p.src = src.view(np.uint16)
    got, name = run_gpu(p, IMPLS[layout][0])
    want = oracle.run_oracle(p)
    g, w = (decode(p.dst_dt, x, M * 192).astype(np.float64).reshape(M, 192)[:3] for x in (got, want))
    np.testing.assert_array_equal(g, w)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", IMPLS)
@pytest.mark.parametrize("M,K,group,fill", [(2, 8320, 64, "a row"), (32, 1056, 1056, "a row"), (5, 2048, 128, "every 37th"),
                                            (17, 4096, 512, "scales")])
def test_f16_sums_that_are_not_finite(gpu, oracle, layout, M, K, group, fill):
    """rows of infinities and infinite scales; no w is 0, so no term is NaN"""
    N = 192
    p = f16_problem(M, N, K, group, layout, sdt="f32", zkind="none", ddt="f32")
    r = np.random.default_rng(K)
    p.wei = dtp.pack_nibbles(r.integers(1, 16, size=(K, N), dtype=np.uint8))
    src = np.asarray(p.src).view(np.float16).reshape(M, K)
    src[src == 0] = 1
    bad = M - 1
    if fill == "a row":
        src[bad] = np.inf
    elif fill == "every 37th":
        src[bad, 5::37] = -np.inf
    else:
        src[...] = np.abs(src)
        p.quant["wei_scale"].data.reshape(-1, N)[-1, ::7] = np.inf
    p.src = src.view(np.uint16)
    got, name = run_gpu(p, IMPLS[layout][0])
    want = oracle.run_oracle(p)
    g, w = (decode(p.dst_dt, x, M * N).astype(np.float64).reshape(M, N) for x in (got, want))
    special = ~np.isfinite(w)
    assert special.any()
    np.testing.assert_array_equal(g[special], w[special])
    assert np.isfinite(g[~special]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("layout", IMPLS)
@pytest.mark.parametrize("M,times", [(1, 8), (32, 32)])
def test_f16_infinite_activations_take_no_walk_along_k(gpu, layout, M, times):
    """An infinity in a row is looked up in a pass over the row's activations, a few latencies for a wavefront's part of K and row:
    at most a launch more where M is 1 (measured 1.2 times the time), and 2.9 and 4.1 times with one in each of 32 rows.  A
    walk of every element over all of K, a term after the other, took 16384 latencies: 400 to 900 times."""
    import ctypes as C
    lib = cabi.load_kernels()
    p = f16_problem(M, 8192, 16384, 128, layout)
    clean, src = p.src, np.asarray(p.src).view(np.float16).reshape(M, -1).copy()
    src[:, 4097] = np.inf
    ms = {}
    for what, values in (("finite", clean), ("infinite", src.view(np.uint16))):
        p.src = values
        run = GpuRun(p, IMPLS[layout][0])
        ev = [C.c_void_p(), C.c_void_p()]
        for e in ev:
            cabi.check(lib.mi355_event_create(C.byref(e)))
        try:
            run.launch()
            cabi.check(lib.mi355_event_record(ev[0], None))
            for _ in range(4):
                run.launch()
            cabi.check(lib.mi355_event_record(ev[1], None))
            cabi.check(lib.mi355_event_sync(ev[1]))
            t = C.c_float()
            cabi.check(lib.mi355_event_elapsed_ms(C.byref(t), ev[0], ev[1]))
            ms[what] = t.value / 4
        finally:
            run.free()
            for e in ev:
                lib.mi355_event_destroy(e)
    assert ms["infinite"] < times * ms["finite"], ms


@pytest.mark.parametrize("dt,M,N,K", [("f16", 1, 14336, 4096), ("f16", 32, 64, 128), ("f16", 4, 1024, 16384), ("bf16", 8, 8128, 4096),
                                      ("bf16", 24, 6144, 11776)])
def test_format_any_weights_that_are_row_major(dt, M, N, K):
    """what a caller does with them: asks for strides, quantizes f32 into them, hands them to a primitive of more rows"""
    from onednn_amd import dnnl
    eng = dnnl.engine(dnnl.gpu, 0)
    attr = dnnl.primitive_attr()
    attr.set_scales(dnnl.ARG_WEIGHTS, 3, (128, 1), cabi.DT_NAMES[dt])
    attr.set_fpmath_mode(dnnl.fpmath_bf16 if dt == "bf16" else dnnl.fpmath_f16, True)
    md = lambda dims, t, tag=dnnl.tag_ab: dnnl.memory_desc(dims, cabi.DT_NAMES[t], tag=tag)  # noqa: E731
    pd = dnnl.matmul_primitive_desc(eng, md([M, K], dt), md([K, N], "u4", dnnl.tag_any), md([M, N], dt), attr=attr)
    assert pd.impl_info_str().startswith("hip:woq_gemv")
    wmd = pd.query_md(dnnl.query_weights_md)
    assert wmd.strides() == [N, 1]
    quantize = dnnl.primitive_attr()
    quantize.set_scales(dnnl.ARG_SRC, 3, (128, 1), cabi.DT_F32)
    dnnl.reorder_primitive_desc(eng, md([K, N], "f32"), eng, wmd, attr=quantize)
    prompt = dnnl.matmul_primitive_desc(eng, md([512, K], dt), wmd, md([512, N], dt), attr=attr)
    assert prompt.impl_info_str().startswith("hip:mfma_h16")

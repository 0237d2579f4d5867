"""32 x 32 tiles of 16-bit, fp8 and block-scaled operands (onednn_amd/csrc/kern_chain_small.hip): where the steps, K and the
rows and columns of dst end, every compiled-in epilogue; and the 256 x 128 tiles of the 16-bit types at the sizes that are now
the small ones' by themselves.  Exact data (any order of the sum gives the same bits) against the oracle, bit for bit."""
import numpy as np
import pytest

from onednn_amd import cabi, configs
from onednn_amd import dtypes as dtp
from onednn_amd.problem import PostOp, decode, run_gpu
from tests.helpers import assert_bit_exact
from tests.test_line_loops import BYTES, FAMILY, RELU, SWITCH, check, problem

pytestmark = pytest.mark.gpu


# a wavefront's steps: none, one, its two in flight, more; K that ends inside a step
@pytest.mark.parametrize("kbytes", [64, 112, 128, 144, 384, 512, 528, 1024, 1152, 1648])
@pytest.mark.parametrize("dt,ddt", [("bf16", "bf16"), ("f16", "f16"), ("bf16", "f16"), ("f16", "f32"), ("f8_e4m3", "bf16"), ("f8_e4m3", "f32"), ("f8_e4m3", "f16")])
def test_where_the_steps_end(gpu, oracle, kbytes, dt, ddt):
    for M, N, batch in ((1, 8, 1), (35, 72, 2), (64, 100 if ddt == "f32" else 104, 1)):
        check(oracle, problem(M, N, kbytes // BYTES[dt], dt, ddt, bias=True, batch=batch), dt, "small", chain=True)


@pytest.mark.parametrize("N", [33, 34, 35, 36, 47])
@pytest.mark.parametrize("dt,ddt,kw", [
    ("bf16", "bf16", dict(bias=True)), ("f16", "f16", dict(post=[RELU])), ("bf16", "f32", {}),
    ("f8_e4m3", "bf16", dict(row_scales=True, post=[RELU])), ("f8_e4m3", "f32", dict(bias=True))])
def test_rows_of_dst_that_end_inside_a_piece(gpu, oracle, dt, ddt, kw, N):
    check(oracle, problem(17, N, 256 // BYTES[dt], dt, ddt, batch=2, pitch=48, **kw), dt, "small", chain=True)


@pytest.mark.parametrize("act", [None, "gelu_tanh", "swish"])
@pytest.mark.parametrize("alg", ["add", "mul"])
@pytest.mark.parametrize("dt", ["bf16", "f8_e4m3"])
def test_a_second_tensor(gpu, oracle, act, alg, dt):
    """with an activation within its few ulp of the oracle, rounded to bf16: two units of bf16"""
    M, N, K = 50, 72, 192
    other = dtp.f32_to_bf16(np.random.default_rng(5).integers(-4, 5, size=2 * M * N).astype(np.float32)).reshape(2, M, N)
    post = [PostOp(cabi.PO_ELTWISE, alg=cabi.ELTWISE[act], alpha=1.0)] if act else []
    post.append(PostOp(cabi.PO_BINARY, alg=cabi.BINARY[alg], dt=cabi.DT_BF16, stride=(M * N, N, 1), data=other))
    p = problem(M, N, K, dt, "bf16", bias=True, post=post, batch=2)
    if dt == "f8_e4m3":
        p.quant["src_scale"].data[:] /= 64
    with cabi.tuning("MI355_EPILOGUE", "chain"):
        got, name = run_gpu(p)  # (small by itself)
    assert name.startswith(FAMILY[dt])
    want = oracle.run_oracle(p)
    if not act:
        assert_bit_exact(p, got, want, name)
        return
    g, w = (dtp.bf16_to_f32(np.asarray(x).view(np.uint16).reshape(-1)) for x in (got, want))
    assert np.all(np.abs(g - w) <= 2.0 ** -7 * np.abs(w) + 2.0 ** -20)


@pytest.mark.parametrize("fmt,K", [("mxf8", 64), ("mxf8", 96), ("mxf8", 128), ("mxf8", 544), ("mxf8", 1184), ("mxf4", 128), ("mxf4", 160),
                                   ("mxf4", 256), ("mxf4", 1056), ("mxf4", 2336)])
@pytest.mark.parametrize("ddt", ["f32", "bf16", "f16"])
def test_block_scales(gpu, oracle, fmt, K, ddt):
    """a scale of its own for every block, read where it lies; batches of them (MXFP8)"""
    from tests.test_mxf8_gemm import problem as mx_problem
    from tests.test_split_k import mx
    for p in ([mx(35, 72, K, fmt, ddt)] + ([mx_problem(35, 72, K, ddt=ddt, seed=K, batch=2, bias=True)] if fmt == "mxf8" and K < 256 else [])):
        with cabi.tuning("MI355_F8_TILES", "small"), cabi.tuning("MI355_EPILOGUE", "chain"):
            got, name = run_gpu(p)
        assert_bit_exact(p, got, oracle.run_oracle(p), name)


# more than 256 tiles: rows and columns that end inside a tile, steps that K does not fill, up to two rounds of the three in flight
@pytest.mark.parametrize("K", [64, 96, 128, 384, 416, 544, 800, 1184])
@pytest.mark.parametrize("ddt,M,N,batch", [("f32", 520, 532, 1), ("bf16", 520, 536, 1), ("f32", 300, 532, 2), ("bf16", 289, 536, 2)])
def test_mxfp8_in_the_large_tiles_order(gpu, K, ddt, M, N, batch):
    """random data, the bits of the 256 x 128 tiles; the chain of either or an error"""
    from tests.test_mxf8_gemm import problem as mx_problem
    p = mx_problem(M, N, K, ddt=ddt, exact=False, seed=K, bias=True, batch=batch)
    out = []
    with cabi.tuning("MI355_EPILOGUE", "chain"):
        for tiles in ("small", "narrow"):
            with cabi.tuning("MI355_F8_TILES", tiles):
                out.append(np.asarray(run_gpu(p)[0]))
    bits = np.uint32 if ddt == "f32" else np.uint16
    assert np.isfinite(decode(p.dst_dt, out[0], out[0].size)).all() and len(np.unique(out[0].view(bits))) > 1000
    assert np.array_equal(*(o.view(bits) for o in out))


@pytest.mark.parametrize("K", [96, 384, 544, 1184])
@pytest.mark.parametrize("ddt", ["f32", "bf16", "f16"])
def test_mxfp8_of_more_than_256_tiles(gpu, oracle, K, ddt):
    """exact data, a scale of its own for every block"""
    from tests.test_split_k import mx
    p = mx(520, 536, K, "mxf8", ddt)
    with cabi.tuning("MI355_F8_TILES", "small"), cabi.tuning("MI355_EPILOGUE", "chain"):
        got, name = run_gpu(p)
    assert_bit_exact(p, got, oracle.run_oracle(p), name)


# infinities and NaN in the chunks that lanes beyond K load a second time
@pytest.mark.parametrize("K", [8, 40, 72, 200])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_nan_at_the_end_of_k(gpu, oracle, K, dt):
    p = problem(40, 72, K, dt, "f32", bias=True)
    inf, nan = (0x7F80, 0x7FC0) if dt == "bf16" else (0x7C00, 0x7E00)
    for name, rows in (("src", 40), ("wei", 72)):
        wide = np.full((rows, K + 24), nan, np.uint16)
        wide[:, :K] = np.asarray(getattr(p, name)).reshape(rows, K)
        wide[rows // 3, K - 1], wide[rows // 2, K - 5] = inf, nan
        setattr(p, name, wide.reshape(-1))
    p.src_stride, p.wei_stride = (0, K + 24, 1), (0, 1, K + 24)
    with cabi.tuning("MI355_H16_TILES", "small"):
        got, _ = run_gpu(p)
    g, w = decode(p.dst_dt, got, 40 * 72), decode(p.dst_dt, oracle.run_oracle(p), 40 * 72)
    assert np.isnan(w).any() and np.isfinite(w).any()
    assert np.array_equal(g, w, equal_nan=True)


def test_which_problems_take_them():
    """by what the scratch tells: block scales keep room for their packed copy, parts of K are the large tiles'"""
    for dt in ("bf16", "f8_e4m3"):
        small = problem(64, 1024, 2048 // BYTES[dt], dt, "bf16")
        assert cabi.scratch_bytes(small.desc()) == 0, dt
        with cabi.tuning(SWITCH[dt], "narrow"):
            assert cabi.scratch_bytes(small.desc()) > 0
        assert cabi.scratch_bytes(problem(64, 640, 32768 // BYTES[dt], dt, "bf16").desc()) > 0


@pytest.mark.parametrize("kbytes", [64, 112, 128, 144, 192, 256, 272, 384, 448, 496, 512, 640, 656])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_steps_of_the_256_x_128_tiles(gpu, oracle, kbytes, dt):
    check(oracle, problem(300, 328, kbytes // 2, dt, dt, bias=True), dt, "narrow", chain=True)


@pytest.mark.parametrize("K", [128, 160, 288, 544, 1120])
@pytest.mark.parametrize("fmt", ["mxf8", "mxf4"])
def test_steps_of_the_256_x_128_tiles_with_block_scales(gpu, oracle, K, fmt):
    from tests.test_split_k import mx
    p = mx(300, 328, K, fmt, "bf16")
    with cabi.tuning("MI355_F8_TILES", "narrow"):
        got, name = run_gpu(p)
    assert_bit_exact(p, got, oracle.run_oracle(p), name)

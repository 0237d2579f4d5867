"""The K loops of 128-byte steps (onednn_amd/csrc/line_loops.hpp) and the kernels with a compiled-in epilogue on top of
them (chain_gemm.hpp): where the steps end, on both tile geometries, and where the rows of dst do.

Exact data (small integers, power-of-two scales: any order of the sum gives the same bits) against the oracle, bit for
bit.  K in bytes: a lone partial step, one chunk short of a step and one past it, one / two / three / four steps (the
loops load two ahead and are unrolled by two) and a partial step behind each count."""
import numpy as np
import pytest

from onednn_amd import cabi, configs
from onednn_amd import dtypes as dtp
from onednn_amd.problem import MatmulProblem, PostOp, QuantParam, decode, run_gpu, storage_dtype, strides_for
from tests.helpers import assert_bit_exact

pytestmark = pytest.mark.gpu
DT = cabi.DT_NAMES
BYTES = {"bf16": 2, "f16": 2, "s8": 1, "u8": 1, "f8_e4m3": 1}
SWITCH = {"bf16": "MI355_H16_TILES", "f16": "MI355_H16_TILES", "s8": "MI355_I8_TILES", "u8": "MI355_I8_TILES",
          "f8_e4m3": "MI355_F8_TILES"}
FAMILY = {"bf16": "hip:mfma_h16", "f16": "hip:mfma_h16", "s8": "hip:mfma_i8", "u8": "hip:mfma_i8", "f8_e4m3": "hip:mfma_f8"}


def encode(v, dt):
    v = np.asarray(v, np.float32)
    if dt == "bf16":
        return dtp.f32_to_bf16(v.reshape(-1)).reshape(v.shape)
    if dt == "f16":
        return v.astype(np.float16).view(np.uint16)
    if dt == "f8_e4m3":
        return dtp.f32_to_e4m3(v.reshape(-1)).reshape(v.shape)
    return v.astype(np.int8 if dt == "s8" else np.uint8)


def problem(M, N, K, dt, ddt, *, bias=False, post=(), batch=1, pitch=0, dst_scale=None, src_zp=None, row_scales=False):
    r = np.random.default_rng(M + N + K)
    lo, hi = (0, 7) if dt == "u8" else (-3, 4)
    src = encode(r.integers(lo, hi, size=(batch, M, K)), dt)
    wdt = "s8" if dt == "u8" else dt
    wei = encode(r.integers(-2, 3, size=(batch, N, K)), wdt)
    quant = {}
    if dt in ("s8", "u8", "f8_e4m3"):
        quant["src_scale"] = QuantParam(cabi.DT_F32, 0, np.array([0.5], np.float32))
        quant["wei_scale"] = QuantParam(cabi.DT_F32, configs.MASK_COL, r.choice([0.25, 0.5, 1.0], size=N).astype(np.float32))
    if row_scales:
        quant["src_scale"] = QuantParam(cabi.DT_F32, 2, r.choice([0.25, 0.5, 1.0], size=M).astype(np.float32))
    if src_zp is not None:
        quant["src_zp"] = QuantParam(cabi.DT_S32, 0, np.array([src_zp], np.int32))
    if dst_scale is not None:
        quant["dst_scale"] = QuantParam(cabi.DT_F32, 0, np.array([dst_scale], np.float32))
    b = (r.integers(-8, 9, size=N) / 4).astype(np.float32) if bias else None
    kw = {}
    if pitch:  # what lies between the rows stays as it is
        kw = dict(dst_stride=(M * pitch, pitch, 1),
                  dst_init=np.full((batch * M - 1) * pitch + N, 0x5A, storage_dtype(DT[ddt])))
    return MatmulProblem(M=M, N=N, K=K, batch=batch, src_dt=DT[dt], wei_dt=DT[wdt], dst_dt=DT[ddt], src=src, wei=wei,
                         wei_stride=strides_for("ba", batch, K, N), bias_dt=cabi.DT_F32 if bias else cabi.DT_UNDEF, bias=b,
                         quant=quant, post_ops=list(post), name=f"lines-{dt}-{ddt}-{M}x{N}x{K}", **kw)


def check(oracle, p, dt, tiles=None, chain=False):
    """chain: a compiled-in epilogue's kernel or an error"""
    with cabi.tuning(SWITCH[dt], tiles), cabi.tuning("MI355_EPILOGUE", "chain" if chain else None):
        got, name = run_gpu(p)
    assert name.startswith(FAMILY[dt]), name
    assert_bit_exact(p, got, oracle.run_oracle(p), f"{name} {tiles}")


# 300 x 328 runs on 256 x 128 tiles by itself (int8: when told to), on 256 x 256 ones when told to
@pytest.mark.parametrize("kbytes", [64, 112, 128, 144, 192, 256, 272, 384, 448, 496, 512, 640, 656])
@pytest.mark.parametrize("dt,ddt", [("bf16", "bf16"), ("f16", "f16"), ("s8", "f32"), ("u8", "bf16"), ("f8_e4m3", "bf16")])
@pytest.mark.parametrize("tiles", ["wide", "narrow"])
def test_where_the_steps_end(gpu, oracle, kbytes, dt, ddt, tiles):
    p = problem(300, 328, kbytes // BYTES[dt], dt, ddt, bias=True, src_zp=3 if dt == "u8" else None)
    check(oracle, p, dt, "wide" if tiles == "wide" else None if BYTES[dt] == 2 else "narrow")


RELU = PostOp(cabi.PO_ELTWISE, alg=cabi.ELTWISE["relu"], alpha=0.0)


# rows of dst that end inside a wavefront's 64 columns, dense ones of whole and of no whole 16-byte pieces (a 16-bit or f32
# dst of the latter is the general epilogue's), M inside a wavefront's 128 rows, every compiled-in dst type, batches
@pytest.mark.parametrize("M,N", [(1, 136), (129, 200), (130, 268), (257, 388)])
@pytest.mark.parametrize("dt,ddt,kw", [
    ("bf16", "bf16", {}), ("bf16", "f32", dict(bias=True)), ("f16", "f16", dict(bias=True, post=[RELU])),
    ("f16", "f32", dict(post=[RELU])), ("f16", "bf16", dict(bias=True)), ("bf16", "f16", dict(post=[RELU])), ("s8", "s8", dict(post=[RELU], dst_scale=3.0)), ("s8", "u8", dict(bias=True, dst_scale=0.7)),
    ("u8", "s8", dict(bias=True, src_zp=5)), ("u8", "f32", dict(src_zp=2, post=[RELU])), ("f8_e4m3", "f32", dict(bias=True)),
    ("f8_e4m3", "bf16", dict(row_scales=True, post=[RELU]))])
def test_where_the_rows_of_dst_end(gpu, oracle, M, N, dt, ddt, kw):
    for tiles in ("wide", "narrow"):
        p = problem(M, N, 256 // BYTES[dt], dt, ddt, batch=2, **kw)
        check(oracle, p, dt, "wide" if tiles == "wide" else None if BYTES[dt] == 2 else "narrow")


# ... and that end inside a 16-byte piece of a pitch of whole ones (8-bit: of dwords, too): every length of the last piece,
# on each tile's chain
@pytest.mark.parametrize("dt,ddt,kw", [
    ("bf16", "bf16", dict(bias=True)), ("bf16", "f16", {}), ("f16", "f16", dict(post=[RELU])), ("f16", "f32", {}),
    ("s8", "s8", dict(post=[RELU], dst_scale=3.0)), ("s8", "f32", dict(bias=True)), ("u8", "u8", dict(bias=True, src_zp=5)),
    ("u8", "bf16", dict(src_zp=2)), ("f8_e4m3", "bf16", dict(row_scales=True)), ("f8_e4m3", "f32", {})])
@pytest.mark.parametrize("N", [257, 258, 259, 260, 261, 262, 263, 195])
def test_rows_of_dst_that_end_inside_a_piece(gpu, oracle, dt, ddt, kw, N):
    piece = {"f32": 4, "s8": 16, "u8": 16}.get(ddt, 8)
    for tiles in ("wide", "narrow", "small")[:3 if BYTES[dt] == 1 and dt != "f8_e4m3" else 2]:
        for pitch in {-(-N // piece) * piece, -(-N // 4) * 4 if piece == 16 else -(-N // piece) * piece + piece}:
            p = problem(131, N, 256 // BYTES[dt], dt, ddt, batch=2, pitch=pitch, **kw)
            check(oracle, p, dt, None if BYTES[dt] == 2 and tiles == "narrow" else tiles, chain=True)


@pytest.mark.parametrize("act", [None, "gelu_tanh", "swish"])
@pytest.mark.parametrize("alg", ["add", "mul"])
@pytest.mark.parametrize("dt", ["bf16", "f8_e4m3", "f8_e4m3 rows", "mxfp8"])
@pytest.mark.parametrize("tiles", ["wide", None])
@pytest.mark.parametrize("M,N,batch", [(150, 200, 1), (300, 328, 2)])
def test_a_staged_tensor_at_ragged_edges(gpu, oracle, act, alg, dt, tiles, M, N, batch):
    """Both tiles (the narrow one by itself at these sizes); the last wavefront's columns end after one chunk of eight, rows
    inside a row block; scales per row, whose loads the waits for the tensor's have to reckon with; a tensor of two batches.
    Without an activation the sums are exact; with one the result is within the activation's few ulp of the oracle, rounded to
    bf16: two units of bf16."""
    K, rows = 128, dt.endswith("rows")
    dt = dt.split()[0]
    r = np.random.default_rng(5)
    other = dtp.f32_to_bf16(r.integers(-4, 5, size=batch * M * N).astype(np.float32)).reshape(batch, M, N)
    post = [PostOp(cabi.PO_ELTWISE, alg=cabi.ELTWISE[act], alpha=1.0)] if act else []
    post.append(PostOp(cabi.PO_BINARY, alg=cabi.BINARY[alg], dt=cabi.DT_BF16, stride=(M * N, N, 1), data=other))
    if dt == "mxfp8":
        from tests.test_mxf8_gemm import problem as mx_problem
        p = mx_problem(M, N, K, ddt="bf16", bias=True, post_ops=post, batch=batch)
        p.quant["src_scale"].data[:] = 127 - 6
        p.quant["wei_scale"].data[:] = 127
    else:
        p = problem(M, N, K, dt, "bf16", bias=True, post=post, batch=batch, row_scales=rows)
    if dt == "f8_e4m3":
        p.quant["src_scale"].data[:] /= 64
    with cabi.tuning(SWITCH.get(dt, "MI355_F8_TILES"), tiles), cabi.tuning("MI355_EPILOGUE", "chain"):
        got, name = run_gpu(p)
    assert name.startswith(FAMILY.get(dt, "hip:mfma_f8")), name
    want = oracle.run_oracle(p)
    if not act:
        assert_bit_exact(p, got, want, name)
        return
    g, w = (dtp.bf16_to_f32(np.asarray(x).view(np.uint16).reshape(-1)) for x in (got, want))
    assert np.all(np.abs(g - w) <= 2.0 ** -7 * np.abs(w) + 2.0 ** -20)


def across_problem(M, N, K, dt, ddt, src_across, *, batch=1, wei_pad=0, src_pad=0, bias=True, pads=(77, 99)):
    """weights row-major ([K][N], a pitch of N + wei_pad), src row-major or ([K][M], a pitch of M + src_pad)"""
    r = np.random.default_rng(M * 3 + N * 5 + K)
    sv = r.integers(-3, 4, size=(batch, M, K)).astype(np.float32)
    wv = np.full((batch, K, N + wei_pad), pads[1], np.float32)
    wv[:, :, :N] = r.integers(-2, 3, size=(batch, K, N))
    ss = (M * K, K, 1)
    if src_across:
        full = np.full((batch, K, M + src_pad), pads[0], np.float32)
        full[:, :, :M] = sv.transpose(0, 2, 1)
        sv, ss = full, (K * (M + src_pad), 1, M + src_pad)
    b = (r.integers(-8, 9, size=N) / 4).astype(np.float32) if bias else None
    return MatmulProblem(M=M, N=N, K=K, batch=batch, src_dt=DT[dt], wei_dt=DT[dt], dst_dt=DT[ddt], src=encode(sv, dt),
                         wei=encode(wv, dt), src_stride=ss, wei_stride=(K * (N + wei_pad), N + wei_pad, 1),
                         bias_dt=cabi.DT_F32 if bias else cabi.DT_UNDEF, bias=b, name=f"across-{dt}-{ddt}-{M}x{N}x{K}")


# operands that are contiguous across K: every place where a step, a half of its 64 k or a 32-byte unit of a line can end
@pytest.mark.parametrize("K", [8, 24, 32, 56, 64, 72, 96, 104, 128, 160, 192, 200, 320])
@pytest.mark.parametrize("dt,ddt", [("bf16", "bf16"), ("f16", "f16"), ("bf16", "f32")])
@pytest.mark.parametrize("tiles", [None, "wide"])
@pytest.mark.parametrize("src_across", [False, True])
def test_operands_contiguous_across_k(gpu, oracle, K, dt, ddt, tiles, src_across):
    check(oracle, across_problem(304, 328, K, dt, ddt, src_across), dt, tiles)


# both across K: any K; row pitches beyond the rows; ragged edges in steps of eight; what is not whole 16-byte pieces is
# copied as before
@pytest.mark.parametrize("M,N,K,pads", [(264, 264, 1, (0, 0)), (512, 136, 63, (8, 16)), (520, 392, 65, (0, 8)), (8, 264, 127, (16, 0)),
                                        (296, 520, 193, (0, 0)), (300, 328, 70, (0, 0)), (304, 330, 70, (0, 0)), (304, 328, 70, (3, 5))])
def test_both_across_k_ragged(gpu, oracle, M, N, K, pads):
    for tiles in (None, "wide"):
        check(oracle, across_problem(M, N, K, "bf16", "bf16", True, batch=2, src_pad=pads[0], wei_pad=pads[1]), "bf16", tiles)


# block scales on both geometries (their loads ride along with the steps'): a scale of its own for every block
@pytest.mark.parametrize("K", [64, 96, 128, 160, 256, 288, 384, 512, 672])
@pytest.mark.parametrize("tiles", [None, "wide"])
def test_mxfp8_steps(gpu, oracle, K, tiles):
    from tests.test_mxf8_gemm import problem as mx_problem
    for M, N, ddt in ((300, 328, "f32"), (129, 200, "bf16")):
        p = mx_problem(M, N, K, ddt=ddt, seed=K)
        with cabi.tuning("MI355_F8_TILES", tiles):
            got, name = run_gpu(p)
        assert name.startswith("hip:mfma_f8"), name
        assert_bit_exact(p, got, oracle.run_oracle(p), f"{name} {tiles}")


@pytest.mark.parametrize("K", [128, 160, 256, 288, 512, 544, 768, 1024, 1120])
@pytest.mark.parametrize("tiles", [None, "wide"])
@pytest.mark.parametrize("ddt", ["f32", "f16"])
def test_mxfp4_steps(gpu, oracle, K, tiles, ddt):
    """one block of some rows and columns scaled up: every block of every step has to meet its own scale; f16: the general
    epilogue's kernels"""
    p = configs.config5(M=300, N=328, K=K)
    p.dst_dt = DT[ddt]
    ss, ws = p.quant["src_scale"].data, p.quant["wei_scale"].data
    ss[:] = 127
    ws[:] = 126
    kb = K // 32
    s2, w2 = ss.reshape(300, kb), ws.reshape(kb, 328)
    for i in range(kb):
        s2[(37 * i) % 300, i] = 129
        w2[i, (53 * i) % 328] = 128
    with cabi.tuning("MI355_F8_TILES", tiles):
        got, name = run_gpu(p)
    assert name.startswith("hip:mfma_mxf4"), name
    assert_bit_exact(p, got, oracle.run_oracle(p), f"{name} {tiles}")


def check_with_nan(oracle, p, tiles):
    """NaN and infinities where the oracle has them, the rest bit for bit"""
    switch = "MI355_H16_TILES" if p.src_dt in (cabi.DT_BF16, cabi.DT_F16) else "MI355_F8_TILES"
    with cabi.tuning(switch, tiles):
        got, name = run_gpu(p)
    n = p.batch * p.M * p.N
    g, w = decode(p.dst_dt, got, n), decode(p.dst_dt, oracle.run_oracle(p), n)
    assert np.isnan(w).any() and np.isfinite(w).any()
    assert np.array_equal(g, w, equal_nan=True), (p.name, name, tiles)


# What lies behind K, or is loaded twice by the lanes of a partial last step, adds nothing, whatever it is: NaN behind the
# rows of both operands, and infinities and NaN in the last chunk of some rows and columns.
@pytest.mark.parametrize("tiles", [None, "wide"])
@pytest.mark.parametrize("K", [8, 40, 72, 104, 136, 200, 328])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_nan_at_the_end_of_k(gpu, oracle, tiles, K, dt):
    p = problem(300, 328, K, dt, "f32", bias=True)
    inf, nan = (0x7F80, 0x7FC0) if dt == "bf16" else (0x7C00, 0x7E00)
    for name, rows in (("src", 300), ("wei", 328)):
        wide = np.full((rows, K + 24), nan, np.uint16)
        wide[:, :K] = np.asarray(getattr(p, name)).reshape(rows, K)
        wide[rows // 3, K - 1], wide[rows // 2, K - 5] = inf, nan
        setattr(p, name, wide.reshape(-1))
    p.src_stride, p.wei_stride = (0, K + 24, 1), (0, 1, K + 24)
    check_with_nan(oracle, p, tiles)


@pytest.mark.parametrize("tiles", [None, "wide"])
@pytest.mark.parametrize("K", [8, 24, 40, 72, 136, 200])
@pytest.mark.parametrize("src_across", [False, True])
def test_nan_across_k(gpu, oracle, tiles, K, src_across):
    p = across_problem(304, 328, K, "bf16", "f32", src_across, wei_pad=8, src_pad=16, pads=(np.nan, np.nan))
    wei = p.wei.reshape(K, 336)
    wei[K - 1, 17], wei[K - 3, 200] = 0x7F80, 0x7FC0
    src = p.src.reshape(K, 320) if src_across else p.src.reshape(304, K).T
    src[K - 1, 40], src[K - 2, 250] = 0x7F80, 0x7FC0
    check_with_nan(oracle, p, tiles)


@pytest.mark.parametrize("tiles", [None, "wide"])
@pytest.mark.parametrize("K", [96, 160, 224, 288])
def test_nan_at_the_end_of_block_scaled_k(gpu, oracle, tiles, K):
    from tests.test_mxf8_gemm import problem as mx_problem
    p = mx_problem(300, 328, K, seed=K)
    p.src.reshape(300, K)[70, K - 9] = p.wei.reshape(328, K)[201, K - 2] = 0x7F
    p.quant["src_scale"].data.reshape(300, K // 32)[155, K // 32 - 1] = 0xFF
    check_with_nan(oracle, p, tiles)

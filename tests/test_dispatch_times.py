"""Calls that a dispatch rule sends to one of several kernels take no longer than the kernel the rule should have found.
Both sides run on one GPU in turn, as graphs of many launches; the least of several turns counts."""
import ctypes as C

import numpy as np
import pytest

from onednn_amd import cabi, configs
from onednn_amd import dtypes as dtp
from onednn_amd.problem import GpuRun, MatmulProblem, PostOp, QuantParam, strides_for
from onednn_amd.reorder import GpuReorder, ReorderProblem
from tests.test_gpu_i8_small import int8_problem

pytestmark = pytest.mark.gpu


def in_turn(*launches, n=20, turns=12):
    """The least microseconds a launch of each; a launch takes the stream's handle."""
    lib, s = cabi.load_kernels(), cabi.Stream()
    ev = [C.c_void_p(), C.c_void_p()]
    for e in ev:
        cabi.check(lib.mi355_event_create(C.byref(e)))
    graphs, best = [], [np.inf] * len(launches)
    for launch in launches:
        launch(s.ptr)
        s.sync()
        with cabi.Graph(s) as g:
            for _ in range(n):
                launch(s.ptr)
        g.launch()
        s.sync()
        graphs.append(g)
    for _ in range(turns):
        for i, g in enumerate(graphs):
            cabi.check(lib.mi355_event_record(ev[0], s.ptr))
            g.launch()
            cabi.check(lib.mi355_event_record(ev[1], s.ptr))
            s.sync()
            ms = C.c_float()
            cabi.check(lib.mi355_event_elapsed_ms(C.byref(ms), ev[0], ev[1]))
            best[i] = min(best[i], ms.value * 1e3 / n)
    for g in graphs:
        g.destroy()
    for e in ev:
        lib.mi355_event_destroy(e)
    s.destroy()
    return best


def launches(p, switch=None, value=None):
    """A launch of p for in_turn, a tuning switch set around it (and around the scratch query)."""
    if switch is None:
        g = GpuRun(p)
    else:
        with cabi.tuning(switch, value):
            g = GpuRun(p)

    def go(s):
        g.stream = s
        if switch is None:
            g.launch()
            return
        with cabi.tuning(switch, value):
            g.launch()
    return go


@pytest.mark.parametrize("rows,cols", [(2, 512), (8, 14336), (16, 50000), (32, 200000)])
def test_column_sums_of_few_rows(gpu, rows, cols):
    """x off a 16-byte boundary is the plain kernel's, a load per row and column; aligned x is no slower."""
    x, out = cabi.DeviceBuffer(4 * (rows * cols + 1)), cabi.DeviceBuffer(4 * cols)
    lib = cabi.load_kernels()

    def launch(at):
        return lambda s: cabi.check(lib.mi355_colsum_launch(x.ptr + at, cabi.DT_F32, rows, cols, cols, out.ptr, cabi.DT_F32, s))

    aligned, plain = in_turn(launch(0), launch(4))
    assert aligned <= 1.2 * plain, (aligned, plain)


@pytest.mark.parametrize("M,N,K", [(32, 25600, 1024), (32, 20480, 256), (256, 3712, 1024), (22, 28672, 1024)])
def test_int8_layers_with_a_short_m(gpu, M, N, K):
    """s8 x s8 -> s8 without zero points on whole columns: the LDS tiles from three small tiles a compute unit on."""
    p = int8_problem(M, N, K, cabi.DT_S8, cabi.DT_S8, cabi.DT_S8, dst_scale=20.0,
                     post_ops=[PostOp(kind=cabi.PO_ELTWISE, alg=cabi.ELTWISE["relu"])])

    chosen, lds = in_turn(*(launches(p, "MI355_I8_TILES", tiles) for tiles in (None, "large")))
    assert chosen <= 1.06 * lds, (chosen, lds)


@pytest.mark.parametrize("src_dt,wei_dt,dims", [(cabi.DT_U8, cabi.DT_S8, (64, 128, 128, 256)), (cabi.DT_S8, cabi.DT_U8, (64, 128, 128, 256)),
                                                (cabi.DT_U8, cabi.DT_S8, (256, 128, 128, 48))])
def test_int8_sums_of_a_batch_are_one_launch(gpu, src_dt, wei_dt, dims):
    """Column or row sums in front of the LDS tiles, against signed operands without: one kernel more of a few us (and the
    general epilogue's terms, for u8 weights), not one of 2 us for every batch."""
    B, M, N, K = dims
    with_sums, plain = in_turn(*(launches(int8_problem(M, N, K, s, w, cabi.DT_F32, batch=B), "MI355_I8_TILES", "large")
                                 for s, w in ((src_dt, wei_dt), (cabi.DT_S8, cabi.DT_S8))))
    assert with_sums <= plain + 20, (with_sums, plain)


# what decides between the small and the LDS tiles: K, whole 64 bytes of it or not, M, sums of their own and the epilogue.  (u8
# weights, a zero point that is not s32 and relu with a slope are the general kernels'.)
@pytest.mark.parametrize("M,N,K", [(256, 4096, 8208), (256, 6144, 1040), (256, 4096, 4112), (256, 5120, 1024), (256, 3840, 16384),
                                   (16, 32768, 2176), (32, 49152, 1040)])
@pytest.mark.parametrize("form", ["s8", "u8 src", "u8 weights", "f16 dst", "slope"])
def test_int8_small_or_lds_tiles(gpu, M, N, K, form):
    kw = {"s8": dict(dst_dt=cabi.DT_S8, dst_scale=20.0), "u8 src": dict(src_dt=cabi.DT_U8), "u8 weights": dict(wei_dt=cabi.DT_U8),
          "f16 dst": dict(dst_dt=cabi.DT_F16), "slope": dict(post_ops=[PostOp(kind=cabi.PO_ELTWISE, alg=cabi.ELTWISE["relu"], alpha=0.1)])}
    p = int8_problem(M, N, K, **{**dict(src_dt=cabi.DT_S8, wei_dt=cabi.DT_S8, dst_dt=cabi.DT_BF16), **kw[form]})
    chosen, small, lds = in_turn(*(launches(p, "MI355_I8_TILES", tiles) for tiles in (None, "small", "large")))
    assert chosen <= 1.12 * min(small, lds), (chosen, small, lds)


@pytest.mark.parametrize("pitch,offset", [(8196, 0), (8192, 4), (8200, 8)])
def test_transposition_out_of_rows_that_are_4_byte_aligned(gpu, pitch, offset):
    """Four elements a load: about half of what rows off a 4-byte boundary, an element a load, take."""
    n = 8192
    raw = np.zeros(offset + n * pitch + 1, np.int8)

    def launch(pitch, offset):
        g = GpuReorder(ReorderProblem(dims=(n, n), src_dt=cabi.DT_S8, dst_dt=cabi.DT_S8, src=raw, src_stride=(pitch, 1),
                                      dst_stride=(1, n), name="transposition"))
        g.args.src += offset
        return g.launch

    by_4, by_1 = in_turn(launch(pitch, offset), launch(n, 1))
    assert by_4 <= 0.75 * by_1, (by_4, by_1)


def float_problem(M, N, K, dt, ddt, **kw):
    r = np.random.default_rng(M + N + K)
    enc = {"bf16": dtp.f32_to_bf16, "f16": lambda v: v.astype(np.float16).view(np.uint16), "f8_e4m3": dtp.f32_to_e4m3}[dt]
    src, wei = (enc(r.standard_normal(n).astype(np.float32)) for n in (M * K, N * K))
    return MatmulProblem(M=M, N=N, K=K, src_dt=cabi.DT_NAMES[dt], wei_dt=cabi.DT_NAMES[dt], dst_dt=cabi.DT_NAMES[ddt], src=src, wei=wei,
                         wei_stride=strides_for("ba", 1, K, N), **kw)


@pytest.mark.parametrize("M,N,K", [(1024, 4096, 512), (4096, 4096, 256), (64, 4096, 1024)])
@pytest.mark.parametrize("dt,ddt", [("f16", "bf16"), ("bf16", "f16")])
def test_a_dst_of_the_other_16_bit_type(gpu, M, N, K, dt, ddt):
    """Against operands of dst's own type, which take the same instructions and the same conversion to dst.  The general
    epilogue costs these sizes 6 us and more of 16 to 22 (1.3 to 1.45 times)."""
    mixed, same = in_turn(*(launches(float_problem(M, N, K, d, ddt)) for d in (dt, ddt)))
    assert mixed <= 1.15 * same, (mixed, same)


@pytest.mark.parametrize("M,N,K", [(1, 512, 64), (64, 4096, 128)])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_a_16_bit_dst_of_a_small_product(gpu, M, N, K, dt):
    """A launch of one round and few steps is its epilogue's instruction fetches: against an f32 dst, which knows no second
    tensor, 1.1 to 1.6 us for the conversion; 2.1 to 2.6 with that tensor's code in the way of a chain that has none."""
    half, f32 = in_turn(*(launches(float_problem(M, N, K, dt, d)) for d in (dt, "f32")))
    assert half <= f32 + 1.9, (half, f32)


@pytest.mark.parametrize("M,N,K", [(1024, 4096, 512), (64, 4096, 1024), (4096, 4096, 256)])
@pytest.mark.parametrize("act,residual", [(True, False), (False, True), (True, True)])
def test_mxfp8_layers_with_an_activation_or_a_residual(gpu, M, N, K, act, residual):
    """Against the same sums with a bias alone.  The two together are a tensor more to read (at 5 TB/s), behind a latency of
    its own, and about 20 instructions an element more (5.5 us in all); through the general epilogue they cost 13 to 20."""
    def scaled(**kw):
        p = float_problem(M, N, K, "f8_e4m3", "bf16", bias_dt=cabi.DT_BF16, bias=np.zeros(N, np.uint16), **kw)
        for name, rows, groups in (("src_scale", M, (1, 32)), ("wei_scale", N, (32, 1))):
            p.quant[name] = QuantParam(cabi.DT_E8M0, 6, np.full(rows * K // 32, 127, np.uint8), groups)
        return launches(p)

    post = [PostOp(cabi.PO_ELTWISE, alg=cabi.ELTWISE["gelu_tanh"])] if act else []
    if residual:
        post.append(PostOp(cabi.PO_BINARY, alg=cabi.BINARY["add"], dt=cabi.DT_BF16, stride=(0, N, 1), data=np.zeros(M * N, np.uint16)))
    with_post, plain = in_turn(scaled(post_ops=post), scaled())
    assert with_post <= plain + (2 * M * N / 5e6 if residual else 0) + 5.5, (with_post, plain)


@pytest.mark.parametrize("M,N,K", [(64, 4096, 1024), (512, 4096, 1024), (1024, 4096, 512), (64, 4096, 4096)])
def test_mxfp4_through_the_general_epilogue(gpu, M, N, K):
    """A dst type that no chain stores (f16) against bf16, which one does: the general epilogue's 4 to 6 us, and not
    those of a kernel that keeps its addresses in scratch memory or of tiles that leave half of the device idle."""
    def launch(ddt):
        p = configs.config5(M=M, N=N, K=K, wtag="ba")
        p.dst_dt = cabi.DT_NAMES[ddt]
        return launches(p)

    general, chain = in_turn(launch("f16"), launch("bf16"))
    assert general <= chain + 7.5, (general, chain)


@pytest.mark.parametrize("M,N,K", [(4096, 5120, 256), (3072, 8192, 1024), (4096, 4352, 2048), (2560, 8192, 4096)])
@pytest.mark.parametrize("dt,ddt", [("bf16", "bf16"), ("bf16", "f8_e4m3"), ("f8_e4m3", "bf16"), ("f8_e4m3", "f16")])
def test_three_rounds_of_narrow_tiles_or_two_of_wide(gpu, M, N, K, dt, ddt):
    """257 to 384 large tiles: the wide tiles are never better by more than 7 %, where three narrow rounds cost a short K or
    the general epilogue a quarter and more."""
    p = float_problem(M, N, K, dt, ddt)
    chosen, wide = in_turn(*(launches(p, "MI355_H16_TILES" if dt == "bf16" else "MI355_F8_TILES", t) for t in (None, "wide")), n=10)
    assert chosen <= 1.07 * wide, (chosen, wide)


def test_int8_sums_are_no_reason_for_small_tiles_without_them(gpu):
    """A K that ends inside 64 bytes, signed operands: nothing to add up, so no scratch, and the LDS tiles all the same."""
    p = int8_problem(2048, 4096, 2064, cabi.DT_S8, cabi.DT_S8, cabi.DT_S8, dst_scale=20.0)
    assert cabi.scratch_bytes(p.desc()) == 0
    chosen, small = in_turn(*(launches(p, "MI355_I8_TILES", t) for t in (None, "small")))
    assert chosen <= 0.6 * small, (chosen, small)

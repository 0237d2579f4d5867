"""Operands off 16-byte boundaries and launches without scratch, where a K that ends inside 64 bytes has always taken them: the
K loops of 128-byte steps load 16 bytes straight to LDS, so such calls run on a copy (16-bit types) or on the small tiles
(int8).  Bit for bit against the oracle."""
import ctypes as C

import numpy as np
import pytest

from onednn_amd import cabi
from onednn_amd.problem import GpuRun
from tests.helpers import assert_bit_exact
from tests.test_gpu_i8_small import int8_problem
from tests.test_line_loops import problem

pytestmark = pytest.mark.gpu


def move(run, name, offset):
    """The operand again, `offset` bytes behind an aligned address."""
    raw = np.ascontiguousarray(getattr(run.prob, name)).view(np.uint8).reshape(-1)
    buf = cabi.DeviceBuffer.from_numpy(np.concatenate([np.full(offset, 0x7F, np.uint8), raw]))
    run.bufs[name + "_moved"] = buf
    setattr(run.args, name, buf.ptr + offset)


def check(oracle, p, family, src=0, wei=0):
    run = GpuRun(p)
    try:
        assert cabi.impl_name(run.impl).startswith(family)
        if src:
            move(run, "src", src)
        if wei:
            move(run, "wei", wei)
        run.launch()
        assert_bit_exact(p, run.result(), oracle.run_oracle(p), f"{p.name} +{src} +{wei}")
    finally:
        run.free()


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("K", [40, 72, 136, 200])
@pytest.mark.parametrize("src,wei", [(2, 0), (0, 6), (8, 14)])
def test_16_bit_operands(gpu, oracle, dt, K, src, wei):
    check(oracle, problem(300, 328, K, dt, dt, bias=True, batch=2), "hip:mfma_h16", src, wei)


@pytest.mark.parametrize("dt,ddt", [("s8", "s8"), ("u8", "f32")])
@pytest.mark.parametrize("src,wei", [(1, 0), (0, 4), (3, 7)])
def test_int8_operands(gpu, oracle, dt, ddt, src, wei):
    """4096 small tiles, more than the line between the tiles"""
    check(oracle, problem(512, 8192, 80, dt, ddt, src_zp=3 if dt == "u8" else None), "hip:mfma_i8", src, wei)


@pytest.mark.parametrize("dt,ddt", [("s8", "s8"), ("u8", "f32")])
@pytest.mark.parametrize("src,wei", [(1, 0), (0, 4), (8, 7)])
def test_int8_operands_where_k_would_be_split(gpu, oracle, dt, ddt, src, wei):
    """1024 small tiles by themselves; K in parts on the LDS tiles only where both operands lie on 16-byte boundaries"""
    p = problem(1024, 1024, 4096, dt, ddt, src_zp=3 if dt == "u8" else None)
    assert cabi.scratch_bytes(p.desc()) > 1 << 20
    check(oracle, p, "hip:mfma_i8", src, wei)


@pytest.mark.parametrize("wei_zp", [False, True])
def test_int8_sums_without_scratch(gpu, oracle, wei_zp):
    p = int8_problem(512, 8192, 80, cabi.DT_U8, cabi.DT_S8, cabi.DT_F32, src_zp=5, wei_zp=wei_zp)
    run = GpuRun(p)
    try:
        assert run.scratch is not None
        run.scratch.free()
        run.scratch = None
        run.launch()
        assert_bit_exact(p, run.result(), oracle.run_oracle(p), "no scratch")
    finally:
        run.free()


def test_int8_sums_beyond_the_static_scratch(gpu, oracle):
    """4 bytes of sums a column: more than mi355_matmul_launch_noalloc holds.  (Of up to 64 rows the small tiles have any
    number.)"""
    N = cabi.NOALLOC_SCRATCH_BYTES // 4 + 64
    p = int8_problem(65, N, 16, cabi.DT_U8, cabi.DT_S8, cabi.DT_S8, src_zp=5, dst_scale=4.0)
    assert cabi.scratch_bytes(p.desc()) > cabi.NOALLOC_SCRATCH_BYTES
    run = GpuRun(p)
    try:
        cabi.check(run.lib.mi355_matmul_launch_noalloc(C.byref(run.desc), C.byref(run.args), None))
        assert_bit_exact(p, run.result(), oracle.run_oracle(p), "noalloc")
    finally:
        run.free()

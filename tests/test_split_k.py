"""Products of few tiles and a long K, whose K is split over workgroups (onednn_amd/csrc/chain_gemm.hpp): where the parts
end, every compiled-in epilogue of the kernel that adds them, and the launches that have no scratch for parts.

Exact data (any order of the sum gives the same bits) against the oracle, bit for bit.
"""
import os
import re
import subprocess

import numpy as np
import pytest

from onednn_amd import cabi, configs
from onednn_amd import dtypes as dtp
from onednn_amd.problem import GpuRun, PostOp, run_gpu
from tests.helpers import assert_bit_exact
from tests.test_line_loops import BYTES, FAMILY, RELU, across_problem, problem

PART = 256 * 128 * 4  # bytes of a part of a tile


def parts_of(p, tile=PART):
    """bytes of scratch in whole parts (what else a problem wants there is smaller, or a copy)"""
    return cabi.scratch_bytes(p.desc()) // tile


def mx(M, N, K, fmt, ddt):
    from tests.test_mxf8_gemm import problem as mx_problem
    p = configs.config5(M=M, N=N, K=K) if fmt == "mxf4" else mx_problem(M, N, K, ddt=ddt)
    p.dst_dt = cabi.DT_NAMES[ddt]
    kb = K // 32
    ss, ws = p.quant["src_scale"].data, p.quant["wei_scale"].data
    ss[...] = 127
    ws[...] = 126
    for i in range(kb):  # every block of every part meets its own scale
        ss.reshape(M, kb)[(37 * i) % M, i] = 129
        ws.reshape(kb, N)[i, (53 * i) % N] = 128
    return p


@pytest.fixture(autouse=True)
def large_tiles():
    """no 32 x 32 tiles, which take many of these sizes by themselves; int8 has its own line"""
    with cabi.tuning("MI355_F8_TILES", "narrow"), cabi.tuning("MI355_H16_TILES", "narrow"):
        yield


def test_which_problems_are_split():
    # few tiles and many steps; not where steps are few, tiles many, or the epilogue is not a chain
    assert parts_of(problem(100, 200, 4096, "bf16", "bf16")) >= 2 * 2
    assert cabi.scratch_bytes(problem(100, 200, 256, "bf16", "bf16").desc()) == 0
    assert cabi.scratch_bytes(problem(2300, 2000, 2048, "f8_e4m3", "bf16").desc()) == 0
    p = problem(100, 200, 8192, "f8_e4m3", "bf16", post=[PostOp(cabi.PO_ELTWISE, alg=cabi.ELTWISE["tanh"])])
    assert cabi.scratch_bytes(p.desc()) == 0
    # the parts of one problem are never more than the device's workgroups
    for M, N, K in [(1, 128, 1 << 16), (300, 328, 32768), (256, 4096, 8192), (2048, 2048, 16384)]:
        n = parts_of(problem(M, N, K, "f8_e4m3", "bf16"))
        assert 2 <= n <= 256


@pytest.mark.parametrize("K,parts", [(1 << 24, True), ((1 << 24) + 64, False)])
def test_int8_rows_beyond_the_offsets_of_the_lds_tiles(K, parts):
    """their offsets are 32-bit: longer rows stay on the small tiles, which need no scratch (u8: nor column sums)"""
    d = problem(8, 64, 128, "u8", "f32", src_zp=3).desc()
    d.K = K
    for s in (d.src_stride, d.wei_stride):
        for i in range(2 if s is d.src_stride else 3):
            if s[i] == 128:
                s[i] = K
    assert list(d.wei_stride)[1:] == [1, K] and list(d.src_stride)[1:] == [K, 1]
    assert (cabi.scratch_bytes(d) > 0) == parts


@pytest.mark.parametrize("dt,shape", [("f8_e4m3", (8, 64, 1 << 30)), ("mxf8", (8, 16384, 1 << 23)), ("mxf4", (8, 16384, 1 << 23))])
def test_what_the_offsets_of_the_small_tiles_do_not_reach(dt, shape):
    """by the scratch when they are told to run: K that is split instead is the large tiles'"""
    M, N, K = shape
    for k, fits in ((K, False), (K - 256, True)):
        d = (mx(8, 64, 256, dt, "bf16") if dt.startswith("mx") else problem(8, 64, 256, dt, "bf16")).desc()
        d.N, d.K = N, k
        for s in (d.src_stride, d.wei_stride):
            for i in range(3):
                if s[i] == 256:
                    s[i] = k
        d.dst_stride[1] = N
        with cabi.tuning("MI355_F8_TILES", "wide"):
            unsplit = cabi.scratch_bytes(d)
        with cabi.tuning("MI355_F8_TILES", "small"):
            assert (cabi.scratch_bytes(d) == unsplit) == fits, k


def test_kernels_that_read_no_parts_have_no_arguments_for_them(tmp_path):
    """the launch of a small int8 product is a few microseconds, and every argument is written to the device for it"""
    from tests.test_loop_isa import OBJDUMP
    readelf = OBJDUMP.replace("objdump", "readelf")
    if not os.path.exists(readelf):
        pytest.skip("no disassembler")
    os.symlink(os.path.abspath(cabi.KERNEL_LIB_PATH), tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    size = {}
    for f in os.listdir(tmp_path):
        if "gfx950" in f:
            notes = subprocess.run([readelf, "--notes", f], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
            for k in notes.split("- .agpr_count")[1:]:
                name = re.search(r"\.name: +(\S*chain_\S*kernel\S*)", k)
                if name:
                    size[name.group(1)] = int(re.search(r"\.kernarg_segment_size: (\d+)", k).group(1))
    part = re.compile(r"chain_gemm_kernel.*Li4EE|chain_sum_kernel|chain_small_float")
    with_parts, without = ({v for k, v in size.items() if bool(part.search(k)) == w} for w in (True, False))
    assert len(size) > 60 and len(without) == 1 and max(without) <= min(with_parts) - 48, (with_parts, without)


# steps of the last part: whole, one chunk, a chunk short of a step
@pytest.mark.gpu
@pytest.mark.parametrize("tail", [0, 16, 112])
@pytest.mark.parametrize("dt,ddt,kw", [
    ("bf16", "bf16", dict(bias=True)), ("bf16", "f16", {}), ("bf16", "f32", {}), ("f16", "f16", dict(post=[RELU])), ("f16", "bf16", {}),
    ("s8", "s8", dict(post=[RELU], dst_scale=3.0)), ("s8", "f32", dict(bias=True)), ("u8", "u8", dict(bias=True, src_zp=5, dst_scale=0.7)),
    ("u8", "bf16", dict(src_zp=2)), ("f8_e4m3", "bf16", dict(row_scales=True, post=[RELU])), ("f8_e4m3", "f32", dict(bias=True))])
def test_split_sums(gpu, oracle, dt, ddt, kw, tail):
    steps = 41 if BYTES[dt] == 2 else 257  # (int8: beyond where the 32 x 32 tiles are taken)
    for M, N, batch in ((130, 333 if ddt == "s8" else 268, 1), (260, 136, 2)):
        pitch = -(-N // 16) * 16
        p = problem(M, N, (steps * 128 + tail) // BYTES[dt], dt, ddt, batch=batch, pitch=pitch, **kw)
        assert parts_of(p) >= 4
        with cabi.tuning("MI355_EPILOGUE", "chain"):
            got, name = run_gpu(p)
        assert name.startswith(FAMILY[dt]), name
        assert_bit_exact(p, got, oracle.run_oracle(p), name)


@pytest.mark.gpu
@pytest.mark.parametrize("act", [None, "gelu_tanh", "swish"])
@pytest.mark.parametrize("alg", ["add", "mul"])
@pytest.mark.parametrize("dt", ["bf16", "f8_e4m3"])
def test_split_sums_with_a_second_tensor(gpu, oracle, act, alg, dt):
    """with an activation within its few ulp of the oracle, rounded to bf16: two units of bf16"""
    M, N, K = 150, 200, 8192
    other = dtp.f32_to_bf16(np.random.default_rng(5).integers(-4, 5, size=M * N).astype(np.float32)).reshape(M, N)
    post = [PostOp(cabi.PO_ELTWISE, alg=cabi.ELTWISE[act], alpha=1.0)] if act else []
    post.append(PostOp(cabi.PO_BINARY, alg=cabi.BINARY[alg], dt=cabi.DT_BF16, stride=(M * N, N, 1), data=other))
    p = problem(M, N, K, dt, "bf16", bias=True, post=post)
    if dt == "f8_e4m3":
        p.quant["src_scale"].data[:] /= 64
    assert parts_of(p) >= 4
    got, name = run_gpu(p)
    want = oracle.run_oracle(p)
    if not act:
        assert_bit_exact(p, got, want, name)
        return
    g, w = (dtp.bf16_to_f32(np.asarray(x).view(np.uint16).reshape(-1)) for x in (got, want))
    assert np.all(np.abs(g - w) <= 2.0 ** -7 * np.abs(w) + 2.0 ** -20)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [2560, 2568, 2616])
@pytest.mark.parametrize("src_across", [False, True])
@pytest.mark.parametrize("dt,ddt", [("bf16", "bf16"), ("f16", "f32")])
def test_split_operands_across_k(gpu, oracle, K, src_across, dt, ddt):
    p = across_problem(304, 328, K, dt, ddt, src_across, batch=2, wei_pad=8, src_pad=16)
    assert parts_of(p) >= 4
    got, name = run_gpu(p)
    assert_bit_exact(p, got, oracle.run_oracle(p), name)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,K", [("mxf8", 8192), ("mxf8", 8288), ("mxf4", 16384), ("mxf4", 16416), ("mxf4", 16640)])
@pytest.mark.parametrize("ddt", ["f32", "bf16"])
def test_split_block_scales(gpu, oracle, fmt, K, ddt):
    p = mx(300, 200, K, fmt, ddt)
    assert parts_of(p) >= 4
    got, name = run_gpu(p)
    assert_bit_exact(p, got, oracle.run_oracle(p), name)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["bf16", "s8", "f8_e4m3"])
def test_without_scratch(gpu, oracle, dt):
    """a problem whose scratch is for parts alone runs without"""
    p = problem(260, 264, 32768 // BYTES[dt], dt, "f32", bias=True)
    want = oracle.run_oracle(p)
    run = GpuRun(p)
    try:
        assert run.scratch is not None
        run.launch()
        assert_bit_exact(p, run.result(), want, "split")
        run.reset_dst()
        run.scratch.free()
        run.scratch = None
        run.launch()
        assert_bit_exact(p, run.result(), want, "without scratch")
        run.reset_dst()
        cabi.check(run.lib.mi355_matmul_launch_noalloc(run.desc, run.args, None))
        assert_bit_exact(p, run.result(), want, "noalloc")
    finally:
        run.free()

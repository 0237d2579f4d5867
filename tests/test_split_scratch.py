"""Where the partial sums of a split K lie (onednn_amd/host/dnnl_api.cpp, parts_pool_t): in buffers that the primitives of a device
share, so that a primitive holds no memory for them, its executions on several streams do not wait for each other, and a
captured one keeps none.

Exact data (any order of the sum gives the same bits) against the oracle, bit for bit.
"""
import ctypes as C
import os
import threading

import numpy as np
import pytest

os.environ["ONEDNN_AMD_ALLOW_NO_DEVICE"] = "1"

from onednn_amd import cabi, dnnl  # noqa: E402
from onednn_amd.problem import GpuRun, storage_dtype  # noqa: E402
from tests.helpers import assert_bit_exact  # noqa: E402
from tests.test_line_loops import across_problem, problem  # noqa: E402

MIB = 1 << 20
DT = cabi.DT_NAMES
# type, dst, M, N, K: with K-contiguous operands they need no scratch of their own
ALONE = [("bf16", "bf16", 512, 1024, 8192), ("f16", "f32", 260, 264, 16384), ("f8_e4m3", "bf16", 256, 4352, 12224),
         ("s8", "s8", 1024, 1024, 4096), ("u8", "f32", 1024, 1024, 4096)]


def make(case):
    dt, ddt, M, N, K = case
    return problem(M, N, K, dt, ddt, src_zp=3 if dt == "u8" else None)


def pd_of(p, user=False, eng=None):
    eng = eng or dnnl.engine(dnnl.gpu, 0)
    attr = dnnl.primitive_attr()
    if "src_scale" in p.quant:
        attr.set_scales_mask(dnnl.ARG_SRC, 0)
        attr.set_scales_mask(dnnl.ARG_WEIGHTS, 2)
    if "src_zp" in p.quant:
        attr.set_zero_points_mask(dnnl.ARG_SRC, 0)
    if user:
        attr.set_scratchpad_mode(dnnl.scratchpad_user)
    return dnnl.matmul_primitive_desc(
        eng, dnnl.memory_desc([p.M, p.K], p.src_dt, strides=list(p.src_stride[1:])),
        dnnl.memory_desc([p.K, p.N], p.wei_dt, strides=list(p.wei_stride[1:])),
        dnnl.memory_desc([p.M, p.N], p.dst_dt, tag=dnnl.tag_ab), attr=attr)


def consumption(pd):
    v = C.c_int64(-1)
    assert dnnl.lib().dnnl_primitive_desc_query(pd.h, dnnl.query_memory_consumption, 0, C.byref(v)) == dnnl.success
    return v.value


@pytest.mark.parametrize("case", ALONE, ids=str)
def test_a_primitive_holds_nothing_for_the_parts(case):
    """and is created where there is no memory for them (without a device: none at all)"""
    p = make(case)
    own, parts = cabi.scratch_parts(p.desc())
    assert own == 0 and MIB < parts <= 64 * MIB and parts == cabi.scratch_bytes(p.desc())
    pd = pd_of(p)
    assert consumption(pd) == 0 and pd.scratchpad_desc().get_size() == 0
    dnnl.matmul(pd)
    assert pd_of(p, user=True).scratchpad_desc().get_size() == parts


def test_what_a_launch_cannot_do_without():
    """both operands across K: room for their copies; weights across K: the transposed ones and the sums"""
    p = across_problem(512, 512, 8192, "bf16", "bf16", True)
    own, parts = cabi.scratch_parts(p.desc())
    assert own == 2 * 512 * 8192 * 2 and MIB < parts <= 64 * MIB and own + parts == cabi.scratch_bytes(p.desc())
    assert consumption(pd_of(p)) == own
    for K, N in ((1024, 1024), (4096, 1024)):   # not split, split
        d = problem(1024, N, K, "u8", "f32", src_zp=3).desc()
        d.wei_stride[0], d.wei_stride[1], d.wei_stride[2] = K * N, N, 1
        own, parts = cabi.scratch_parts(d)
        assert own == K * N + 4 * N and own + parts == cabi.scratch_bytes(d) and (parts > 0) == (K == 4096)


class Device:
    """The problem's tensors on the device, a dst for every stream."""

    def __init__(self, p, streams=1):
        self.p, self.eng = p, dnnl.engine(dnnl.gpu, 0)
        md = lambda dims, dt, strides: dnnl.memory_desc(dims, dt, strides=list(strides))  # noqa: E731
        self.args = {dnnl.ARG_SRC: dnnl.memory(md([p.M, p.K], p.src_dt, p.src_stride[1:]), self.eng, p.src),
                     dnnl.ARG_WEIGHTS: dnnl.memory(md([p.K, p.N], p.wei_dt, p.wei_stride[1:]), self.eng, p.wei)}
        for q, arg in (("src_scale", dnnl.ARG_ATTR_SCALES | dnnl.ARG_SRC), ("wei_scale", dnnl.ARG_ATTR_SCALES | dnnl.ARG_WEIGHTS),
                       ("src_zp", dnnl.ARG_ATTR_ZERO_POINTS | dnnl.ARG_SRC)):
            if q in p.quant:
                data = p.quant[q].data
                self.args[arg] = dnnl.memory(dnnl.memory_desc([data.size], p.quant[q].dt, tag=dnnl.tag_a), self.eng, data)
        self.dst_md = dnnl.memory_desc([p.M, p.N], p.dst_dt, tag=dnnl.tag_ab)
        self.dst = [dnnl.memory(self.dst_md, self.eng) for _ in range(streams)]

    def with_dst(self, i):
        return {**self.args, dnnl.ARG_DST: self.dst[i]}

    def clear(self, i):
        self.dst[i].write(np.full(self.dst_md.get_size(), 0x5A, np.uint8))

    def check(self, i, want, what):
        assert_bit_exact(self.p, self.dst[i].read(storage_dtype(self.p.dst_dt)), want, what)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [ALONE[0], ALONE[2], ALONE[4]], ids=str)
def test_primitives_threads_and_streams(gpu, oracle, case):
    """two primitives of a problem, six threads with a stream each, three executions in flight on each"""
    p = make(case)
    want = oracle.run_oracle(p)
    D = Device(p, 18)
    prims = [dnnl.matmul(pd_of(p, eng=D.eng)) for _ in range(2)]
    errors = []

    def worker(t):
        try:
            s = dnnl.stream(D.eng)
            for _ in range(8):
                for i in range(3):
                    prims[(t + i) % 2].execute(s, D.with_dst(3 * t + i))
                s.wait()
                for i in range(3):
                    D.check(3 * t + i, want, f"thread {t}")
                    D.clear(3 * t + i)
        except BaseException as e:  # noqa: B902
            errors.append(e)

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(6)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors[0]


@pytest.mark.gpu
def test_one_thread_and_more_streams_than_buffers(gpu, oracle):
    p = make(ALONE[0])
    want = oracle.run_oracle(p)
    D = Device(p, 20)
    prim = dnnl.matmul(pd_of(p, eng=D.eng))
    streams = [dnnl.stream(D.eng) for _ in range(20)]
    for _ in range(3):
        for i, s in enumerate(streams):
            prim.execute(s, D.with_dst(i))
        for i, s in enumerate(streams):
            s.wait()
            D.check(i, want, f"stream {i}")
            D.clear(i)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [ALONE[0], ALONE[4]], ids=str)
def test_captured_after_it_ran_on_another_stream(gpu, oracle, case):
    """and replayed beside eager executions of the same primitive and of another one"""
    p = make(case)
    want = oracle.run_oracle(p)
    D = Device(p, 3)
    prim, other = (dnnl.matmul(pd_of(p, eng=D.eng)) for _ in range(2))
    eager = dnnl.stream(D.eng)
    hs = cabi.Stream()
    captured = dnnl.stream(D.eng, hip_stream=hs.ptr)
    try:
        prim.execute(eager, D.with_dst(0))
        with cabi.Graph(hs) as g:
            prim.execute(captured, D.with_dst(1))
            other.execute(eager, D.with_dst(2))     # not the capture's concern
        for _ in range(4):
            eager.wait()
            for i in range(3):
                D.clear(i)
            g.launch()
            prim.execute(eager, D.with_dst(0))
            other.execute(eager, D.with_dst(2))
            hs.sync()
            eager.wait()
            for i in range(3):
                D.check(i, want, "captured" if i == 1 else "eager")
        g.destroy()
    finally:
        hs.destroy()


@pytest.mark.gpu
def test_the_users_scratchpad(gpu, oracle):
    """one that is for the parts alone may be left out, as where there were no parts; another may not"""
    p = make(ALONE[0])
    want = oracle.run_oracle(p)
    D = Device(p)
    s = dnnl.stream(D.eng)
    pd = pd_of(p, user=True, eng=D.eng)
    prim = dnnl.matmul(pd)
    for extra in ({}, {dnnl.ARG_SCRATCHPAD: dnnl.memory(pd.scratchpad_desc(), D.eng)}):
        D.clear(0)
        prim.execute(s, {**D.with_dst(0), **extra})
        s.wait()
        D.check(0, want, "scratchpad" if extra else "none")
    p = across_problem(512, 512, 8192, "bf16", "bf16", True)
    D = Device(p)
    prim = dnnl.matmul(pd_of(p, user=True, eng=D.eng))
    with pytest.raises(dnnl.error) as e:
        prim.execute(dnnl.stream(D.eng), D.with_dst(0))
    assert e.value.status == dnnl.invalid_arguments


@pytest.mark.gpu
@pytest.mark.parametrize("across", [False, True])
def test_both_buffers_of_a_launch(gpu, oracle, across):
    p = across_problem(512, 512, 8192, "bf16", "bf16", True) if across else make(ALONE[4])
    want = oracle.run_oracle(p)
    run = GpuRun(p)
    own, parts = (cabi.DeviceBuffer(n) if n else None for n in cabi.scratch_parts(run.desc))
    try:
        for second in (parts, None):
            run.reset_dst()
            cabi.check(run.lib.mi355_matmul_launch_parts(C.byref(run.desc), C.byref(run.args), own.ptr if own else None,
                                                         second.ptr if second else None, None))
            assert_bit_exact(p, run.result(), want, "split" if second else "not split")
        if across:
            assert run.lib.mi355_matmul_launch_parts(C.byref(run.desc), C.byref(run.args), None, parts.ptr, None) == cabi.INVALID_ARGUMENTS
    finally:
        run.free()
        for b in (own, parts):
            if b:
                b.free()

"""mi355_colsum_launch: column sums in the order of the rows, bit for bit, at the edges of the chunks the kernel walks
(128 rows of a 16-bit type, 64 of f32; 64 columns a workgroup) and of its 16-byte column groups."""
import numpy as np
import pytest

from onednn_amd import cabi
from onednn_amd import dtypes as dtp


def in_order(x):
    acc = np.zeros(x.shape[1], np.float32)
    for row in x:
        acc = acc + row
    return acc


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("rows", [1, 2, 63, 65, 127, 128, 129, 256, 300, 1000])
@pytest.mark.parametrize("cols,ld", [(8, 8), (64, 64), (72, 80), (100, 100), (200, 264)])
def test_column_sums_keep_the_order_of_the_rows(gpu, dt, rows, cols, ld):
    v = np.random.default_rng([rows, cols]).standard_normal((rows, ld)).astype(np.float32)
    raw, x = {"bf16": lambda: (dtp.f32_to_bf16(v.reshape(-1)).reshape(v.shape), None),
              "f16": lambda: (v.astype(np.float16), v.astype(np.float16).astype(np.float32)), "f32": lambda: (v, v)}[dt]()
    if x is None:
        x = dtp.bf16_to_f32(raw.reshape(-1)).reshape(v.shape)
    src, out = cabi.DeviceBuffer.from_numpy(raw), cabi.DeviceBuffer.from_numpy(np.full(cols + 1, 7, np.float32))
    lib = cabi.load_kernels()
    cabi.check(lib.mi355_colsum_launch(src.ptr, cabi.DT_NAMES[dt], rows, cols, ld, out.ptr, cabi.DT_F32, None))
    cabi.check(lib.mi355_stream_sync(None))
    got = out.to_numpy(np.float32, (cols + 1,))
    assert np.array_equal(got[:cols], in_order(x[:, :cols])) and got[cols] == 7

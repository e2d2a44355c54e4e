"""The device quantisers' vector forms against the element-wise ones and the host rules, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from tests.gpu_util import Dev, lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    import atlas_amd
    atlas_amd.load()
    if not lib().atlas_cuda_available():
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def _matrix(rows, cols, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    f = w.reshape(-1)
    f[rng.integers(0, f.size, max(1, f.size // 50))] = 0.0
    f[0], f[f.size // 3], f[f.size // 2], f[-1] = np.nan, np.inf, -np.inf, np.float32(1e-40)
    if rows > 2:
        w[1] = 0.0                                   # all zero: scale 1
        w[2, :min(cols, 6)] = np.float32(0.01) * np.array([127, 2.5, -2.5, 0.5, -0.5, 7], np.float32)[:min(cols, 6)]
    return w


# columns on both sides of one load per lane, of one wave's and of one block's
# registers; columns that are no multiple of 8 and sources off a 16-byte line
# take the element-wise kernel
@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("rows,cols,off", [(5, 8, 0), (3, 504, 0), (6, 4096, 0), (7, 4104, 0), (3, 16384, 0),
                                           (3, 16392, 0), (5, 100, 0), (4, 512, 4), (1, 2048, 0)])
def test_int8_rows(orc, bf16, rows, cols, off):
    print(f"quant int8 bf16={bf16} {rows}x{cols} off={off}", flush=True)
    w = _matrix(rows, cols, rows * cols)
    src = orc.bf16_from_f32(w) if bf16 else w
    wide = np.ascontiguousarray(orc.bf16_to_f32(src) if bf16 else w, np.float32)
    q = np.empty(rows * cols, np.int8)
    s = np.empty(rows, np.float32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    assert lib().atlas_quantize_int8_host(p(wide), rows, cols, p(q), p(s)) == 0
    raw = np.concatenate([np.zeros(off, np.uint8), np.frombuffer(np.ascontiguousarray(src).tobytes(), np.uint8)])
    d, dq, ds = Dev(raw), Dev(np.full(rows * cols + 16, 99, np.int8)), Dev.empty(rows)
    assert lib().atlas_quantize_int8_dev(d.ptr + off, bf16, rows, cols, dq.ptr, ds.ptr) == 0
    got = dq.get()
    assert np.array_equal(got[:-16], q) and np.all(got[-16:] == 99) and np.array_equal(ds.get(), s)


# blocks of one lane's elements up to a whole wave's and beyond, blocks that are
# no power of two, a last block that is cut, element counts off a multiple of 8
@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("n,block,off", [(4096, 8, 0), (4096, 32, 0), (8192, 512, 0), (4096, 1024, 0), (4104, 64, 0),
                                         (1000, 512, 0), (2040, 50, 0), (1030, 32, 0), (1024, 32, 4), (24, 256, 0)])
def test_int4_blocks(orc, bf16, n, block, off):
    print(f"quant int4 bf16={bf16} n={n} block={block} off={off}", flush=True)
    w = _matrix(1, n, n + block)
    src = orc.bf16_from_f32(w) if bf16 else w
    wide = np.ascontiguousarray(orc.bf16_to_f32(src) if bf16 else w, np.float32)
    nb = (n + block - 1) // block
    q = np.empty((n + 1) // 2, np.uint8)
    s = np.empty(nb, np.float32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    assert lib().atlas_quantize_int4_host(p(wide), 1, n, block, p(q), p(s)) == 0
    raw = np.concatenate([np.zeros(off, np.uint8), np.frombuffer(np.ascontiguousarray(src).tobytes(), np.uint8)])
    d, dq, ds = Dev(raw), Dev(np.full(q.size + 16, 99, np.uint8)), Dev(np.full(nb + 4, 7, np.float32))
    assert lib().atlas_quantize_int4_dev(d.ptr + off, bf16, n, block, dq.ptr, ds.ptr) == 0
    got, gs = dq.get(), ds.get()
    assert np.array_equal(got[:-16], q) and np.all(got[-16:] == 99)
    assert np.array_equal(gs[:-4], s) and np.all(gs[-4:] == 7)

"""The prompt chunks' and ragged batches' GEMMs at the edges of their tiles, rings and K splits."""
import ctypes as C
import threading

import numpy as np
import pytest

from tests.gpu_util import Dev, lib
from tests.test_gpu_kernels import _hip_runtime

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    import atlas_amd
    atlas_amd.load()
    if not lib().atlas_cuda_available():
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def _stored(orc, w, fmt, block):
    """(data, scales, the matrix in f64, the largest |stored integer step| per element)"""
    if fmt == "bf16":
        b = orc.bf16_from_f32(w)
        return b, None, orc.bf16_to_f32(b).astype(np.float64)
    if fmt == "int8":
        q, s = orc.int8_quantize(w)
        return q, s, orc.int8_dequantize(q, s).astype(np.float64)
    q, s = orc.int4_quantize(w, block)
    return q, s, orc.int4_dequantize(q, s, w.shape[0], w.shape[1], block).astype(np.float64)


# rows on both sides of the 64- and 128-row tiles, weight rows on both sides of
# the 128-, 192- and 256-row tiles, one unit of K, fewer steps than a ring, odd
# split remainders, enough weight rows that nothing splits, blocks over several
# steps, and weights that start 4 or 8 bytes off a 16-byte line
@pytest.mark.parametrize("fmt,n,M,K,block,off", [
    (f, n, M, K, 32, 0) for f in ("bf16", "int8", "int4")
    for n, M, K in [(2, 65, 4224), (3, 640, 128), (8, 129, 896), (9, 64, 1152), (16, 1000, 11008),
                    (13, 22016, 128), (32, 127, 1280), (17, 1, 128), (33, 130, 128), (64, 255, 256), (65, 257, 384), (127, 193, 640),
                    (128, 128, 1152), (129, 2050, 512), (200, 384, 4224), (257, 100, 2048),
                    (300, 6144, 896), (1001, 320, 256), (40, 33000, 256), (130, 33000, 128)]] + [
    ("int8", 100, 300, 640, 32, 8), ("int8", 30, 129, 256, 32, 8), ("int4", 100, 300, 640, 32, 4),
    ("int4", 30, 129, 256, 64, 12), ("int4", 150, 260, 1280, 128, 0), ("int4", 70, 97, 512, 256, 0)])
@pytest.mark.parametrize("epi", ["store", "swiglu"])
def test_prompt_gemm(orc, fmt, n, M, K, block, off, epi):
    print(f"prompt gemm {fmt} n={n} M={M} K={K} block={block} off={off} {epi}", flush=True)
    if epi == "swiglu":
        if M > 3000:
            pytest.skip("one epilogue is enough at this size")
        M += M % 2
    rng = np.random.default_rng(M * K + n)
    w = (rng.standard_normal((M, K)) * 0.02).astype(np.float32)
    x = (rng.standard_normal((n, K)) * np.exp(0.7 * rng.standard_normal(K))).astype(np.float32)
    data, scales, w64 = _stored(orc, w, fmt, block)
    raw = np.frombuffer(np.ascontiguousarray(data).tobytes(), np.uint8)
    dw = Dev(np.concatenate([np.zeros(off, np.uint8), raw]))
    ds, dx = (Dev(scales) if scales is not None else None), Dev(x)
    f = {"bf16": 1, "int8": 2, "int4": 3}[fmt]
    cols = M // 2 if epi == "swiglu" else M
    dy = Dev(np.full((n, cols), np.nan, np.float32))
    fn = lib().atlas_gemm_skinny_swiglu_f32 if epi == "swiglu" else lib().atlas_gemm_skinny_f32
    assert fn(f, dw.ptr + off, ds.ptr if ds else None, block, dx.ptr, dy.ptr, cols, n, K) == 0
    got = dy.get().astype(np.float64)
    x64 = x.astype(np.float64)
    ref, mag = x64 @ w64.T, np.abs(x64) @ np.abs(w64).T
    if fmt == "int8":
        # three digits, where they are taken: 2^-24 of the row's largest element per
        # product, the sums exact, a few roundings to combine them
        dig = 2.0**-24 * np.max(np.abs(x64), 1)[:, None] * np.sum(np.abs(w64), 1)[None, :] + 8 * 2.0**-24 * np.abs(ref)
    # x in two bf16 parts: the remainder of an 8-bit truncation rounded to 8 bits,
    # 2^-16 of each product; sums of K products in f32: K/2 roundings of 2^-24
    # (tree or chain, both within K 2^-24 of the magnitudes)
    tol = (2.0**-16 + K * 2.0**-24) * mag
    if fmt == "int8":
        tol = np.maximum(tol, dig)
    if fmt == "int4":
        # each step's 32 products run around the offset 24: 33 roundings of
        # sums of at most 32 s |x| per element
        s_el = np.repeat(scales.astype(np.float64), block)[:M * K].reshape(M, K)
        tol = tol + 33 * 2.0**-24 * (np.abs(x64) @ (32.0 * s_el).T)
    if epi == "swiglu":
        g, u, tg, tu = ref[:, 0::2], ref[:, 1::2], tol[:, 0::2], tol[:, 1::2]
        sg = 1.0 / (1.0 + np.exp(-g))
        ref = g * sg * u
        # |silu'| <= 1.1; the epilogue itself rounds a few times
        tol = 1.1 * tg * np.abs(u) + np.abs(g * sg) * tu + 1.1 * tg * tu + 8 * 2.0**-24 * np.abs(ref)
    assert np.all(np.abs(got - ref) <= tol), float(np.max(np.abs(got - ref) / tol))


def test_int8_digits_special_rows(orc):
    # rows with a NaN, an infinity, only zeros, one huge element; the others are
    # untouched by them
    n, M, K = 300, 6200, 512
    print(f"int8 digits special rows n={n} M={M} K={K}", flush=True)
    rng = np.random.default_rng(5)
    w = (rng.standard_normal((M, K)) * 0.02).astype(np.float32)
    x = rng.standard_normal((n, K)).astype(np.float32)
    x[3, 17], x[130, 0], x[131], x[299, 511] = np.nan, np.inf, 0.0, 1e30
    q, s = orc.int8_quantize(w)
    w64 = orc.int8_dequantize(q, s).astype(np.float64)
    dw, ds, dx, dy = Dev(q), Dev(s), Dev(x), Dev(np.full((n, M), 7, np.float32))
    assert lib().atlas_gemm_skinny_f32(2, dw.ptr, ds.ptr, 0, dx.ptr, dy.ptr, M, n, K) == 0
    got = dy.get().astype(np.float64)
    assert np.all(np.isnan(got[3])) and not np.any(np.isfinite(got[130])) and np.all(got[131] == 0)
    rest = [i for i in range(n) if i not in (3, 130)]
    ref = x[rest].astype(np.float64) @ w64.T
    tol = (2.0**-24 * np.max(np.abs(x[rest]).astype(np.float64), 1)[:, None] * np.sum(np.abs(w64), 1)[None, :]
           + 8 * 2.0**-24 * np.abs(ref))
    assert np.all(np.abs(got[rest] - ref) <= tol)


# int8 shapes whose plan without the digits (a captured call has none) splits K
# more than the plan with them: six times against five, twice against not at all
@pytest.mark.parametrize("n,M,K", [(300, 2048, 4096), (700, 2048, 1024)])
def test_int8_captured_after_a_call_of_the_same_shape(orc, n, M, K):
    print(f"int8 prompt gemm captured n={n} M={M} K={K}", flush=True)
    hip = _hip_runtime()
    rng = np.random.default_rng(n)
    w = (rng.standard_normal((M, K)) * 0.02).astype(np.float32)
    x = rng.standard_normal((n, K)).astype(np.float32)
    q, s = orc.int8_quantize(w)
    w64, x64 = orc.int8_dequantize(q, s).astype(np.float64), x.astype(np.float64)
    res = {}

    def worker():                           # a thread of its own: its scratch starts empty
        st, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
        try:
            dw, ds, dx, dy = Dev(q), Dev(s), Dev(x), Dev(np.full((n, M), np.nan, np.float32))
            assert hip.hipStreamCreate(C.byref(st)) == 0
            lib().atlas_set_thread_stream(st)

            def call():
                return lib().atlas_gemm_skinny_f32(2, dw.ptr, ds.ptr, 0, dx.ptr, dy.ptr, M, n, K)

            assert call() == 0
            lib().atlas_stream_sync()
            res["eager"] = dy.get()
            assert hip.hipStreamBeginCapture(st, 0) == 0
            res["code"] = call()
            assert hip.hipStreamEndCapture(st, C.byref(graph)) == 0
            if res["code"]:
                return
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
            res["replays"] = []
            for _ in range(3):
                lib().atlas_memset_zero(dy.ptr, n * M * 4)     # eager work between replays
                lib().atlas_stream_sync()
                assert hip.hipGraphLaunch(exe, st) == 0
                assert hip.hipStreamSynchronize(st) == 0
                res["replays"].append(dy.get())
        except BaseException as e:          # reported on the main thread
            res["exc"] = e
        finally:
            lib().atlas_clear_thread_stream()
            if exe.value:
                hip.hipGraphExecDestroy(exe)
            if graph.value:
                hip.hipGraphDestroy(graph)
            if st.value:
                hip.hipStreamSynchronize(st)
                hip.hipStreamDestroy(st)

    t = threading.Thread(target=worker)
    t.start()
    t.join()
    if "exc" in res:
        raise res["exc"]
    assert res["code"] == 0, lib().atlas_last_error()
    # two bf16 parts of x and f32 sums, as above
    ref, tol = x64 @ w64.T, (2.0**-16 + K * 2.0**-24) * (np.abs(x64) @ np.abs(w64).T)
    for got in [res["eager"]] + res["replays"]:
        assert np.all(np.abs(got.astype(np.float64) - ref) <= tol)
        assert np.array_equal(got, res["replays"][0]) or got is res["eager"]

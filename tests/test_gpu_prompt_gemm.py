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


def _sum_tol(x64, w64):
    """|error| of Y = X W^T that x in two bf16 parts and f32 sums may show, per output, with S = |w x|_2:
    each product's error is at most 2^-16 of it and zero in the mean, so 2e-11 of the outputs leave 7 * 2^-16 S
    (Hoeffding); the same 7 S bounds the running sums, whose K / 16 additions (one per MFMA) and the few of the
    K split and the scale each lose at most 2^-22 of them, the alignment of an MFMA's own products included."""
    S = np.sqrt(np.square(x64) @ np.square(w64).T)
    return 7 * (2.0**-16 + (x64.shape[1] / 16 + 8) * 2.0**-22) * S


# rows on both sides of the 64- and 128-row tiles, weight rows on both sides of
# the 128-, 192- and 256-row tiles, one unit of K, fewer steps than a ring, odd
# split remainders, enough weight rows that nothing splits, blocks over several
# steps, and weights that start 4 or 8 bytes off a 16-byte line
@pytest.mark.parametrize("fmt,n,M,K,block,off", [
    (f, n, M, K, 32, 0) for f in ("bf16", "int8", "int4")
    for n, M, K in [(2, 65, 4224), (3, 640, 128), (8, 129, 896), (9, 64, 1152), (16, 1000, 11008),
                    (13, 22016, 128), (32, 127, 1280), (17, 1, 128), (33, 130, 128), (64, 255, 256), (65, 257, 384), (127, 193, 640),
                    (128, 128, 1152), (129, 2050, 512), (200, 384, 4224), (257, 100, 2048),
                    (300, 6144, 896), (1001, 320, 256), (40, 33000, 256), (130, 33000, 128),
                    # (of 256 CUs) 192 x 128, 256 x 128 split in three, 256 x 64, and 128 weight rows at 1, 2 and 4
                    # activation tiles of the few-rows kernel; the ones above take 128 x 128, 64 rows and 256 x 64
                    (200, 16902, 1152), (600, 4100, 4224), (130, 17002, 1152), (13, 17002, 1152), (24, 17002, 1152),
                    (40, 17002, 1152)]] + [
    ("int8", 100, 300, 640, 32, 8), ("int8", 30, 129, 256, 32, 8), ("int4", 100, 300, 640, 32, 4),
    ("int4", 30, 129, 256, 64, 12), ("int4", 150, 260, 1280, 128, 0), ("int4", 70, 97, 512, 256, 0)])
@pytest.mark.parametrize("epi", ["store", "swiglu"])
def test_prompt_gemm(orc, fmt, n, M, K, block, off, epi):
    print(f"prompt gemm {fmt} n={n} M={M} K={K} block={block} off={off} {epi}", flush=True)
    if epi == "swiglu":
        if M > 3000 and n != 200:
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
    ref, tol = x64 @ w64.T, _sum_tol(x64, w64)
    if epi == "swiglu":
        g, u, tg, tu = ref[:, 0::2], ref[:, 1::2], tol[:, 0::2], tol[:, 1::2]
        sg = 1.0 / (1.0 + np.exp(-g))
        ref = g * sg * u
        # |silu'| <= 1.1; the epilogue itself rounds a few times
        tol = 1.1 * tg * np.abs(u) + np.abs(g * sg) * tu + 1.1 * tg * tu + 8 * 2.0**-24 * np.abs(ref)
    assert np.all(np.abs(got - ref) <= tol), float(np.max(np.abs(got - ref) / tol))


@pytest.mark.parametrize("n", [13, 60, 300])        # the few-rows and the tiled kernel
@pytest.mark.parametrize("fmt", ["bf16", "int8", "int4"])
def test_rows_with_outliers_and_tiny_rows(orc, fmt, n):
    # Every element keeps 16 bits of its own, whatever the rest of its row is: rows with one element 2^8 to 2^20
    # times the others' size, whose weights there are stored as 0 in the first outputs; and rows so small that
    # 127 / max |x| is no f32 number.
    M, K = 6200, 1024
    print(f"outliers and tiny rows {fmt} n={n}", flush=True)
    rng = np.random.default_rng(11)
    w = (rng.standard_normal((M, K)) * 0.02).astype(np.float32)
    w[:M // 2, 100] = 0.0
    x = rng.standard_normal((n, K)).astype(np.float32)
    tiny = np.arange(n) % 3 == 2
    big = np.flatnonzero(~tiny)
    x[big, 100] = 2.0 ** (8 + big % 13)
    x[tiny] *= np.float32(1e-37)
    data, scales, w64 = _stored(orc, w, fmt, 32)
    dw, dx, dy = Dev(data), Dev(x), Dev(np.full((n, M), np.nan, np.float32))
    ds = Dev(scales) if scales is not None else None
    f = {"bf16": 1, "int8": 2, "int4": 3}[fmt]
    assert lib().atlas_gemm_skinny_f32(f, dw.ptr, ds.ptr if ds else None, 32, dx.ptr, dy.ptr, M, n, K) == 0
    got, x64 = dy.get().astype(np.float64), x.astype(np.float64)
    err, tol = np.abs(got - x64 @ w64.T), _sum_tol(x64, w64)
    assert np.all(err[~tiny] <= tol[~tiny]), float(np.max(err[~tiny] / tol[~tiny]))
    # a tiny row's low parts are below 2^-126, where the matrix cores may take them for 0: 2^-7 of the element,
    # all of one that is itself below; its f32 products with int8 or int4 weights are not
    if fmt != "bf16":
        tol = tol[tiny] + 7 * (2.0**-7 * np.sqrt(np.square(x64[tiny]) @ np.square(w64).T)
                               + 2.0**-126 * np.sqrt(np.sum(np.square(w64), 1)))
        assert np.all(err[tiny] <= tol), float(np.max(err[tiny] / tol))


def test_int8_special_rows(orc):
    # rows with a NaN, an infinity, only zeros, one huge element; the others are
    # untouched by them
    n, M, K = 300, 6200, 512
    print(f"int8 special rows n={n} M={M} K={K}", flush=True)
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
    x64 = x[rest].astype(np.float64)
    assert np.all(np.abs(got[rest] - x64 @ w64.T) <= _sum_tol(x64, w64))


# shapes whose plan splits K six times and twice
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
    assert np.all(np.abs(res["eager"].astype(np.float64) - x64 @ w64.T) <= _sum_tol(x64, w64))
    for got in res["replays"]:
        assert np.array_equal(got, res["eager"])


def _thread(fn):
    """fn(res) on a thread of its own (its scratch starts empty); what it raises is raised here"""
    res = {}

    def worker():
        try:
            fn(res)
        except BaseException as e:
            res["exc"] = e
        finally:
            lib().atlas_clear_thread_stream()

    t = threading.Thread(target=worker)
    t.start()
    t.join()
    if "exc" in res:
        raise res["exc"]
    return res


# A graph's K-split partials stay when a larger eager call outgrows them: the launches after it give the bits
# of the ones before, and leave memory allocated since alone.
def test_captured_scratch_outlives_growth(orc):
    M, K, n, n2 = 2048, 8192, 64, 700
    print(f"captured scratch outlives growth M={M} K={K} n={n} then {n2}", flush=True)
    hip = _hip_runtime()
    rng = np.random.default_rng(3)
    w = orc.bf16_from_f32((rng.standard_normal((M, K)) * 0.02).astype(np.float32))
    x = rng.standard_normal((n2, K)).astype(np.float32)

    def run(res):
        st, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
        dw, dx, dy, dz = Dev(w), Dev(x), Dev(np.zeros((n, M), np.float32)), Dev(np.zeros((n2, M), np.float32))
        assert hip.hipStreamCreate(C.byref(st)) == 0
        lib().atlas_set_thread_stream(st)
        small = lambda: lib().atlas_gemm_skinny_f32(1, dw.ptr, None, 0, dx.ptr, dy.ptr, M, n, K)
        try:
            assert small() == 0
            lib().atlas_stream_sync()
            res["eager"], held = dy.get(), lib().atlas_thread_scratch_bytes()
            assert held >= 2 * n * M * 4              # K is split
            assert hip.hipStreamBeginCapture(st, 0) == 0
            code = small()
            assert hip.hipStreamEndCapture(st, C.byref(graph)) == 0 and code == 0
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
            assert lib().atlas_gemm_skinny_f32(1, dw.ptr, None, 0, dx.ptr, dz.ptr, M, n2, K) == 0
            res["grown"] = lib().atlas_thread_scratch_bytes() - held
            others = [Dev(np.full(held // 16, 5, np.float32)) for _ in range(8)]
            for _ in range(3):
                lib().atlas_memset_zero(dy.ptr, n * M * 4)
                lib().atlas_stream_sync()
                assert hip.hipGraphLaunch(exe, st) == 0
                assert hip.hipStreamSynchronize(st) == 0
                assert np.array_equal(dy.get(), res["eager"])
            assert all(np.all(o.get() == 5) for o in others)
        finally:
            if exe.value:
                hip.hipGraphExecDestroy(exe)
            if graph.value:
                hip.hipGraphDestroy(graph)
            hip.hipStreamSynchronize(st)
            hip.hipStreamDestroy(st)

    # the larger call's buffer beside the graph's, which it does not replace
    assert _thread(run)["grown"] >= 2 * n2 * M * 4


# One thread's calls on two streams at once do not meet in its split-K scratch.
def test_scratch_of_two_streams(orc):
    M, K, n = 4096, 11008, 127
    print(f"scratch of two streams M={M} K={K} n={n}", flush=True)
    hip = _hip_runtime()
    rng = np.random.default_rng(4)
    w = orc.bf16_from_f32((rng.standard_normal((M, K)) * 0.02).astype(np.float32))
    xs = [rng.standard_normal((n, K)).astype(np.float32) for _ in range(4)]

    def run(res):
        streams = [C.c_void_p(), C.c_void_p()]
        dw, dx = Dev(w), [Dev(x) for x in xs]
        for st in streams:
            assert hip.hipStreamCreate(C.byref(st)) == 0

        def calls(pick, between):
            out = [Dev(np.full((n, M), np.nan, np.float32)) for _ in xs]
            lib().atlas_sync()
            for i, (x, y) in enumerate(zip(dx, out)):
                lib().atlas_set_thread_stream(streams[pick(i)])
                assert lib().atlas_gemm_skinny_f32(1, dw.ptr, None, 0, x.ptr, y.ptr, M, n, K) == 0
                between()
            lib().atlas_sync()
            return [y.get() for y in out]

        try:
            want = calls(lambda i: 0, lib().atlas_sync)
            assert lib().atlas_thread_scratch_bytes() >= 2 * n * M * 4          # K is split
            for _ in range(5):
                got = calls(lambda i: i % 2, lambda: None)
                assert all(np.array_equal(g, r) for g, r in zip(got, want))
        finally:
            lib().atlas_sync()
            lib().atlas_clear_thread_stream()
            for st in streams:
                hip.hipStreamDestroy(st)

    _thread(run)


def _rand_weights(fmt, M, K, seed):
    rng = np.random.default_rng(seed)
    if fmt == "bf16":
        w = (rng.standard_normal((M, K), np.float32) * np.float32(0.02)).view(np.uint32) >> 16
        return w.astype(np.uint16), None
    q = rng.integers(0, 256, M * K // (2 if fmt == "int4" else 1)).astype(np.uint8)
    return q, rng.uniform(1e-4, 2e-4, M if fmt == "int8" else M * K // 32).astype(np.float32)


def _eager_then_captured(fmt, M, K, rows, seed=9):
    """On a thread of its own: eager calls of all but the last of `rows`, then one of the last recorded and
    replayed three times.  (the last call's code, the replays, the data)"""
    hip = _hip_runtime()
    data, scales = _rand_weights(fmt, M, K, seed)
    x = np.random.default_rng(seed + 1).standard_normal((max(rows), K), np.float32)
    f = {"bf16": 1, "int8": 2, "int4": 3}[fmt]

    def run(res):
        st, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
        dw, dx, ds = Dev(data), Dev(x), Dev(scales) if scales is not None else None
        dy, n = Dev(np.zeros((max(rows), M), np.float32)), rows[-1]
        assert hip.hipStreamCreate(C.byref(st)) == 0
        lib().atlas_set_thread_stream(st)
        call = lambda r: lib().atlas_gemm_skinny_f32(f, dw.ptr, ds.ptr if ds else None, 32, dx.ptr, dy.ptr, M, r, K)
        try:
            for r in rows[:-1]:
                assert call(r) == 0
            lib().atlas_stream_sync()
            assert hip.hipStreamBeginCapture(st, 0) == 0
            res["code"] = call(n)
            assert hip.hipStreamEndCapture(st, C.byref(graph)) == 0
            if res["code"]:
                return
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
            res["got"] = []
            for _ in range(3):
                lib().atlas_memset_zero(dy.ptr, n * M * 4)     # eager work between replays
                lib().atlas_stream_sync()
                assert hip.hipGraphLaunch(exe, st) == 0
                assert hip.hipStreamSynchronize(st) == 0
                res["got"].append(dy.get()[:n])
            assert call(n) == 0
            lib().atlas_stream_sync()
            res["eager"] = dy.get()[:n]
        finally:
            if exe.value:
                hip.hipGraphExecDestroy(exe)
            if graph.value:
                hip.hipGraphDestroy(graph)
            hip.hipStreamSynchronize(st)
            hip.hipStreamDestroy(st)

    res = _thread(run)
    return res["code"], res.get("got"), res.get("eager"), data, x[:rows[-1]]


# fewer rows split K more, or take another kernel: 8 times against not at all, twice against not at all
@pytest.mark.parametrize("fmt,M,K,rows", [("bf16", 4096, 4096, (1024, 127)), ("int8", 22016, 4096, (1024, 127)),
                                          ("int4", 4096, 11008, (13, 6)), ("int4", 4096, 11008, (300, 6)),
                                          ("bf16", 4096, 11008, (40, 16, 9))])
def test_captured_after_a_larger_call(fmt, M, K, rows):
    print(f"captured after a larger call {fmt} M={M} K={K} rows={rows}", flush=True)
    code, got, eager, _, _ = _eager_then_captured(fmt, M, K, rows)
    assert code == 0, lib().atlas_last_error()
    assert all(np.array_equal(g, eager) for g in got)


# with no scratch, or too little, K is split less
@pytest.mark.parametrize("rows", [(64,), (13,), (128, 1000)])
def test_captured_with_less_scratch(rows):
    M, K = 2048, 8192
    print(f"captured with less scratch M={M} K={K} rows={rows}", flush=True)
    code, got, eager, data, x = _eager_then_captured("bf16", M, K, rows)
    assert code == 0, lib().atlas_last_error()
    w64 = (data.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    x64 = x.astype(np.float64)
    ref, tol = x64 @ w64.T, _sum_tol(x64, w64)
    assert np.all(np.abs(eager.astype(np.float64) - ref) <= tol)
    for g in got:
        assert np.array_equal(g, got[0]) and np.all(np.abs(g.astype(np.float64) - ref) <= tol)


def test_no_memory_for_the_partials():
    M, K, n = 2048, 8192, 64
    print(f"no memory for the partials M={M} K={K} n={n}", flush=True)
    data, _ = _rand_weights("bf16", M, K, 21)
    x = np.random.default_rng(22).standard_normal((n, K), np.float32)

    def run(res):
        dw, dx, dy = Dev(data), Dev(x), Dev(np.full((n, M), np.nan, np.float32))
        try:
            lib().atlas_debug_fail_allocations(0, 2)
            res["code"] = lib().atlas_gemm_skinny_f32(1, dw.ptr, None, 0, dx.ptr, dy.ptr, M, n, K)
        finally:
            lib().atlas_debug_fail_allocations(0, 0)
        res["error"], res["bytes"] = lib().atlas_last_error_code(), lib().atlas_thread_scratch_bytes()
        lib().atlas_stream_sync()
        res["got"] = dy.get().astype(np.float64)

    res = _thread(run)
    assert res["code"] == 0 and res["error"] == 0 and res["bytes"] == 0
    w64 = (data.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    x64 = x.astype(np.float64)
    assert np.all(np.abs(res["got"] - x64 @ w64.T) <= _sum_tol(x64, w64))


# Streams whose owner has destroyed them by the thread's next call, on another one; eight of them have scratch.
def test_scratch_after_its_stream_is_gone():
    M, K, n = 4096, 11008, 127
    print(f"scratch after its stream is gone M={M} K={K} n={n}", flush=True)
    hip = _hip_runtime()
    data, _ = _rand_weights("bf16", M, K, 23)
    x = np.random.default_rng(24).standard_normal((n, K), np.float32)

    def run(res):
        streams = [C.c_void_p() for _ in range(10)]
        dw, dx = Dev(data), Dev(x)
        for st in streams:
            assert hip.hipStreamCreate(C.byref(st)) == 0
        res["got"], res["bytes"] = [], []
        for st in streams:
            dy = Dev(np.full((n, M), np.nan, np.float32))
            lib().atlas_set_thread_stream(st)
            assert lib().atlas_gemm_skinny_f32(1, dw.ptr, None, 0, dx.ptr, dy.ptr, M, n, K) == 0
            lib().atlas_stream_sync()
            res["got"].append(dy.get())
            res["bytes"].append(lib().atlas_thread_scratch_bytes())
            lib().atlas_clear_thread_stream()
            assert hip.hipStreamDestroy(st) == 0

    res = _thread(run)
    assert all(np.array_equal(g, res["got"][0]) for g in res["got"])
    assert res["bytes"] == [min(i, 8) * res["bytes"][0] for i in range(1, 11)]

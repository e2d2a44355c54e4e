"""Pre-norm (Llama-wired) models on the fused decode step and in prompt chunks."""
import numpy as np
import pytest

from tests import modelgen

pytestmark = pytest.mark.gpu

LOGIT_TOL = 1e-3


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    import atlas_amd
    if not atlas_amd.load().atlas_cuda_available():
        pytest.fail("no HIP device visible: GPU tests need an MI355X")


def _rel(a, b):
    return float(np.max(np.abs(np.asarray(a, np.float64) - b)) / np.max(np.abs(b)))


def _cfg(**kw):
    base = dict(vocab=520, d_model=256, n_layers=2, n_heads=4, n_kv_heads=2, ffn_hidden=512, max_seq=420,
                post_norm=False, qk_norm=False, sliding_window=40, layer_sliding=[1, 0])
    return modelgen.tiny_config(**dict(base, **kw))


# head dims 64 and 128, grouped-query ratios 1, 2 and 4, with and without
# QK-norm, inner dimensions that allow prompt chunks and ones that do not
# (d 320, ffn 352), and a d_model past the register staging of the norms
@pytest.mark.parametrize("fmt", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("kw", [dict(), dict(n_heads=2, n_kv_heads=2), dict(n_kv_heads=1, qk_norm=True),
                                dict(d_model=320, n_heads=5, n_kv_heads=5, ffn_hidden=352),
                                dict(d_model=4352, n_heads=34, n_kv_heads=17, n_layers=1, layer_sliding=[0])])
def test_decode_matches_oracle(orc, fmt, kw):
    if kw.get("d_model") == 4352 and fmt != "bf16":
        pytest.skip("one format is enough for the wide model")
    cfg = _cfg(**kw)
    print(f"pre-norm decode {fmt} {kw}", flush=True)
    W = modelgen.make_weights(cfg, seed=23, fmt=fmt)
    m, o = modelgen.engine_model(W), modelgen.oracle_model(W, threads=8)
    toks = [int(t) for t in np.random.default_rng(2).integers(0, cfg["vocab"], 50)]
    for i, t in enumerate(toks):
        lg, lo = m.forward_one(t), o.forward_one(t)
        assert _rel(lg, lo) <= LOGIT_TOL, i
    m.reset()
    o.reset()
    lg, hid = m.forward_one_hidden(7)
    lo, ho = o.forward_one(7, hidden=True)
    for li in range(cfg["n_layers"]):
        assert _rel(hid[li], ho[li]) <= LOGIT_TOL, li
    from atlas_amd.model import SamplingConfig
    want = o.generate_greedy(toks[:9], 12)
    got = m.generate_with_sampling(toks[:9], 12, SamplingConfig.greedy())
    assert got[0] == want[0]
    m.use_graph(False)
    m.reset()
    eager = [m.forward_one(t) for t in toks[:5]]
    m.use_graph(True)
    m.reset()
    assert all(np.array_equal(m.forward_one(t), e) for t, e in zip(toks[:5], eager))


# bf16 and int8: a chunk carries the 24 bits of the decode step's f32 products.
# Both sides then differ by f32 rounding alone: a sum of K <= 512 terms walks to
# about 2^-25 sqrt(K / 2) / sqrt(3) < 3e-7 of its value, 2 layers x 4 products x
# 2 sides of it 1.1e-6, the largest of 520 logits three times that.  (Two bf16
# parts would leave 1.4e-5.)  int4's decode step holds 16-bit products.
@pytest.mark.parametrize("fmt,tol", [("bf16", 4e-6), ("int8", 4e-6), ("int4", LOGIT_TOL)])
@pytest.mark.parametrize("kw", [dict(), dict(n_heads=2, n_kv_heads=2, ffn_hidden=640, d_model=256)])
def test_prompt_chunks_match_token_by_token(orc, fmt, tol, kw):
    cfg = _cfg(**kw)
    W = modelgen.make_weights(cfg, seed=29, fmt=fmt)
    m = modelgen.engine_model(W, max_batch=3)
    toks = [int(t) for t in np.random.default_rng(3).integers(0, cfg["vocab"], 402)]
    ns = (2, 3, 8, 9, 16, 17, 33, 65, 130, 401)
    m.set_prefill_chunk(1)
    ref = {}
    for n in ns:
        m.reset()
        m.prefill(toks[:n])
        ref[n] = m.forward_one(toks[n])
    m.set_prefill_chunk(1024)
    for n in ns:
        print(f"pre-norm chunk {fmt} {kw} n={n}", flush=True)
        m.reset()
        m.prefill(toks[:n])
        assert m.pos == n
        assert _rel(m.forward_one(toks[n]), ref[n]) <= tol, n
    # a ragged batch of them: each sequence's tokens are its own generate's
    from atlas_amd.model import SamplingConfig
    prompts = [toks[:5], toks[10:60], toks[100:101]]
    got = m.generate_batch(prompts, 4)
    for p, g in zip(prompts, got):
        assert len(g) == 4 and g[0] == m.generate_with_sampling(p, 4, SamplingConfig.greedy())[0]


# A 1B model's widths, in two layers so that every product of the first reaches the logits: chunks of 13, 30 and 60
# rows take the few-rows kernel's 64- and 128-row blocks, 300 and 600 the four tiles (of 256 CUs: 256 x 64, 128 x 128,
# 256 x 128; 128 x 128, 192 x 128, 256 x 128).  Running sums of K / 32 <= 256 steps walk to 2^-25 / sqrt(3) * 2
# sqrt(256 / 2) = 4e-7 of their value, 16 of them to 1.6e-6, of the largest of the logits' differences and of the
# logits alike; two and a half times that.  Two bf16 parts in place of three would leave 1.4e-5.
@pytest.mark.parametrize("fmt", ["bf16", "int8"])
def test_prompt_chunks_of_a_1b_layer(orc, fmt):
    cfg = _cfg(d_model=2048, n_heads=16, n_kv_heads=4, ffn_hidden=8192, max_seq=640, sliding_window=0,
               layer_sliding=[0, 0])
    m = modelgen.engine_model(modelgen.make_weights(cfg, seed=31, fmt=fmt))
    toks = [int(t) for t in np.random.default_rng(5).integers(0, cfg["vocab"], 601)]
    for n in (13, 30, 60, 300, 600):
        print(f"pre-norm 1B chunk {fmt} n={n}", flush=True)
        got = []
        for chunk in (1, 1024):
            m.set_prefill_chunk(chunk)
            m.reset()
            m.prefill(toks[:n])
            got.append(m.forward_one(toks[n]))
        assert _rel(got[1], got[0]) <= 4e-6, n

"""GPU parity of the BERT text encoder (gsvk_bert_*, csrc/bert.hip) against the float64 oracle
(oracle/bert_oracle.py, a restatement of src/gsv_bert.cpp:128-155) on synthetic BERT-large-shaped
models (hidden 1024, 16 heads of 64, FFN 4096; fewer layers). The encoder computes in fp32; the
bar here is max |gpu - oracle| <= 2e-4 * max |oracle| per output (the fp bar of the projections
and attention is 2e-3 relative)."""
import numpy as np
import pytest

import bert_oracle as BO
import gsvk
import synth_model as sm
from conftest import FIXTURE_DIR

pytestmark = pytest.mark.gpu

TOL = 2e-4


def _model(tmp_path_factory, wtype, n_layer, layers_used, vocab=1000):
    d = tmp_path_factory.mktemp("bert_" + wtype)
    path, W = sm.write_bert_model(str(d / "bert.gguf"), n_layer=n_layer, layers_used=layers_used, vocab=vocab,
                                  wtype=wtype)
    return gsvk.Bert(path), W


@pytest.fixture(scope="module")
def bert_f32(gpu, tmp_path_factory):
    # (gpu: torch initialises the device first, as in every GPU test of the suite)
    m, W = _model(tmp_path_factory, "f32", 4, 2)
    yield m, W
    m.close()


def _ids(rng, T, vocab=1000):
    return rng.integers(0, vocab, size=T).astype(np.int32)


def _check(got, ref):
    err = np.max(np.abs(got.astype(np.float64) - ref)) / np.max(np.abs(ref))
    assert err <= TOL, err
    return err


@pytest.mark.parametrize("T", [1, 5, 64, 130])
def test_encode_matches_oracle(bert_f32, T):
    m, W = bert_f32
    ids = _ids(np.random.default_rng(T), T)
    got = m.encode([ids])[0]
    assert got.shape == (1024, T)
    _check(got, BO.encode(W, ids, 2, 1024, 16, 1e-12))


def test_every_layer_matches_oracle(bert_f32):
    m, W = bert_f32
    ids = _ids(np.random.default_rng(11), 40)
    for k in range(3):
        _check(m.encode([ids], n_layers=k)[0], BO.encode(W, ids, k, 1024, 16, 1e-12))


def test_batch_matches_one_by_one(bert_f32):
    m, W = bert_f32
    rng = np.random.default_rng(5)
    seqs = [_ids(rng, n) for n in (5, 64, 17, 3)]
    batch = m.encode(seqs, tmax=70)
    for q, got in zip(seqs, batch):
        one = m.encode([q])[0]
        np.testing.assert_allclose(got, one, rtol=0, atol=1e-5 * np.max(np.abs(one)))
        _check(got, BO.encode(W, q, 2, 1024, 16, 1e-12))


def test_longest_sequence_and_limits(bert_f32):
    m, W = bert_f32
    ids = _ids(np.random.default_rng(2), 512)
    _check(m.encode([ids])[0], BO.encode(W, ids, 2, 1024, 16, 1e-12))
    with pytest.raises(gsvk.GsvkError):
        m.encode([_ids(np.random.default_rng(2), 513)])
    with pytest.raises(gsvk.GsvkError):
        m.encode([np.array([1, 1000, 2], np.int32)])    # id == vocab


@pytest.mark.parametrize("wtype,T", [("f16", 33), ("q8_0", 33), ("q8_0", 300)])
def test_quantised_weight_files(gpu, tmp_path_factory, wtype, T):
    """F16 weights: the activations rounded to fp16 before each projection; Q8_0 weights: the
    activations quantised to Q8_0 (x86) and multiplied on the int8 GEMM with exact block sums;
    both as ggml-cpu does, the oracle likewise. 300 tokens take the int8 kernel of more than 256 rows."""
    m, W = _model(tmp_path_factory, wtype, 2, 1)
    try:
        assert m.info["weight_type"] == (1 if wtype == "f16" else 8)
        ids = _ids(np.random.default_rng(7), T)
        got = m.encode([ids])[0].astype(np.float64)
        ref = BO.encode(W, ids, 1, 1024, 16, 1e-12, act_f16=wtype == "f16", act_q8=wtype == "q8_0")
        if wtype == "f16":
            _check(got, ref)
            return
        # Q8_0: the integer block sums are exact, so a token's row agrees with the oracle to fp32
        # rounding, unless a last-bit difference of an activation (fp32 here, float64 there) lands
        # on a rounding boundary of its re-quantisation and moves one int8 value by one step (of
        # amax / 127), which shifts that token's row by ~1e-3 of the scale. Measured at 300
        # tokens: median row 2e-7, 10 rows above 1e-4, the worst 2.0e-3.
        row = np.abs(got - ref).max(axis=0) / np.abs(ref).max()
        assert np.median(row) <= 1e-5, np.median(row)
        assert np.mean(row > 1e-4) <= 0.1, np.mean(row > 1e-4)
        assert row.max() <= 5e-3, row.max()
    finally:
        m.close()


@pytest.mark.parametrize("wtype,lens", [
    ("f32", (96,)), ("f32", (97,)), ("f32", (64, 1, 64)), ("f32", (300, 3, 210)),   # direct / planes, tiles + 1
    ("f16", (512,)), ("f16", (512, 1)), ("f16", (400, 240, 1)),                     # direct / 64-row tiles
    ("f16", (512, 512, 1)), ("f16", (301, 512, 150, 62)),                            # 128-row tiles: 1025 rows
])
def test_tiled_projections(gpu, tmp_path_factory, wtype, lens):
    """The LDS-tiled GEMM at the edges of its tiles and of its dispatch. F32 rows (three bf16 planes)
    also within fp32 rounding: 2e-6 of the scale (measured 3e-7; a product of plain bf16 planes h + m
    would be 2^-17 = 8e-6 off)."""
    m, W = _model(tmp_path_factory, wtype, 2, 1)
    try:
        rng = np.random.default_rng(sum(lens))
        seqs = [_ids(rng, n) for n in lens]
        for q, got in zip(seqs, m.encode(seqs)):
            err = _check(got, BO.encode(W, q, 1, 1024, 16, 1e-12, act_f16=wtype == "f16"))
            if wtype == "f32":
                assert err <= 2e-6, err
    finally:
        m.close()


def _mfma_wgs(lens, heads=16):
    """Workgroups of the matrix-core attention, which is taken above 64 of them."""
    return heads * sum((n + 127) // 128 for n in lens)


# An encoder of one layer whose output is the attention's, so that its error stands alone: every
# projection one power of two per row (exact in fp32 and in three bf16 planes), FFN zero, LayerNorms
# without weights. q = 4 x, k = x turned by one dim of the head, v = x / 4 + b, b = +-2 (values of one
# size, keys weighted unequally), out projection 64: x1 = LN(x + 64 a), output LN(x1).
KQ, KV, KO = 4.0, 0.25, 64.0
K_TURN = np.arange(1024) // 64 * 64 + (np.arange(1024) + 1) % 64
V_BIAS = 2.0 * np.random.default_rng(7).choice([-1.0, 1.0], 1024)


def _attention_model(name, a):
    if ".l0." not in name:
        return a
    a = np.zeros_like(a)
    i = np.arange(1024)
    if name.endswith("qkv_w"):
        a[i, i], a[1024 + i, K_TURN], a[2048 + i, i] = KQ, 1.0, KV
    elif name.endswith("qkv_b"):
        a[2048:] = V_BIAS
    elif name.endswith("attn_out_w"):
        a[i, i] = KO
    elif name.endswith("ln_w"):
        a[:] = 1.0
    return a


def _attention_reference(x, drop=None):
    """The layer on rows x in float64. drop: (which product, "score" or "sum"; the plane pairs left out),
    the operands then as bf16 planes h + m + l."""
    import torch
    one, zero = np.ones(1024), np.zeros(1024)

    def planes(t):
        out = {}
        for p in "hml":
            out[p] = torch.from_numpy(t.astype(np.float32)).bfloat16().double().numpy()
            t = t - out[p]
        return out

    def mul(a, b, what):
        if drop is None or drop[0] != what:
            return a @ b
        pa, pb = planes(a.astype(np.float32).astype(np.float64)), planes(b)
        return sum(pa[e[0]] @ pb[e[1]] for e in ("hh", "hm", "mh", "mm", "hl", "lh") if e not in drop[1])

    v = (KV * x + V_BIAS).astype(np.float32).astype(np.float64)
    a = np.empty_like(x)
    for h in range(16):
        sl = slice(64 * h, 64 * h + 64)
        s = mul(KQ * x[:, sl], x[:, K_TURN[sl]].T, "score") / 8
        p = np.exp(s - s.max(axis=1, keepdims=True))
        a[:, sl] = mul(p, v[:, sl], "sum") / p.sum(axis=1, keepdims=True)
    return BO.layernorm(BO.layernorm(x + KO * a, one, zero, 1e-12), one, zero, 1e-12)


# Of the largest output. fp32: scores up to 16, rounded at 2^-24 of that where they enter the exponent,
# move a weight by 1e-6, of which an output averages several (measured: at most 6.0e-7). A plane product
# left out: 2^-9 x 2^-9 (mm) or 2^-18 (hl, lh) of a product, rounded planes; 1.5e-6 to 5e-6 here.
ATTN_TOL = 1e-6


@pytest.mark.parametrize("lens", [(32, 31, 33, 1, 64), (127, 128, 129, 1), (257, 2, 96, 160), (512, 1), (128, 64, 200, 3),
                                  (32, 31, 1, 2, 30)])   # (96 rows in all: plain rows for the direct-load GEMM)
def test_attention_on_the_matrix_cores(gpu, tmp_path, lens):
    """Key and query tiles with remainders (tiles of 32 keys, 128 queries), at fp32's precision: the
    reference with any one of the six plane products left out misses the bound."""
    assert _mfma_wgs(lens) > 64
    path, _ = sm.write_bert_model(str(tmp_path / "b.gguf"), n_layer=1, layers_used=1, vocab=1000, edit=_attention_model)
    m = gsvk.Bert(path)
    try:
        rng = np.random.default_rng(sum(lens))
        seqs = [_ids(rng, n) for n in lens]
        worst = 0.0
        for x0, got in zip(m.encode(seqs, n_layers=0), m.encode(seqs)):
            x = x0.T.astype(np.float64)
            ref = _attention_reference(x)
            top = np.abs(ref).max()
            worst = max(worst, np.abs(got.T - ref).max() / top)
            if len(x) == 128:
                for what in ("score", "sum"):
                    for e in ("mm", "hl", "lh"):
                        d = np.abs(_attention_reference(x, (what, (e,))) - ref).max() / top
                        assert d > 1.3 * ATTN_TOL, (what, e, d)
        print(f"attention {lens}: {worst:.1e}")
        assert worst <= ATTN_TOL, worst
    finally:
        m.close()


def test_attention_on_the_matrix_cores_q8_0(gpu, tmp_path_factory):
    """A Q8_0 batch: the kernel stores plain fp32 rows, which are then quantised. Against one-by-one
    calls (the other attention kernel): a last-bit difference moves a row where it flips one of its 6144
    quants after the attention, as in test_quantised_weight_files (a flip before it would move every row
    of the sequence, but the rows that enter the attention are quantised alike)."""
    lens = (90, 33, 64, 47, 128)
    assert _mfma_wgs(lens) > 64 and _mfma_wgs(lens[-1:]) <= 64
    m, W = _model(tmp_path_factory, "q8_0", 2, 1)
    try:
        rng = np.random.default_rng(9)
        seqs = [_ids(rng, n) for n in lens]
        rows = []
        for q, got in zip(seqs, m.encode(seqs)):
            one = m.encode([q])[0]
            rows.append(np.abs(got - one).max(axis=0) / np.abs(one).max())
        row = np.concatenate(rows)
        print(f"Q8_0 batch: median row {np.median(row):.1e}, {np.sum(row > 1e-4)} of {len(row)} moved, worst {row.max():.1e}")
        assert np.median(row) <= 1e-5 and np.mean(row > 1e-4) <= 0.1 and row.max() <= 5e-3
    finally:
        m.close()


@pytest.mark.parametrize("lens", [(40,), (96, 104), (300, 301)])   # both direct, F32 tiled, both tiled
@pytest.mark.parametrize("hidden", [512, 1024])
@pytest.mark.parametrize("f16", [("qkv_w", "ff1_w"), ("attn_out_w", "ff2_w")])
def test_layer_of_mixed_projection_types(gpu, tmp_path, f16, hidden, lens):
    """F16 and F32 projections in one layer: each producer writes the operand that its consumer takes."""
    is16 = lambda name: name.endswith(f16)  # noqa: E731
    path, W = sm.write_bert_model(str(tmp_path / "b.gguf"), n_layer=1, layers_used=1, hidden=hidden, heads=hidden // 64,
                                  inter=2048, vocab=1000, wtype=lambda n: "f16" if is16(n) else "f32")
    m = gsvk.Bert(path)
    try:
        rng = np.random.default_rng(hidden + sum(lens))
        seqs = [_ids(rng, n) for n in lens]
        for q, got in zip(seqs, m.encode(seqs)):
            _check(got, BO.encode(W, q, 1, hidden, hidden // 64, 1e-12, act_f16=is16))
    finally:
        m.close()


@pytest.mark.parametrize("wtype,rows", [("f16", (40, 512, 600)), ("f32", (40, 96, 200))])
def test_refused_ffn_width_is_refused_at_every_row_count(gpu, tmp_path, wtype, rows):
    """The direct-load GEMM's loop exists for 1 to 16 groups of steps in powers of two; FFN 1536 (3 or 6
    groups) is refused also where the tiled GEMM takes the rows."""
    path, _ = sm.write_bert_model(str(tmp_path / "b.gguf"), n_layer=1, layers_used=1, hidden=512, heads=8, inter=1536,
                                  vocab=100, wtype=wtype)
    m = gsvk.Bert(path)
    try:
        for n in rows:
            seqs = [np.zeros(min(512, n - i), np.int32) for i in range(0, n, 512)]
            with pytest.raises(gsvk.GsvkError, match="groups per wave"):
                m.encode(seqs)
    finally:
        m.close()


def test_gsv_bert_class_drop_in(bert_f32, tmp_path_factory):
    """The C++ gsv_bert class (include/gsv_bert.h) through every member, driven by
    tests/dropin/gsv_bert_check.cpp (built by oracle/Makefile, target bertcheck)."""
    import os
    import subprocess
    binp = os.path.join(os.path.dirname(os.path.abspath(__file__)), "dropin", "gsv_bert_check")
    if not os.path.exists(binp):
        pytest.skip("tests/dropin/gsv_bert_check was not built")
    m, W = bert_f32
    d = tmp_path_factory.mktemp("bert_class")
    path, _ = sm.write_bert_model(str(d / "b.gguf"), n_layer=4, layers_used=2, vocab=1000)   # same seed
    p = subprocess.run([binp, path], capture_output=True, text=True, timeout=180)
    print(p.stdout, p.stderr)
    assert p.returncode == 0, p.stderr
    out = {l.split()[0]: l.split()[1:] for l in p.stdout.splitlines() if l.strip()}
    assert out["load_cpu_null"] == ["1"] and out["load_missing_null"] == ["1"]
    assert out["info"] == ["1024", "2", "512"]
    s1 = np.array([1, 17, 29, 4, 811, 2], np.int32)
    e = m.encode([s1])[0].astype(np.float64).ravel()
    ref = float(np.sum(e * (np.arange(e.size) % 7 + 1)))
    assert abs(float(out["encode_checksum"][0]) - ref) <= 1e-6 * np.sum(np.abs(e) * 7)
    assert out["feat_ok"] == ["1"]
    assert out["cache"] == ["1", "4", "1"]                         # hits, misses, cached == uncached
    assert out["lru"] == ["2", "1"]                                # recency, not insertion order, evicts
    ok, n1, n2, rel = out["batch"]
    assert ok == "1" and int(n1) == 1024 * 4 and int(n2) == 1024 * 7 and float(rel) <= 1e-5
    assert out["batch_bad_args"] == ["1"]
    assert out["layers"] == ["3", "1"]                             # depths 0..2; the last equals encode
    assert out["too_long_empty"] == ["1"]
    assert "done" in out

"""GPU parity of the prompt forward's f16 activation chain (bitnet_hip_matmul_f16_dev, kernels_gemm.hip k_gemm_f16a<.., EPI = 1>; the
operators it replaces: T:683-691 per-row loop / K/cpu/quantized_matmul.rs:57-96, LayerNorm T:67-100, silu * up T:756-781, residual
T:1073) against the CPU oracle, through the C ABI.

Error model (written in the gates): an activation element is held as f16 (11-bit significand, rounded to nearest: relative error
uniform in +-2^-12, rms 2^-12 / sqrt(3)); weights (code map value x f16 block scale) are exact in f16 and products are exact in the
f32 accumulator, so an output errs by sigma = 2^-12 / sqrt(3) * sqrt(sum_k (w_k x_k)^2) plus f32 accumulation noise.  Gate: 7 sigma per
output (+ 1e-6 * sum |w_k x_k| for the accumulation order) and cosine >= 0.99999 per row (benches/qk256_gemv.rs:234)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LUT_QK = np.array([-2, -1, 1, 2], np.float64)
LUT_T = np.array([0, 1, 0, -1], np.float64)


def cosine(a, b):
    a, b = np.asarray(a, np.float64).ravel(), np.asarray(b, np.float64).ravel()
    return float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-300))


@pytest.fixture(scope="module")
def torch_():
    import torch

    return torch


RAW = {}  # handle -> the packed matrix as the ORACLE takes it (oracle_rows below)


def oracle_rows(oracle, h, xrows):
    """The same matrix through the oracle .so -- gemv_qk256 (Q/i2s_qk256.rs:346) / i2s_matmul_f32 (K/cpu/quantized_matmul.rs:57-96) -- on a few
    activation rows: the dense f64 products this file gates against are built in the test, and would not notice a quirk shared by the test's
    decoding and the kernel's."""
    kind, a, b, rows, cols = RAW[h]
    if kind == "qk256":
        return np.stack([oracle.gemv_qk256(a, r, rows, cols, cols // 256 * 64) for r in xrows]).astype(np.float64)
    return np.stack([oracle.i2s_matmul(r, a, b, 1, rows, cols, 32) for r in xrows]).astype(np.float64)


def make_matrix(hip, rng, fmt, rows, cols):
    """-> (handle, dense f64 matrix [rows, cols])"""
    if fmt == "qk256":
        stride = cols // 256 * 64
        qs = rng.integers(0, 256, rows * stride, dtype=np.uint8)
        pk = qs.reshape(rows, cols // 4)
        codes = np.stack([(pk >> (2 * i)) & 3 for i in range(4)], axis=-1).reshape(rows, cols)
        h = hip.weights_upload_qk256(qs, rows, cols, stride)
        RAW[h] = ("qk256", qs, None, rows, cols)
        return h, LUT_QK[codes]
    codes = rng.choice(np.array([0, 1, 3], np.uint8), size=(rows, cols), p=[0.5, 0.25, 0.25])
    packed = (codes[:, 0::4] | codes[:, 1::4] << 2 | codes[:, 2::4] << 4 | codes[:, 3::4] << 6).astype(np.uint8)
    scales = (1.0 / ((np.arange(rows * (cols // 32)) % 100) + 1)).astype(np.float16).astype(np.float32)
    dense = LUT_T[codes] * np.repeat(scales.reshape(rows, cols // 32).astype(np.float64), 32, axis=1)
    h = hip.weights_upload_i2s(packed.reshape(-1), scales, rows, cols, 32)
    RAW[h] = ("i2s", packed.reshape(-1), scales, rows, cols)
    return h, dense


def gate(got, want, w, xa):
    """7 sigma of the f16 rounding of the activations + f32 accumulation slack; cosine per row"""
    sigma = 2.0 ** -12 / np.sqrt(3.0) * np.sqrt((xa.astype(np.float64) ** 2) @ (w ** 2).T)
    slack = 1e-6 * (np.abs(xa).astype(np.float64) @ np.abs(w).T) + 1e-7
    bad = np.abs(got - want) > 7.0 * sigma + slack
    assert not bad.any(), float(np.max(np.abs(got - want) / (7.0 * sigma + slack)))
    for i in range(got.shape[0]):
        assert cosine(got[i], want[i]) >= 0.99999, i


@pytest.mark.parametrize("fmt", ["qk256", "i2s"])
@pytest.mark.parametrize("rows,cols,m", [(256, 256, 1), (512, 2560, 100), (2560, 768, 64), (768, 6912, 300), (2560, 768, 4000)])
def test_f16_chain_plain_residual_and_handover(hip, oracle, torch_, fmt, rows, cols, m):
    """y = residual + W xh (in place), the f16 copy f16(gamma_out * y) and the LayerNorm partials the next projection reads"""
    rng = np.random.default_rng(rows + cols + m)
    h, w = make_matrix(hip, rng, fmt, rows, cols)
    assert hip.matmul_f16_supported(h)
    mp = -(-m // 64) * 64
    x = (rng.normal(0, 1, (m, cols)) * np.exp(rng.uniform(-2, 2, (m, 1)))).astype(np.float32)
    res = rng.normal(0, 1, (m, rows)).astype(np.float32)
    gout = rng.uniform(0.5, 1.5, rows).astype(np.float32)
    xh = torch_.zeros(mp, cols, dtype=torch_.float16, device="cuda")
    hip.rows_to_f16_dev(torch_.from_numpy(x).cuda(), None, m, cols, xh, None)
    torch_.cuda.synchronize()
    x16 = x.astype(np.float16)
    assert np.array_equal(xh[:m].cpu().numpy(), x16)  # round to nearest even, as numpy
    y = torch_.from_numpy(res).cuda()
    yh = torch_.full((mp, rows), float("nan"), dtype=torch_.float16, device="cuda")
    st = torch_.full((rows // 64, mp, 2), float("nan"), device="cuda")
    hip.matmul_f16_dev(h, xh, m, y=y, residual=y, yh=yh, gamma_out=torch_.from_numpy(gout).cuda(), stats_out=st)
    torch_.cuda.synchronize()
    got = y.cpu().numpy()
    want = res.astype(np.float64) + x16.astype(np.float64) @ w.T
    assert np.isfinite(got).all()
    # the activations ARE f16 values here (xh is the input): only accumulation order separates the kernel from the f64 product
    assert np.max(np.abs(got - want) / (np.abs(x16).astype(np.float64) @ np.abs(w).T + np.abs(res) + 1e-6)) <= 2e-6
    # ... and the oracle's own loop on the same f16-valued rows (f32, left to right: its accumulation error is the larger of the two)
    pick = np.unique(np.r_[0, m - 1, rng.integers(0, m, 3)])
    oref = oracle_rows(oracle, h, x16[pick].astype(np.float32))
    mag = np.abs(x16[pick]).astype(np.float64) @ np.abs(w).T + 1e-6
    assert np.max(np.abs(got[pick] - res[pick] - oref) / mag) <= 3e-5, float(np.max(np.abs(got[pick] - res[pick] - oref) / mag))
    # hand-over: the f16 copy is the f32 output times gamma_out, rounded once; partials are the 64-row slab sums of the f32 output
    assert np.array_equal(yh[:m].cpu().numpy(), (got * gout).astype(np.float16))
    stn = st.cpu().numpy()[:, :m, :]
    wr = hip.matmul_last_wave_rows()  # 64, or 80 in the 320-row workgroups a long 2560-row launch takes (4000 tokens: 504 workgroups, one round)
    assert wr == (80 if (rows, m) == (2560, 4000) else 64)
    if wr == 80:
        assert np.all(stn[rows // 80 :] == 0)  # the surplus entries of the [rows / 64] array are written as zero
        stn = stn[: rows // 80]
    slabs = got.reshape(m, rows // wr, wr).astype(np.float64)
    # (f32 sums of 64 terms in the kernel: 2^-24 relative per addition, against the sum of the magnitudes)
    assert np.all(np.abs(stn[:, :, 0].T - slabs.sum(axis=2)) <= 4e-6 * np.abs(slabs).sum(axis=2) + 1e-6)
    assert np.all(np.abs(stn[:, :, 1].T - (slabs ** 2).sum(axis=2)) <= 4e-6 * (slabs ** 2).sum(axis=2) + 1e-6)
    if mp > m:
        assert np.all(st.cpu().numpy()[:, m:, :] == 0)  # padding tokens: zero partials
    hip.weights_free(h)


@pytest.mark.parametrize("fmt", ["qk256", "i2s"])
@pytest.mark.parametrize("m", [17, 511, 800, 1025])
def test_f16_chain_half_slab_waves(hip, torch_, fmt, m):
    """2560 rows around the lines of the short-prompt forms: 32-row waves of 16 tokens (17; 511: 320 workgroups if they had 256 rows) and of 32 (800: 260), 64-row waves (1025: 340)"""
    rows, cols, mp = 2560, 512, -(-m // 64) * 64
    rng = np.random.default_rng(m)
    h, w = make_matrix(hip, rng, fmt, rows, cols)
    x = rng.normal(0, 1, (mp, cols)).astype(np.float16)
    res = rng.normal(0, 1, (m, rows)).astype(np.float32)
    y, st = torch_.from_numpy(res).cuda(), torch_.full((rows // 64, mp, 2), float("nan"), device="cuda")
    hip.matmul_f16_dev(h, torch_.from_numpy(x).cuda(), m, y=y, residual=y, stats_out=st)
    assert (hip.matmul_last_workgroup_rows(), hip.matmul_last_tile()["wave_tokens"]) == {17: (128, 16), 511: (128, 16), 800: (128, 32), 1025: (256, 32)}[m]
    torch_.cuda.synchronize()
    got, xd = y.cpu().numpy().astype(np.float64), x[:m].astype(np.float64)
    assert np.max(np.abs(got - (res + xd @ w.T)) / (np.abs(xd) @ np.abs(w).T + np.abs(res) + 1e-6)) <= 2e-6  # f16 inputs: accumulation order alone
    slabs, s = got.reshape(m, rows // 64, 64), st.cpu().numpy()
    for e in (1, 2):  # f32 sums of 64 terms: 2^-24 per addition against the magnitudes
        assert np.all(np.abs(s[:, :m, e - 1].T - (slabs ** e).sum(axis=2)) <= 4e-6 * (np.abs(slabs) ** e).sum(axis=2) + 1e-6)
    assert np.all(s[:, m:] == 0)
    hip.weights_free(h)


@pytest.mark.parametrize("fmt,m,tile", [("qk256", 65, (128, 16)), ("i2s", 65, (128, 16)), ("qk256", 833, (128, 16)), ("i2s", 833, (128, 32)), ("qk256", 1281, (256, 32)), ("i2s", 1281, (256, 32))])
def test_f16_chain_no_tile_past_the_last_token(hip, torch_, fmt, m, tile):
    """Tiles chosen by their measured cost; token counts that end in a tile ahead of the padding's end, grids that are no multiple of eight workgroups: every live value is written, the
    partials of the padding that no workgroup computes are zero, and nothing behind the last token's row is touched"""
    rows, cols, mp = 2560, 1024, -(-m // 64) * 64
    rng = np.random.default_rng(m)
    h, w = make_matrix(hip, rng, fmt, rows, cols)
    x = rng.normal(0, 1, (mp, cols)).astype(np.float16)
    res = rng.normal(0, 1, (m, rows)).astype(np.float32)
    y, st = torch_.full((mp, rows), 7.0, device="cuda"), torch_.full((rows // 64, mp, 2), float("nan"), device="cuda")
    y[:m] = torch_.from_numpy(res).cuda()
    hip.matmul_f16_dev(h, torch_.from_numpy(x).cuda(), m, y=y, residual=y, stats_out=st)
    assert (hip.matmul_last_workgroup_rows(), hip.matmul_last_tile()["wave_tokens"]) == tile
    torch_.cuda.synchronize()
    out, xd = y.cpu().numpy().astype(np.float64), x[:m].astype(np.float64)
    got = out[:m]
    assert np.max(np.abs(got - (res + xd @ w.T)) / (np.abs(xd) @ np.abs(w).T + np.abs(res) + 1e-6)) <= 2e-6  # f16 inputs: accumulation order alone
    assert np.all(out[m:] == 7.0)
    slabs, s = got.reshape(m, rows // 64, 64), st.cpu().numpy()
    for e in (1, 2):  # f32 sums of 64 terms: 2^-24 per addition against the magnitudes
        assert np.all(np.abs(s[:, :m, e - 1].T - (slabs ** e).sum(axis=2)) <= 4e-6 * (np.abs(slabs) ** e).sum(axis=2) + 1e-6)
    assert np.all(s[:, m:] == 0)
    hip.weights_free(h)


@pytest.mark.parametrize("fmt", ["qk256", "i2s"])
def test_f16_chain_layernorm_after_product_and_silu(hip, oracle, torch_, fmt):
    """qkv-like (LayerNorm -> f32 rows) and gate|up-like (LayerNorm -> silu(gate) * up -> f16 rows) launches at the 2B-4T widths,
    LayerNorm statistics from one partial (the chain's entry) and from 40 (a producer's slabs), against the oracle's LayerNorm + product"""
    rng = np.random.default_rng(11)
    K, N, m = 2560, 512, 96
    mp = -(-m // 64) * 64
    ha, wa = make_matrix(hip, rng, fmt, N, K)
    hb, wb = make_matrix(hip, rng, fmt, N, K)
    x = rng.normal(0.15, 1.0, (m, K)).astype(np.float32)
    g = (rng.uniform(0.5, 1.5, K) / (80 if fmt == "qk256" else 4)).astype(np.float32)
    gd = torch_.from_numpy(g).cuda()
    xn = np.stack([oracle.layernorm(x[i], g, 1e-5) for i in range(m)]).astype(np.float64)
    ya, yb = xn @ wa.T, xn @ wb.T
    xd = torch_.from_numpy(x).cuda()
    xh = torch_.zeros(mp, K, dtype=torch_.float16, device="cuda")
    st1 = torch_.zeros(1, mp, 2, device="cuda")
    hip.rows_to_f16_dev(xd, gd, m, K, xh, st1)
    # the same statistics as 40 slab partials (what an o- / down-projection leaves)
    st40 = torch_.zeros(40, mp, 2, device="cuda")
    sl = x.reshape(m, 40, 64).astype(np.float64)
    st40[:, :m, 0] = torch_.from_numpy(sl.sum(axis=2).T.astype(np.float32)).cuda()
    st40[:, :m, 1] = torch_.from_numpy((sl ** 2).sum(axis=2).T.astype(np.float32)).cuda()
    hc = hip.weights_concat([ha, hb])
    hip.weights_bind_ln(hc, gd)
    xg = (x * g).astype(np.float64)  # what the f16 rounding acts on: sigma is taken over gamma * x, the mean term is exact
    wcat = np.concatenate([wa, wb], axis=0)
    for st, n_st in ((st1, 1), (st40, 40)):
        y = torch_.full((m, 2 * N), float("nan"), device="cuda")
        hip.matmul_f16_dev(hc, xh, m, stats_in=st, n_stats=n_st, ln_gamma=gd, ln_eps=1e-5, y=y)
        torch_.cuda.synchronize()
        got = y.cpu().numpy()
        denom = np.sqrt(x.astype(np.float64).var(axis=1, keepdims=True) + 1e-5)
        sigma = 2.0 ** -12 / np.sqrt(3.0) * np.sqrt((xg ** 2) @ (wcat ** 2).T) / denom
        want = np.concatenate([ya, yb], axis=1)
        slack = 2e-6 * (np.abs(xg) @ np.abs(wcat).T) / denom + 1e-6
        assert np.all(np.abs(got - want) <= 7.0 * sigma + slack), (n_st, float(np.max(np.abs(got - want) / (7.0 * sigma + slack))))
        for i in range(m):
            assert cosine(got[i], want[i]) >= 0.99999
    hg = hip.weights_concat([ha, hb], interleave16=True)
    hip.weights_bind_ln(hg, gd)
    hh = torch_.full((mp, N), float("nan"), dtype=torch_.float16, device="cuda")
    yf = torch_.full((m, N), float("nan"), device="cuda")
    hip.matmul_f16_dev(hg, xh, m, stats_in=st40, n_stats=40, ln_gamma=gd, ln_eps=1e-5, y=yf, flags=1, yh=hh)
    torch_.cuda.synchronize()
    want = ya / (1 + np.exp(-ya)) * yb
    got = yf.cpu().numpy()
    assert np.max(np.abs(got - want)) <= 2e-3 * np.max(np.abs(want))
    for i in range(m):
        assert cosine(got[i], want[i]) >= 0.99999
    assert np.array_equal(hh[:m].cpu().numpy(), got.astype(np.float16))
    with pytest.raises(Exception, match="bound gamma"):
        hip.matmul_f16_dev(hc, xh, m, stats_in=st1, n_stats=1, ln_gamma=torch_.from_numpy(g.copy()).cuda(), ln_eps=1e-5, y=yf)
    for h in (ha, hb, hc, hg):
        hip.weights_free(h)


def test_f16_chain_refuses_what_it_cannot_take(hip, torch_):
    rng = np.random.default_rng(3)
    n, k = 100, 512  # rows % 256 != 0
    qs = rng.integers(0, 256, n * (k // 256) * 64, dtype=np.uint8)
    h = hip.weights_upload_qk256(qs, n, k, k // 256 * 64)
    assert not hip.matmul_f16_supported(h)
    xh = torch_.zeros(64, k, dtype=torch_.float16, device="cuda")
    y = torch_.zeros(10, n, device="cuda")
    with pytest.raises(Exception, match="does not take the f16 chain"):
        hip.matmul_f16_dev(h, xh, 10, y=y)
    hip.weights_free(h)


def test_f16_hand_over_saturation_is_counted_and_the_decoder_falls_back(pkg, hip, oracle, torch_):
    """the f16 chain stores f16(gamma * x) with no row scale and clamped silently at +-65504.  Now every writer COUNTS a clamp
    (bitnet_hip_f16_saturations) and Decoder::prefill repeats a prompt that clamped anything on the 4-digit planes (30-bit fixed point behind a
    per-row power-of-two scale) before it takes the logits.  Op level: an in-range call leaves the counter at zero, an outlier channel raises it.
    Decoder level: a BitNet32-F16 model whose LAST feed-forward LayerNorm weight has one channel at 2e5 (gamma * x far beyond the f16 range on
    every token, and silu * up beyond it by orders of magnitude; the attention inputs stay in range -- the prompt attention multiplies f16
    operands whatever the projections do): the chain's result would be wrong; the decoder reports one fallback and matches the oracle."""
    import importlib

    synth = importlib.import_module("bitnet-rs_amd.synth")
    rng = np.random.default_rng(5)
    m, cols = 200, 512
    x = rng.normal(0.0, 1.0, (m, cols)).astype(np.float32)
    g = rng.uniform(0.5, 1.5, cols).astype(np.float32)
    xh = torch_.zeros(256, cols, dtype=torch_.float16, device="cuda")
    st = torch_.zeros(2 * 256, device="cuda")
    hip.f16_saturations(True)
    hip.rows_to_f16_dev(torch_.from_numpy(x).cuda(), torch_.from_numpy(g).cuda(), m, cols, xh, st)
    assert hip.f16_saturations(True) == 0
    g2 = g.copy()
    g2[17] = 3e5
    hip.rows_to_f16_dev(torch_.from_numpy(x).cuda(), torch_.from_numpy(g2).cuda(), m, cols, xh, st)
    n = hip.f16_saturations(True)
    assert 0 < n <= m and hip.f16_saturations(False) == 0  # one lane per row whose element 17 left the range; reading resets
    assert np.all(np.abs(xh.cpu().numpy()[:m, 17][np.abs(x[:, 17] * 3e5) > 65504]) == 65504.0)
    # ---- decoder level
    cfg = synth.ModelConfig(hidden=512, n_layers=2, n_heads=4, n_kv_heads=2, head_dim=128, ffn=1024, vocab=2048, max_pos=320, eps=1e-5, rope_theta=10000.0)
    glob = synth.make_globals(cfg)
    layers = [synth.make_layer(cfg, l, fmt="i2s", block=32) for l in range(cfg.n_layers)]
    layers[-1]["ffn_norm"] = layers[-1]["ffn_norm"].copy()
    layers[-1]["ffn_norm"][33] = 2e5
    om = oracle.OracleModel(cfg, [dict(w, ternary=32) for w in layers], glob, n_threads=8)
    T = 256
    prompt = synth.prompt(T, cfg.vocab)
    want = None
    for t in prompt:
        _, want, _ = om.step(int(t), want_logits=True)
    om.close()
    dec = pkg.HostDecoder(cfg)
    for l, w in enumerate(layers):
        dec.set_layer_i2s(l, w, 32)
    dec.set_globals(glob)
    dec.reset()
    dec.feed(prompt)
    dec.prefill(T, with_logits=True, digits=2)
    assert dec.saturation_fallbacks() == 1 and dec.last_prefill_path() == 0
    got = dec.last_logits().astype(np.float64)
    c = float(got @ want / (np.linalg.norm(got) * np.linalg.norm(want)))
    assert c >= 0.9999, c
    assert int(dec.history(T + 1)[T]) == oracle.argmax(want)
    dec.close()


def test_clamps_seen_by_one_sequence_are_not_taken_from_another(hip, torch_):
    """The running total on one stream, takers that clear the count on others: each taker gets what came since the last, the total misses nothing."""
    import ctypes as C

    streams = [torch_.cuda.Stream() for _ in range(3)]
    m, cols = 64, 512
    x, g = torch_.full((m, cols), 1e5, device="cuda"), torch_.ones(cols, device="cuda")
    xh, out = torch_.zeros(m, cols, dtype=torch_.float16, device="cuda"), torch_.full((8,), 77, dtype=torch_.int32).pin_memory()
    P = lambda i: C.c_void_p(out.data_ptr() + 4 * i)
    S = lambda i: C.c_void_p(streams[i].cuda_stream)
    torch_.cuda.synchronize()
    hip.f16_saturations(True)
    hip._call("f16_saturations_total_dev", P(0), S(0))
    for i in (1, 2):
        with torch_.cuda.stream(streams[i]):
            hip.rows_to_f16_dev(x, g, m, cols, xh, None, stream=streams[i].cuda_stream)
        hip._call("f16_saturations_dev", P(i), S(i))
        torch_.cuda.synchronize()
    hip._call("f16_saturations_dev", None, S(0))
    hip._call("f16_saturations_total_dev", P(3), S(0))
    torch_.cuda.synchronize()
    before, a, b, after = out[:4].tolist()
    lanes = m * cols // 4
    assert (a, b) == (lanes, lanes) and (after - before) % 2 ** 32 == 2 * lanes
    assert hip.f16_saturations(True) == 0
    hip.rows_to_f16_dev(x, g, m, cols, xh, None)
    assert hip.f16_saturations(False) == lanes and hip.f16_saturations(True) == lanes and hip.f16_saturations(True) == 0
    with pytest.raises(Exception, match="Null pointer"):
        hip._call("f16_saturations_total_dev", None, S(0))


_F16H_HASH_SCRIPT = r"""
import hashlib, importlib, sys
import numpy as np, torch
sys.path.insert(0, {root!r})
sys.path.insert(0, {root!r} + "/tests")
pkg = importlib.import_module("bitnet-rs_amd"); synth = importlib.import_module("bitnet-rs_amd.synth")
hip = pkg.load(); hip.init(0)
import test_f16_chain as T
print("HASH", T.f16h_case(hip, torch, {fmt!r}, {kind!r})[0])
"""


def f16h_case(hip, torch_, fmt, kind):
    """The wide chain launches of a 4096-token prompt at the 2B-4T widths: kind 'gateup' (13824 x 2560, LayerNorm after the product, silu * up -> f16
    rows) or 'qkv' (3840 x 2560, LayerNorm -> f32 rows).  -> (sha256 of the output bytes, outputs, the pieces a checker needs)."""
    import hashlib

    rng = np.random.default_rng(123)
    K, m = 2560, 4096
    N = 6912 if kind == "gateup" else 1920
    ha, wa = make_matrix(hip, rng, fmt, N, K)
    hb, wb = make_matrix(hip, rng, fmt, N, K)
    x = rng.normal(0.15, 1.0, (m, K)).astype(np.float32)
    g = (rng.uniform(0.5, 1.5, K) / (80 if fmt == "qk256" else 4)).astype(np.float32)
    gd = torch_.from_numpy(g).cuda()
    xh = torch_.zeros(m, K, dtype=torch_.float16, device="cuda")
    st = torch_.zeros(1, m, 2, device="cuda")
    hip.rows_to_f16_dev(torch_.from_numpy(x).cuda(), gd, m, K, xh, st)
    h = hip.weights_concat([ha, hb], interleave16=(kind == "gateup"))
    hip.weights_bind_ln(h, gd)
    if kind == "gateup":
        out = torch_.full((m, N), float("nan"), dtype=torch_.float16, device="cuda")
        hip.matmul_f16_dev(h, xh, m, stats_in=st, n_stats=1, ln_gamma=gd, ln_eps=1e-5, flags=1, yh=out)
    else:
        out = torch_.full((m, 2 * N), float("nan"), device="cuda")
        hip.matmul_f16_dev(h, xh, m, stats_in=st, n_stats=1, ln_gamma=gd, ln_eps=1e-5, y=out)
    torch_.cuda.synchronize()
    tile = dict(hip.matmul_last_tile())
    o = out.cpu().numpy()
    for hh in (ha, hb, h):
        hip.weights_free(hh)
    return hashlib.sha256(o.tobytes()).hexdigest(), o, (x, g, wa, wb, tile)


@pytest.mark.parametrize("fmt", ["i2s", "qk256"])
@pytest.mark.parametrize("kind", ["gateup", "qkv"])
def test_f16h_wide_tile_instances_match_oracle_and_the_64_token_kernel(hip, oracle, torch_, fmt, kind):
    """k_gemm_f16h (round 5): the 64-row x 128-token wave tile the f16 chain's wide launches take at 4096 tokens -- gate|up split 48 + 6 row blocks
    (the six on k_gemm_f16a), q|k|v whole (480 workgroups: one round).  Tile asserted; sampled rows against the oracle's LayerNorm + product
    (+ silu * up); and the WHOLE output bit-identical to the launch with BITNET_HIP_GEMM_F16H=0 (k_gemm_f16a alone: same k-order, same f32
    accumulation per output element) -- the switch is read once per process, hence the child process."""
    import os
    import subprocess
    import sys

    h1, out, (x, g, wa, wb, tile) = f16h_case(hip, torch_, fmt, kind)
    assert tile["wave_tokens"] == 128 and tile["digits"] == 2 and tile["scale_mode"] == (4 if fmt == "i2s" else 5), tile
    assert np.isfinite(out.astype(np.float64)).all()
    rng = np.random.default_rng(9)
    for i in np.unique(np.r_[0, 4095, rng.integers(0, 4096, 6)]):
        xn = oracle.layernorm(x[i], g, 1e-5).astype(np.float64)
        a, b = xn @ wa.T, xn @ wb.T
        want = a / (1 + np.exp(-a)) * b if kind == "gateup" else np.concatenate([a, b])
        got = out[i].astype(np.float64)
        assert cosine(got, want) >= 0.99999, int(i)
        assert np.max(np.abs(got - want)) <= 2.5e-3 * np.max(np.abs(want)), int(i)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-c", _F16H_HASH_SCRIPT.format(root=root, fmt=fmt, kind=kind)], env=dict(os.environ, BITNET_HIP_GEMM_F16H="0"),
                       capture_output=True, text=True, timeout=600)
    assert p.returncode == 0, p.stdout[-1500:] + p.stderr[-3000:]
    h0 = [l.split()[1] for l in p.stdout.splitlines() if l.startswith("HASH ")][0]
    assert h0 == h1, "k_gemm_f16h's outputs differ from k_gemm_f16a's"


# rows x cols x tokens: every form of the launch -- 128-row workgroups of 16 and 32 tokens, 256-row ones of 16, 32 and 64, 320-row ones, 128-token wave tiles whole and beside the others
@pytest.mark.parametrize("fmt", ["qk256", "i2s"])
@pytest.mark.parametrize("rows,cols,m,silu", [(256, 256, 1, 0), (2560, 512, 17, 0), (2560, 768, 300, 0), (5376, 256, 200, 0), (13824, 256, 130, 1), (10240, 512, 513, 1), (2560, 256, 4000, 0),
                                              (3840, 512, 4096, 0), (13824, 256, 2048, 1)])
def test_chain_on_the_image_is_the_expanding_one_bit_for_bit(hip, torch_, fmt, rows, cols, m, silu):
    """A captured launch builds no image and expands the codes in its K loop; the first eager one builds it and reads its operands from there: the same values, the same order of sums."""
    rng = np.random.default_rng(rows + cols + m)
    parts = [make_matrix(hip, rng, fmt, rows // 2, cols)[0] for _ in range(2)]
    h = hip.weights_concat(parts, interleave16=bool(silu))
    mp, out = -(-m // 64) * 64, rows // 2 if silu else rows
    xh = torch_.from_numpy(rng.normal(0, 1, (mp, cols)).astype(np.float16)).cuda()
    flags = 1 if silu else 0

    def buffers():
        return (None if silu else torch_.full((m, out), 7.0, device="cuda")), torch_.full((mp, out), 7.0, dtype=torch_.float16, device="cuda")

    def launch(b, stream):
        hip.matmul_f16_dev(h, xh, m, y=b[0], yh=b[1], flags=flags, stream=stream)

    expanded, image, b0 = buffers(), buffers(), hip.weights_device_bytes(h)
    torch_.cuda.synchronize()
    graph, s = torch_.cuda.CUDAGraph(), torch_.cuda.Stream()
    with torch_.cuda.graph(graph, stream=s):
        launch(expanded, s.cuda_stream)
    assert hip.weights_device_bytes(h) == b0
    graph.replay()
    torch_.cuda.synchronize()
    launch(image, torch_.cuda.current_stream().cuda_stream)
    torch_.cuda.synchronize()
    assert hip.weights_device_bytes(h) == b0 + rows // 16 * (cols // 256) * 2048
    for a, b in zip(expanded, image):
        assert a is None or (torch_.isfinite(a).all() and torch_.equal(a, b))
    hip.weights_fp4_image(h, False)  # given back, and built again where it is wanted again
    assert hip.weights_device_bytes(h) == b0
    again = buffers()
    launch(again, torch_.cuda.current_stream().cuda_stream)
    torch_.cuda.synchronize()
    assert hip.weights_device_bytes(h) == b0 + rows // 16 * (cols // 256) * 2048
    assert all(a is None or torch_.equal(a, b) for a, b in zip(again, image))
    for w in (h, *parts):
        hip.weights_free(w)


def test_tiles_with_and_without_the_image(hip, torch_):
    """A tile that is a little shorter with the image only is not taken where the codes are expanded: the same values and the same statistics, bit for bit"""
    rows, cols, m = 2304, 1024, 897
    rng, mp = np.random.default_rng(7), -(-m // 64) * 64
    h, _ = make_matrix(hip, rng, "qk256", rows, cols)
    xh = torch_.from_numpy(rng.normal(0, 1, (mp, cols)).astype(np.float16)).cuda()
    outs = [(torch_.full((m, rows), 7.0, device="cuda"), torch_.full((rows // 64, mp, 2), float("nan"), device="cuda")) for _ in range(2)]
    torch_.cuda.synchronize()
    graph, s = torch_.cuda.CUDAGraph(), torch_.cuda.Stream()
    with torch_.cuda.graph(graph, stream=s):
        hip.matmul_f16_dev(h, xh, m, y=outs[0][0], stats_out=outs[0][1], stream=s.cuda_stream)
    assert hip.matmul_last_tile()["wave_tokens"] == 32
    graph.replay()
    torch_.cuda.synchronize()
    hip.matmul_f16_dev(h, xh, m, y=outs[1][0], stats_out=outs[1][1])
    assert hip.matmul_last_tile()["wave_tokens"] == 16
    torch_.cuda.synchronize()
    assert torch_.equal(outs[0][0], outs[1][0]) and torch_.equal(outs[0][1], outs[1][1])
    hip.weights_free(h)


@pytest.mark.parametrize("fmt", ["qk256", "i2s"])
@pytest.mark.parametrize("silu", [0, 1])
def test_concatenation_of_parts_that_have_images(hip, torch_, fmt, silu):
    """The images belong to the part: the fused matrix starts without one, builds its own, and either may be freed first."""
    rows, cols, m = 256, 512, 64
    rng = np.random.default_rng(silu)
    parts = [make_matrix(hip, rng, fmt, rows, cols)[0] for _ in range(2)]
    xh = torch_.from_numpy(rng.normal(0, 1, (m, cols)).astype(np.float16)).cuda()
    plain, fresh = hip.weights_device_bytes(parts[0]), hip.weights_concat(parts, interleave16=bool(silu))

    def product(h, n):
        y = torch_.full((m, n), 7.0, dtype=torch_.float16, device="cuda")
        hip.matmul_f16_dev(h, xh, m, yh=y, flags=0)
        torch_.cuda.synchronize()
        return y

    before = product(parts[0], rows)
    if fmt == "qk256":
        hip.weights_fp4_image(parts[0], True)
    image = rows // 16 * (cols // 256) * 2048
    assert hip.weights_device_bytes(parts[0]) == plain + image * (2 if fmt == "qk256" else 1)
    h = hip.weights_concat(parts, interleave16=bool(silu))
    assert hip.weights_device_bytes(h) == 2 * plain
    want = product(fresh, 2 * rows)
    assert torch_.equal(product(h, 2 * rows), want) and hip.weights_device_bytes(h) == 2 * plain + 2 * image
    hip.weights_free(h)
    assert torch_.equal(product(parts[0], rows), before)
    hip.weights_free(parts[0])
    assert torch_.equal(product(fresh, 2 * rows), want)
    for w in (fresh, parts[1]):
        hip.weights_free(w)


FEW_ROWS = 128


# the last number of tokens that takes the form: one round of workgroups, their number past it (longer rows: more), and the token rows within an XCD's L2
@pytest.mark.parametrize("rows,cols,silu,last", [(2560, 2560, 0, 144), (3840, 2560, 0, 96), (2560, 6912, 0, 192), (13824, 2560, 1, 16), (1024, 512, 0, 256), (256, 2048, 0, 1024), (1024, 8192, 0, 256),
                                                 (1024, 512, 1, 256), (4096, 2048, 1, 64), (512, 4096, 0, 512), (1024, 1024, 0, 352),
                                                 (1536, 6912, 0, (240, 303)), (1536, 8192, 0, (240, 256))])
def test_f16_few_rows_only_where_they_are_faster(hip, rows, cols, silu, last):
    rng = np.random.default_rng(rows)
    for fmt, last in zip(("qk256", "i2s"), last if isinstance(last, tuple) else (last, last)):  # (block scales: the wide tiles cost more)
        parts = [make_matrix(hip, rng, fmt, rows // 2, cols)[0] for _ in range(2)]
        h = hip.weights_concat(parts, interleave16=bool(silu))
        assert [hip.matmul_f16_takes_few_rows(h, m, silu) for m in (1, last - 1, last, last + 1, 2 * last, 4096)] == [True, True, True, False, False, False]
        for w in (h, *parts):
            hip.weights_free(w)


# rows x cols x tokens: one, two and four row tiles per workgroup, one block of K (waves without work) to 27, whole and ragged token tiles, pairs
@pytest.mark.parametrize("fmt", ["qk256", "i2s"])
@pytest.mark.parametrize("rows,cols,m,silu,tile", [(256, 256, 1, 0, 16), (2560, 2560, 16, 0, 16), (2560, 768, 17, 0, 32), (2560, 6912, 100, 0, 32), (3840, 2304, 64, 0, 64), (13824, 512, 16, 1, 64),
                                                   (512, 2560, 5, 1, 32), (2560, 1024, 1, 0, 16)])
def test_f16_chain_few_rows(hip, torch_, fmt, rows, cols, m, silu, tile):
    """The form for few rows behind a LayerNorm (partials of 16 and of 64 columns, and one), its residual, f16 copy and partials of 16 rows, against float64."""
    rng = np.random.default_rng(rows + cols + m)
    parts = [make_matrix(hip, rng, fmt, rows // 2, cols) for _ in range(2)]
    h, mp, out = hip.weights_concat([a for a, _ in parts], interleave16=bool(silu)), -(-m // 64) * 64, rows // 2 if silu else rows
    gamma, eps = rng.uniform(0.5, 1.5, cols).astype(np.float32), 1e-5
    gd = torch_.from_numpy(gamma).cuda()
    hip.weights_bind_ln(h, gd)
    x = (rng.normal(0, 1, (m, cols)) * np.exp(rng.uniform(-1, 1, (m, 1))) + 0.3).astype(np.float32)
    xh = torch_.zeros(mp, cols, dtype=torch_.float16, device="cuda")
    xh[:m] = torch_.from_numpy((x * gamma).astype(np.float16)).cuda()
    flags = (1 if silu else 0) | FEW_ROWS
    assert hip.matmul_f16_takes_few_rows(h, m, flags)
    w = np.concatenate([d for _, d in parts])
    xd, x16 = x.astype(np.float64), (x * gamma).astype(np.float16).astype(np.float64)
    mean, denom = xd.mean(1, keepdims=True), np.sqrt(xd.var(1, keepdims=True) + eps)
    g64 = w @ gamma.astype(np.float64)
    plain = (x16 @ w.T - mean * g64) / denom  # f16 inputs are given: accumulation order, and the f32 of mean * g
    mag = (np.abs(x16) @ np.abs(w).T + np.abs(mean) * np.abs(g64)) / denom + 1e-6
    res, gout = rng.normal(0, 1, (m, rows)).astype(np.float32), rng.uniform(0.5, 1.5, rows).astype(np.float32)
    for part in (16, 64, cols):
        n = cols // part
        st = torch_.zeros(n, mp, 2, device="cuda")
        sums = xd.reshape(m, n, part)
        st[:, :m] = torch_.from_numpy(np.stack([sums.sum(2).T, (sums ** 2).sum(2).T], 2).astype(np.float32)).cuda()
        yh = torch_.full((mp, out), 7.0, dtype=torch_.float16, device="cuda")
        so = torch_.full((rows // 16, mp, 2), 7.0, device="cuda")
        if silu:
            hip.matmul_f16_dev(h, xh, m, stats_in=st, n_stats=n, ln_gamma=gd, ln_eps=eps, flags=flags, yh=yh)
        else:
            y = torch_.from_numpy(res).cuda()
            hip.matmul_f16_dev(h, xh, m, stats_in=st, n_stats=n, ln_gamma=gd, ln_eps=eps, y=y, residual=y, flags=flags, yh=yh, gamma_out=torch_.from_numpy(gout).cuda(), stats_out=so)
        torch_.cuda.synchronize()
        assert hip.matmul_last_workgroup_rows() == tile and hip.matmul_last_tile()["wave_tokens"] == 16
        if silu:
            a, b = plain[:, :out], plain[:, out:]
            want = a / (1 + np.exp(-a)) * b
            # the product's 4e-6 through silu * up (slope at most 1.1), and the result's f16
            assert np.all(np.abs(yh[:m].cpu().numpy() - want) <= 1.1 * 4e-6 * (mag[:, :out] * np.abs(b) + mag[:, out:] * np.abs(a)) + 2.0 ** -11 * np.abs(want) + 1e-6)
        else:
            got = y.cpu().numpy()
            assert np.all(np.abs(got - (res + plain)) <= 4e-6 * (mag + np.abs(res)))
            assert np.array_equal(yh[:m].cpu().numpy(), (got * gout).astype(np.float16))
            s, slabs = so.cpu().numpy(), got.reshape(m, rows // 16, 16).astype(np.float64)
            for e in (1, 2):  # f32 sums of 16 terms
                assert np.all(np.abs(s[:, :m, e - 1].T - (slabs ** e).sum(axis=2)) <= 1e-6 * (np.abs(slabs) ** e).sum(axis=2) + 1e-6)
            assert np.all(s[:, m:-(-m // 16) * 16] == 0)
    most = next(k for k in range(m, 5000) if not hip.matmul_f16_takes_few_rows(h, k, flags))
    with pytest.raises(Exception, match="FEW_ROWS"):
        hip.matmul_f16_dev(h, torch_.zeros(-(-most // 64) * 64, cols, dtype=torch_.float16, device="cuda"), most, yh=torch_.zeros(-(-most // 64) * 64, out, dtype=torch_.float16, device="cuda"), flags=flags)
    for a in (h, *(a for a, _ in parts)):
        hip.weights_free(a)

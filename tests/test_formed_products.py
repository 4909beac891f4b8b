"""Matrix-vector products of a vector that is formed on the way (include/bitnet_hip.h section 5: norms, sums, gates, halves), at the edges of what a workgroup takes: rows around one per CU and around
steps of four, columns around chunks of 512, waves per workgroup from one to eight and two chunks per wave; against f64 numpy."""
import ctypes as C

import numpy as np
import pytest

from oracle import stack_oracle as so
from tests import stack_util as u

pytestmark = pytest.mark.gpu
F32_TOL = 3e-6  # sums of up to 8192 f32 products
SIZES = [(1, 264), (3, 512), (255, 520), (256, 1024), (257, 1544), (1022, 768), (1025, 2560), (1200, 4096), (2050, 520), (4100, 1536), (70, 4104), (300, 8192)]


def vectors(n, *seed):
    g = np.random.default_rng([n, *seed])
    return g, [g.standard_normal(n).astype(np.float32) for _ in range(8)]


@pytest.mark.parametrize("rows,cols", SIZES)
@pytest.mark.parametrize("form", ["gated norm", "normed twice", "sum", "layer norm", "halves"])
def test_formed_input(hip, pkg, rows, cols, form):
    g, (x, y, nw, pw, sc, gate, nb, x2) = vectors(cols, rows, len(form))
    eps, ld, mult, n = 1e-3, u.up_to(cols, 64), 0.37, cols // 2 if form == "halves" else cols
    if n % 8:
        pytest.skip("halves in eights")
    w, bias = u.rounded(g.standard_normal((rows, cols)) / np.sqrt(cols)), g.standard_normal(rows).astype(np.float32)
    out, xo, ho = u.zeros_f32(rows), u.zeros_f32(n), u.zeros_f32(n)
    x64, y64 = (x.astype(np.float64) + 1.5)[:n], y.astype(np.float64)[:n]
    kw, inner, formed = dict(n=n, res=u.dev_f32(y[:n]), x_out=xo), x64, None
    if form == "gated norm":
        kw = dict(n=n, kind=pkg.IN_NORM, eps=eps, weight=u.dev_f32(nw), gate=u.dev_f32(gate), mean_n=n - 5)
        vec = x64 / np.sqrt((x64 ** 2).sum() / (n - 5) + eps) * nw * gate
    elif form == "normed twice":
        kw.update(kind=pkg.IN_RESIDUAL_NORM, eps=eps, weight_offset=1.0, weight=u.dev_f32(nw), post_weight=u.dev_f32(pw), scale=u.dev_f32(sc), h_out=ho)
        inner = x64 + sc * so.norm_around_zero(y64, pw, eps)
        vec = formed = so.norm_around_zero(inner, nw, eps)
    elif form == "sum":
        kw.update(kind=pkg.IN_RESIDUAL, eps=eps, post_weight=u.dev_f32(pw))
        vec = inner = x64 + so.norm_plain(y64, pw, eps)
    elif form == "layer norm":
        kw.update(kind=pkg.IN_RESIDUAL_NORM, eps=eps, weight=u.dev_f32(nw), norm_bias=u.dev_f32(nb), center=True, mult=mult, y_gate=u.dev_f32(gate), h_out=ho)
        inner = x64 + mult * y64 * gate
        vec = formed = so.layer_norm(inner, nw, nb, eps)
    else:
        kw.update(kind=pkg.IN_CONCAT, mult=mult, x2=u.dev_f32(x2[:n]))
        inner = x64 + mult * y64
        vec = np.concatenate([inner, x2[:n]])
    wd, xd = u.dev_bf16(u.padded(w, ld)), u.dev_f32(x64.astype(np.float32))
    hip.dense_gemv_dev(xd, wd, rows, cols, ld, out, bias=u.dev_f32(bias), act0=pkg.ACT_NONE, act1=pkg.ACT_RELU2, act_split=rows - rows // 3, **kw)
    want = w.astype(np.float64) @ vec + bias
    want[rows - rows // 3:] = so.relu_squared(want[rows - rows // 3:])
    assert u.rms_error(u.host(out), want) < F32_TOL
    if form != "gated norm":
        assert u.rms_error(u.host(xo), inner) < F32_TOL
    if formed is not None:
        assert u.rms_error(u.host(ho), formed) < F32_TOL
    # an infinite weight in the last column makes its row infinite and no other
    w[rows // 2, cols - 1] = np.inf
    hip.dense_gemv_dev(xd, u.dev_bf16(u.padded(w, ld)), rows, cols, ld, out, **kw)
    got = u.host(out)
    assert np.isinf(got[rows // 2]) and np.isfinite(np.delete(got, rows // 2)).all()


@pytest.mark.parametrize("rows,cols", [(262, 520), (1030, 1536), (2602, 4104)])
@pytest.mark.parametrize("taps,position", [(2, 0), (3, 1), (4, 9), (6, 40)])
def test_formed_input_with_pairs_and_convolution(hip, pkg, rows, cols, taps, position):
    g, (x, y, nw, _, _, _, nb, _) = vectors(cols, rows, taps)
    eps, ld, pairs, channels = 1e-3, u.up_to(cols, 64), 100, 101
    at = rows - channels - 3
    w, bias = u.rounded(g.standard_normal((rows, cols)) / np.sqrt(cols)), g.standard_normal(rows).astype(np.float32)
    conv, ring = g.standard_normal((taps, channels)).astype(np.float32), g.standard_normal((taps, channels)).astype(np.float32)
    cd, rd, pos, out = u.dev_f32(conv), u.dev_f32(ring), u.dev(np.array([position], np.int32)), u.zeros_f32(rows)
    more = pkg.Epilogue(pairs=pairs, act2_from=rows - 3, act2=pkg.ACT_NONE, conv_from=at, channels=channels, taps=taps, conv=cd.data_ptr(), ring=rd.data_ptr(), pos=pos.data_ptr())
    hip.dense_gemv_dev(u.dev_f32(x), u.dev_bf16(u.padded(w, ld)), rows, cols, ld, out, kind=pkg.IN_RESIDUAL_NORM, eps=eps, weight=u.dev_f32(nw), norm_bias=u.dev_f32(nb), center=True,
                       res=u.dev_f32(y), mult=0.5, n=cols, bias=u.dev_f32(bias), act0=pkg.ACT_SILU | pkg.ACT_GATED, act1=pkg.ACT_SIGMOID, act_split=pairs + 1, more=more)
    z = w.astype(np.float64) @ so.layer_norm(x + 0.5 * y.astype(np.float64), nw, nb, eps) + bias
    new = z[at:at + channels].copy()
    z[at:at + channels] *= conv[-1]
    for j in range(1, min(taps - 1, position) + 1):
        z[at:at + channels] += conv[taps - 1 - j].astype(np.float64) * ring[(position - j) % taps]
    want = np.concatenate([so.silu(z[:pairs:2]) * z[1:pairs:2], z[pairs:]])
    want[pairs // 2] = so.silu(z[pairs])
    want[pairs // 2 + 1:-3] = so.sigmoid(z[pairs + 1:-3])
    assert u.rms_error(u.host(out)[:len(want)], want) < F32_TOL
    kept = ring.copy()
    kept[position % taps] = new
    assert u.rms_error(u.host(rd), kept) < F32_TOL


@pytest.mark.parametrize("vocab,cols", [(300, 264), (5000, 1536), (40001, 768)])
def test_formed_input_and_greedy_token(hip, pkg, vocab, cols):
    g, (x, _, nw, *_) = vectors(cols, vocab)
    ld = u.up_to(cols, 64)
    w = u.rounded(g.standard_normal((vocab, cols)))
    best = int(np.argmax(w.astype(np.float64) @ so.norm_plain(x.astype(np.float64), nw, 1e-3)))
    w[vocab - 1] = w[best]  # (the lower of two equal ones)
    xd, nd, wd = u.dev_f32(x), u.dev_f32(nw), u.dev_bf16(u.padded(w, ld))
    logits, scratch, token = u.zeros_f32(vocab), u.zeros_f32(2048), u.dev(np.array([-1], np.int32))
    p = [t.data_ptr() for t in (xd, nd, wd, logits, scratch, token)]
    vi = pkg.VectorInput(x=p[0], weight=p[1], kind=pkg.IN_NORM, eps=1e-3, n=cols)
    hip._call("dense_logits_dev", C.byref(vi), C.c_void_p(p[2]), C.c_size_t(vocab), C.c_size_t(cols), C.c_size_t(ld), C.c_void_p(p[3]), C.c_void_p(p[4]), C.c_void_p(p[5]), None, None, None, None)
    want = w.astype(np.float64) @ so.norm_plain(x.astype(np.float64), nw, 1e-3)
    assert u.rms_error(u.host(logits), want) < F32_TOL and int(u.host(token)[0]) == int(np.argmax(want))


@pytest.mark.parametrize("rows,cols,ld", [(16001, 520, 8192), (7300, 1032, 16384)])
def test_formed_input_of_rows_a_power_of_two_apart(hip, pkg, rows, cols, ld):
    """workgroups that would begin a multiple of 256 KiB apart take four rows more: of two waves, and of three"""
    import torch

    g, (x, _, nw, *_) = vectors(cols, rows)
    w, out = u.rounded(g.standard_normal((rows, cols)) / np.sqrt(cols)), u.zeros_f32(rows)
    wd = torch.zeros((rows, ld), dtype=torch.int16, device="cuda")
    wd[:, :cols] = u.dev_bf16(w).view(torch.int16).reshape(rows, cols)
    hip.dense_gemv_dev(u.dev_f32(x), wd, rows, cols, ld, out, n=cols, kind=pkg.IN_NORM, eps=1e-3, weight=u.dev_f32(nw))
    assert u.rms_error(u.host(out), w.astype(np.float64) @ so.norm_plain(x.astype(np.float64), nw, 1e-3)) < F32_TOL

"""The bf16-weight operators and sequence mixers (include/bitnet_hip.h section 5), one at a time through the C ABI, against the
plain restatement in oracle/stack_oracle.py or f64 numpy."""
import ctypes as C

import numpy as np
import pytest

from oracle import stack_oracle as so
from tests import stack_util as u

pytestmark = pytest.mark.gpu
F32_TOL, BF_TOL = 3e-6, 6e-3


def rng(*seed):
    return np.random.default_rng(list(seed))


@pytest.mark.parametrize("rows,cols", [(5, 8), (33, 32), (100, 80), (64, 200), (300, 264), (1000, 512), (70, 1000), (2500, 2560), (9000, 1288), (40, 6912), (3, 17000)])
def test_gemv_plain(hip, pkg, rows, cols):
    g = rng(rows, cols)
    ld = u.up_to(cols, 64)
    w, x, b = u.rounded(g.standard_normal((rows, cols))), g.standard_normal(cols).astype(np.float32), g.standard_normal(rows).astype(np.float32)
    y = u.zeros_f32(rows)
    hip.dense_gemv_dev(u.dev_f32(x), u.dev_bf16(u.padded(w, ld)), rows, cols, ld, y, bias=u.dev_f32(b), act0=pkg.ACT_NONE, act1=pkg.ACT_RELU2, act_split=rows // 2)
    want = w.astype(np.float64) @ x + b
    want[rows // 2:] = so.relu_squared(want[rows // 2:])
    assert u.rms_error(u.host(y), want) < F32_TOL


@pytest.mark.parametrize("n", [80, 96, 384, 1001, 2560, 2564, 3072, 3076, 4096, 5000])
@pytest.mark.parametrize("kind", ["norm", "gated", "residual", "first"])
def test_gemv_input_transforms(hip, pkg, n, kind):
    g = rng(n, len(kind))
    rows, ld, cols, eps = 90, u.up_to(n, 64), u.up_to(n, 8), 1e-3
    w = u.rounded(g.standard_normal((rows, n)) / np.sqrt(n))
    x, y, nw, pw, ls, gate = (g.standard_normal(n).astype(np.float32) for _ in range(6))
    out, xo = u.zeros_f32(rows), u.zeros_f32(n)
    wd, xd = u.dev_bf16(u.padded(w, ld)), u.dev_f32(x)
    x64 = x.astype(np.float64)
    if kind == "norm":
        hip.dense_gemv_dev(xd, wd, rows, cols, ld, out, kind=pkg.IN_NORM, eps=eps, weight=u.dev_f32(nw), n=n, act0=pkg.ACT_SILU)
        want = so.silu(w @ so.norm_plain(x64, nw, eps))
    elif kind == "gated":
        hip.dense_gemv_dev(xd, wd, rows, cols, ld, out, kind=pkg.IN_NORM, eps=eps, weight=u.dev_f32(nw), gate=u.dev_f32(gate), n=n, mean_n=n - 7, act0=pkg.ACT_SIGMOID)
        want = so.sigmoid(w @ (x64 / np.sqrt((x64 ** 2).sum() / (n - 7) + eps) * nw * gate))
    elif kind == "first":
        hip.dense_gemv_dev(xd, wd, rows, cols, ld, out, kind=pkg.IN_RESIDUAL_NORM, eps=eps, weight_offset=1.0, weight=u.dev_f32(nw), n=n)
        want = w @ so.norm_around_zero(x64, nw, eps)
    else:
        hip.dense_gemv_dev(xd, wd, rows, cols, ld, out, kind=pkg.IN_RESIDUAL_NORM, eps=eps, weight_offset=1.0, weight=u.dev_f32(nw), res=u.dev_f32(y),
                           post_weight=u.dev_f32(pw), scale=u.dev_f32(ls), x_out=xo, n=n)
        x2 = x64 + ls * so.norm_around_zero(y.astype(np.float64), pw, eps)
        want = w @ so.norm_around_zero(x2, nw, eps)
        assert u.rms_error(u.host(xo), x2) < F32_TOL
    assert u.rms_error(u.host(out), want) < F32_TOL


@pytest.mark.parametrize("heads,rows,cols", [(3, 64, 32), (5, 128, 96), (2, 512, 128)])
def test_gemv_batched(hip, heads, rows, cols):
    g = rng(heads, rows)
    ld, step = u.up_to(cols, 64), cols + 32
    w, x = u.rounded(g.standard_normal((heads, rows, cols))), g.standard_normal((heads, step)).astype(np.float32)
    y = u.zeros_f32(heads, rows)
    hip.dense_gemv_dev(u.dev_f32(x), u.dev_bf16(u.padded(w, ld)), rows, cols, ld, y, batch=heads, w_batch=rows * ld, x_batch=step, y_batch=rows)
    assert u.rms_error(u.host(y), np.einsum("hrc,hc->hr", w.astype(np.float64), x[:, :cols])) < F32_TOL


@pytest.mark.parametrize("m,n,k", [(1, 5, 64), (2, 130, 128), (127, 128, 64), (128, 129, 192), (300, 417, 320), (257, 1000, 512), (1030, 258, 2560)])
@pytest.mark.parametrize("f32", [False, True])
def test_matmul(hip, pkg, m, n, k, f32):
    g = rng(m, n, k)
    a, w, b = u.rounded(g.standard_normal((m, k))), u.rounded(g.standard_normal((n, k)) / np.sqrt(k)), g.standard_normal(n).astype(np.float32)
    if f32:
        a = g.standard_normal((m, k)).astype(np.float32)
    ad, wd = (u.dev_f32(a) if f32 else u.dev_bf16(a)), u.dev_bf16(w)
    want = a.astype(np.float64) @ w.T.astype(np.float64) + b
    want[:, n // 3:] = so.silu(want[:, n // 3:])
    for c_f32 in (True, False):
        ldc = n + 3
        c = u.zeros_f32(m, ldc) if c_f32 else u.zeros_bf16(m, ldc)
        hip.dense_matmul_dev(ad, k, f32, wd, k, m, n, k, c, ldc, c_f32, bias=u.dev_f32(b), act0=pkg.ACT_NONE, act1=pkg.ACT_SILU, act_split=n // 3)
        got = u.host(c)
        assert u.rms_error(got[:, :n], want) < (F32_TOL if c_f32 else 3e-3)
        assert not got[:, n:].any()


# the form for few rows: its three tiles at the edges of their ranges (one round of 256 workgroups), K that does not go round its eight waves, rows and columns
# that end inside a tile, batches; the last two lie just behind the ranges.  Tolerances as in test_matmul: sums of k products in f32, one rounding to bf16.
@pytest.mark.parametrize("m,n,k,batch,tile", [(1, 1, 512, 1, (16, 16)), (16, 4096, 576, 1, (16, 16)), (17, 2048, 512, 1, (16, 16)), (19, 40, 1984, 3, (16, 16)), (33, 1000, 640, 1, (16, 16)),
                                              (61, 4096, 512, 1, (32, 32)), (64, 130, 4096, 2, (16, 16)), (65, 4090, 512, 1, None), (257, 1600, 768, 1, None),
                                              (65, 4090, 1536, 1, (32, 64)), (257, 1600, 1600, 1, (32, 64)), (2760, 72, 512, 1, (32, 64)), (1400, 160, 2560, 1, (32, 32)), (1500, 320, 1536, 1, (32, 64)),
                                              (2048, 72, 1536, 1, (32, 32)), (64, 8200, 512, 1, None), (64, 100, 448, 1, None)])
@pytest.mark.parametrize("form", ["f32", "bf16", "gated"])
def test_matmul_few_rows(hip, pkg, m, n, k, batch, tile, form):
    if form == "gated":
        n = u.up_to(n, 2)
    g = rng(m, n, k)
    a, w, b = u.rounded(g.standard_normal((batch, m, k))), u.rounded(g.standard_normal((batch, n, k)) / np.sqrt(k)), g.standard_normal(n).astype(np.float32)
    want = np.stack([x.astype(np.float64) @ y.T.astype(np.float64) for x, y in zip(a, w)]) + b
    ldc, act0, split = n + 4, pkg.ACT_NONE, n // 3
    want[:, :, split:] = so.silu(want[:, :, split:]) if form != "gated" else want[:, :, split:]
    if form == "gated":
        act0, split, ldc = pkg.ACT_SILU | pkg.ACT_GATED, 0, n // 2 + 3
        want = so.silu(want[:, :, ::2]) * want[:, :, 1::2]
    elif split == 0:  # (no split: the first activation for all)
        act0 = pkg.ACT_SILU
    c = u.zeros_f32(batch * m, ldc) if form == "f32" else u.zeros_bf16(batch * m, ldc)
    hip.dense_matmul_dev(u.dev_bf16(a), k, False, u.dev_bf16(w), k, m, n, k, c, ldc, form == "f32", bias=u.dev_f32(b), act0=act0, act1=pkg.ACT_SILU if split else 0, act_split=split,
                         batch=batch, a_batch=m * k, w_batch=n * k, c_batch=m * ldc)
    ran = hip.dense_matmul_last_tile()
    assert ran == (*tile, 8, 8) if tile else ran[3] == 1, ran
    got = u.host(c).reshape(batch, m, ldc)
    assert u.rms_error(got[:, :, :want.shape[2]], want) < (F32_TOL if form == "f32" else 3e-3)
    assert not got[:, :, want.shape[2]:].any()


# the same rows alone (the form for few rows) and among many (tiles of 64 columns and more): sums of these inputs are exact in any order, so that whatever differs comes from
# the epilogue; whole and ragged columns, one activation and two, the split inside and between what a wave holds
@pytest.mark.parametrize("n,split", [(256, 0), (384, 128), (384, 200), (390, 0)])
@pytest.mark.parametrize("form", ["f32", "bf16", "gated"])
def test_matmul_activations_are_those_of_the_call(hip, pkg, n, split, form):
    k, m, g = 512, 4096, rng(n, split)
    gated, f32 = form == "gated", form == "f32"
    a, w = g.integers(-4, 5, (m, k)).astype(np.float32) / 8, g.integers(-4, 5, (n, k)).astype(np.float32) / 16
    ad, wd, b = u.dev_bf16(a), u.dev_bf16(w), u.dev_f32(g.integers(-8, 9, n).astype(np.float32) / 8)
    acts = [pkg.ACT_SILU, pkg.ACT_SIGMOID, pkg.ACT_RELU2, pkg.ACT_GELU_TANH] + ([] if gated else [pkg.ACT_XIELU])
    for i, act in enumerate(acts):
        if gated and split:
            continue
        got = []
        for rows in (16, m):
            c = (u.zeros_f32 if f32 else u.zeros_bf16)(rows, n)
            hip.dense_matmul_dev(ad, k, False, wd, k, rows, n, k, c, n, f32, bias=b, act0=act | (pkg.ACT_GATED if gated else 0), act1=acts[i - 1] if split else 0, act_split=split,
                                 more=pkg.Epilogue(act_a=0.7, act_b=0.9) if pkg.ACT_XIELU in (act, acts[i - 1]) and not gated else None)
            got.append(u.host(c)[:16])
        assert got[0].any() and np.array_equal(*got), (act, np.abs(got[0] - got[1]).max())


# whole numbers of the matmul's tiles and ends inside one, two activations, and outputs that start on no sixteen bytes; test_matmul_by_tile says which tile takes a shape
@pytest.mark.parametrize("m,n", [(4096, 4096), (4000, 4080), (4096, 3072), (3900, 3060), (2048, 3072), (2040, 4056), (2048, 2560), (1537, 2570), (1500, 2568), (700, 2552), (1531, 1528)])
@pytest.mark.parametrize("form", ["f32", "bf16", "gated", "unaligned"])
def test_matmul_tiles(hip, pkg, m, n, form):
    import torch
    k, g = 1088, torch.Generator(device="cuda").manual_seed(m + n)
    a, w = (torch.randn(r, k, device="cuda", generator=g).bfloat16() for r in (m, n))
    b = torch.randn(n, device="cuda", generator=g)
    wd = (w.double() / np.sqrt(k)).bfloat16()
    want = a.double() @ wd.double().T + b.double()
    gated, f32 = form == "gated", form == "f32"
    if gated:
        want = torch.nn.functional.silu(want[:, ::2]) * want[:, 1::2]
    else:
        want[:, n // 3:] = torch.nn.functional.silu(want[:, n // 3:])
    cols = want.shape[1]
    ldc = cols + 5 if form == "unaligned" else u.up_to(cols, 64)
    c = torch.zeros(m, ldc, device="cuda", dtype=torch.float32 if f32 else torch.bfloat16)
    hip.dense_matmul_dev(a, k, False, wd, k, m, n, k, c, ldc, f32, bias=b, act0=pkg.ACT_SILU | pkg.ACT_GATED if gated else pkg.ACT_NONE, act1=0 if gated else pkg.ACT_SILU,
                         act_split=0 if gated else n // 3)
    torch.cuda.synchronize()
    assert ((c[:, :cols].double() - want).norm() / want.norm()).item() < (F32_TOL if f32 else 3e-3)
    assert not c[:, cols:].any()


# every tile by name, for whole and for ragged columns: (columns, rows, waves) of plain outputs, of gated ones and of those whose rows do not start on sixteen bytes; f32 rows
# a multiple of four apart do.  A moved constant of the launcher's costs shows up here.
BY_TILE = [(2000, 7680, 1088, (256, 256, 8), (256, 256, 8), (256, 256, 8)), (1500, 7680, 1088, (192, 256, 8), (192, 256, 8), (192, 256, 8)),
           (1000, 7680, 1088, (128, 256, 8), (128, 256, 8), (128, 256, 8)), (520, 7680, 1088, (128, 192, 8), (128, 192, 8), (128, 192, 8)),
           (700, 4096, 4096, (128, 128, 8), (128, 128, 8), (128, 128, 8)), (2000, 7700, 1088, (128, 128, 4), (256, 256, 8), (256, 256, 8)),
           (1500, 4100, 1088, (128, 128, 4), (128, 256, 8), (128, 128, 4)), (700, 2560, 1088, (64, 128, 4), (64, 128, 4), (64, 128, 4)),
           (520, 4100, 4096, (128, 128, 8), (128, 128, 8), (128, 128, 8)), (1000, 7700, 2048, (128, 128, 4), (128, 256, 8), (128, 256, 8)),
           (300, 1500, 1088, (64, 64, 4), (64, 64, 4), (64, 64, 4)), (4096, 1088, 1024, (64, 64, 4), (64, 64, 4), (64, 64, 4))]


@pytest.mark.parametrize("m,n,k,plain,pairs,odd", BY_TILE)
@pytest.mark.parametrize("form", ["f32", "f32 + 4", "f32 + 3", "bf16", "bf16 + 4", "gated", "gated + 1"])
def test_matmul_by_tile(hip, pkg, m, n, k, plain, pairs, odd, form):
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n)
    a, w = (torch.randn(r, k, device="cuda", generator=g).bfloat16() for r in (m, n))
    b = torch.randn(n, device="cuda", generator=g)
    w = (w.double() / np.sqrt(k)).bfloat16()
    want = a.double() @ w.double().T + b.double()
    gated, f32 = form.startswith("gated"), form.startswith("f32")
    if gated:
        want = torch.nn.functional.silu(want[:, ::2]) * want[:, 1::2]
    cols, more = want.shape[1], int(form[form.index("+") + 2:]) if "+" in form else 0
    ldc = u.up_to(cols, 8) + more
    c = torch.zeros(m, ldc, device="cuda", dtype=torch.float32 if f32 else torch.bfloat16)
    hip.dense_matmul_dev(a, k, False, w, k, m, n, k, c, ldc, f32, bias=b, act0=pkg.ACT_SILU | pkg.ACT_GATED if gated else pkg.ACT_NONE)
    ran = hip.dense_matmul_last_tile()
    torch.cuda.synchronize()
    assert ((c[:, :cols].double() - want).norm() / want.norm()).item() < (F32_TOL if f32 else 3e-3)
    assert not c[:, cols:].any()
    if not (more and gated):  # (half the elements to store one by one: its own choice)
        assert ran == (*(odd if more and form != "f32 + 4" else pairs if gated else plain), 1), ran


def test_matmul_batched_f32(hip):
    g = rng(9)
    heads, m, n, k, step = 3, 70, 64, 64, 96
    a, w = g.standard_normal((m, heads * step)).astype(np.float32), u.rounded(g.standard_normal((heads, n, k)))
    c = u.zeros_f32(m, heads * n)
    hip.dense_matmul_dev(u.dev_f32(a), heads * step, True, u.dev_bf16(w), k, m, n, k, c, heads * n, True, batch=heads, a_batch=step, w_batch=n * k, c_batch=n)
    want = np.concatenate([a[:, h * step:h * step + k].astype(np.float64) @ w[h].T for h in range(heads)], axis=1)
    assert u.rms_error(u.host(c), want) < F32_TOL


@pytest.mark.parametrize("width", [96, 1000, 2560, 4096, 5000])
def test_residual_norm_rows(hip, width):
    g = rng(width)
    m, ldh, eps = 5, u.up_to(width, 64), 1e-2
    x, y = (g.standard_normal((m, width)).astype(np.float32) for _ in range(2))
    pw, ls, nw = (g.standard_normal(width).astype(np.float32) for _ in range(3))
    xd, h = u.dev_f32(x), u.zeros_f32(m, ldh)
    hip.residual_norm_rows_dev(xd, m, width, eps, 1.0, y=u.dev_f32(y), ldy=width, post_weight=u.dev_f32(pw), scale=u.dev_f32(ls), next_weight=u.dev_f32(nw), h=h, ldh=ldh)
    want = x + ls * so.norm_around_zero(y.astype(np.float64), pw, eps)
    assert u.rms_error(u.host(xd), want) < F32_TOL
    assert u.rms_error(u.host(h)[:, :width], so.norm_around_zero(want, nw, eps)) < F32_TOL
    hb = u.zeros_bf16(m, ldh) + 7
    hip.residual_norm_rows_dev(xd, m, width, eps, 1.0, next_weight=u.dev_f32(nw), h=hb, ldh=ldh, h_f32=False)
    assert u.rms_error(u.host(hb)[:, :width], so.norm_around_zero(want, nw, eps)) < BF_TOL
    assert not u.host(hb)[:, width:].any()


# ---- latent attention --------------------------------------------------------------------------------------------------
class Latent:
    """random queries, cache and weights of one latent attention, in the library's layouts, and its output by definition"""

    def __init__(self, pkg, L, nq, heads, dim, rot, vdim, rank, f32, seed=0, spike=None):
        g = rng(L, nq, heads, dim, seed)
        self.L, self.nq, self.heads, self.f32 = L, nq, heads, f32
        store = (lambda a: a.astype(np.float32)) if f32 else u.rounded
        self.dimp, self.rotp, self.vdimp, self.ldc, self.cap = u.up_to(dim, 32), u.up_to(rot, 32), u.up_to(vdim, 32), u.up_to(rank, 64), u.up_to(L, 64)
        self.qd = self.dimp + self.rotp
        q = store(g.standard_normal((nq, heads, dim + rot)))
        c, kr = store(g.standard_normal((L, rank))), store(g.standard_normal((L, rot)))
        uk, uv = u.rounded(g.standard_normal((heads, dim, rank)) / np.sqrt(rank)), u.rounded(g.standard_normal((heads, vdim, rank)) / np.sqrt(rank))
        sink = g.standard_normal(heads).astype(np.float32)
        spec = {"dims": rot, "base": 5000.0, "scaling": {"factor": 4.0, "original": 64, "fast": 16.0, "slow": 1.0}}
        f, mult = so.rotary_frequencies(spec)
        ang = np.arange(self.cap)[:, None] * f
        self.cos, self.sin = u.dev_f32(np.cos(ang) * mult), u.dev_f32(np.sin(ang) * mult)
        scale = 0.2
        if spike is not None:  # one key whose score stands far above the others for every query and head
            c[spike] = store(c[spike] * 0)
            qr = np.stack([so.rotate(q[i:i + 1, :, dim:], [L - nq + i], spec)[0] for i in range(nq)])
            v = qr.mean(axis=(0, 1))
            kr[spike] = store(v / np.linalg.norm(v) * 6)
            q[:, :, dim:] = q[:1, :1, dim:]
            qr = np.stack([so.rotate(q[i:i + 1, :, dim:], [L - nq + i], spec)[0] for i in range(nq)])
            kr[spike] = store(qr[0, 0] / np.linalg.norm(qr[0, 0]) * 30)
        q64 = q.astype(np.float64)
        qr = np.stack([so.rotate(q64[i:i + 1, :, dim:], [L - nq + i], spec)[0] for i in range(nq)])
        out = np.zeros((nq, heads, vdim))
        for h in range(heads):
            k, v = c.astype(np.float64) @ uk[h].T, c.astype(np.float64) @ uv[h].T
            s = (q64[:, h, :dim] @ k.T + qr[:, h] @ kr.T.astype(np.float64)) * scale
            for i in range(nq):
                n = L - nq + i + 1
                top = max(s[i, :n].max(), sink[h])
                e = np.exp(s[i, :n] - top)
                out[i, h] = e @ v[:n] / (e.sum() + np.exp(sink[h] - top))
        self.want = out
        dq = np.zeros((nq, heads, self.qd), np.float32)
        dq[:, :, :dim], dq[:, :, self.dimp:self.dimp + rot] = q[:, :, :dim], q[:, :, dim:]
        self.q = dq
        put = u.dev_f32 if f32 else u.dev_bf16
        cache = np.zeros((self.cap, self.ldc), np.float32)
        cache[:L, :rank] = c
        rc = np.zeros((self.cap, self.rotp), np.float32)
        rc[:L, :rot] = kr
        self.c_host, self.cache, self.rcache, self.sink = cache, put(cache), put(rc), u.dev_f32(sink)
        self.uv_host = np.zeros((heads, self.vdimp, self.ldc), np.float32)
        self.uv_host[:, :vdim, :rank] = uv
        self.uk_host = np.zeros((heads, self.dimp, self.ldc), np.float32)
        self.uk_host[:, :dim, :rank] = uk
        self.vdim = vdim
        self.attn = pkg.LatentAttention(heads, self.dimp, self.qd, self.vdimp, rank, rot, scale, self.sink.data_ptr(), self.cache.data_ptr(), self.rcache.data_ptr(),
                                        self.ldc, self.rotp, self.cap, self.cos.data_ptr(), self.sin.data_ptr())

    def decode(self, hip):
        qabs = np.einsum("nhd,hdc->nhc", self.q[:, :, :self.dimp].astype(np.float64), self.uk_host)
        scratch = u.zeros_f32(hip.latent_scratch_bytes(self.heads, self.ldc, self.nq) // 4)
        pos, out = u.dev(np.array([self.L - self.nq], np.int32)), u.zeros_f32(self.nq, self.heads, self.vdimp)
        hip.latent_decode_dev(self.attn, u.dev_f32(self.q), u.dev_f32(qabs), pos, 0, self.nq, self.f32, scratch)
        hip.latent_merge_dev(self.attn, u.dev_bf16(self.uv_host), pos, 0, self.nq, scratch, out, self.heads * self.vdimp, False)
        return u.host(out)

    def prefill(self, hip):
        k = np.einsum("lc,hdc->lhd", self.c_host, self.uk_host)
        vt = np.einsum("lc,hvc->hvl", self.c_host, self.uv_host)
        out = u.zeros_bf16(self.nq, self.heads, self.vdimp)
        hip.latent_prefill_dev(self.attn, u.dev_bf16(self.q), u.dev_bf16(k), u.dev_bf16(vt), self.cap, self.L, self.nq, out, self.heads * self.vdimp)
        return u.host(out)

    def check(self, got, tol):
        assert u.rms_error(got[:, :, :self.vdim], self.want) < tol
        assert not got[:, :, self.vdim:].any()


SHAPES = [(4, 32, 32, 32, 64), (3, 24, 16, 40, 72), (17, 128, 64, 128, 512), (20, 64, 32, 100, 320), (2, 180, 40, 256, 200)]


@pytest.mark.parametrize("L", [1, 2, 63, 64, 65, 700])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("f32", [True, False])
def test_latent_decode(hip, pkg, shape, L, f32):
    t = Latent(pkg, L, 1, *shape, f32)
    t.check(t.decode(hip), 1e-5 if f32 else 1e-4)  # (bf16 cache values are exact inputs here: only the query's split is rounded)


@pytest.mark.parametrize("f32", [True, False])
def test_latent_decode_long_and_several_queries(hip, pkg, f32):
    t = Latent(pkg, 8500, 2, 5, 32, 32, 32, 64, f32)  # more tiles than records
    t.check(t.decode(hip), 1e-5 if f32 else 1e-4)
    t = Latent(pkg, 130, 70, *SHAPES[1], f32)
    t.check(t.decode(hip), 1e-5 if f32 else 1e-4)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("shape,nq", [(SHAPES[2], 15), (SHAPES[2], 16), (SHAPES[3], 64), ((129, 32, 32, 32, 64), 2), ((65, 32, 32, 256, 1024), 4)])
def test_latent_decode_of_more_queries_than_one_round(hip, pkg, shape, nq, f32):
    t = Latent(pkg, 150, nq, *shape, f32)
    t.check(t.decode(hip), 1e-5 if f32 else 1e-4)


def test_latent_decode_large_latent_in_bf16(hip, pkg):
    t = Latent(pkg, 150, 2, 3, 64, 64, 32, 900, False)  # beyond the matrix-core form's latent
    t.check(t.decode(hip), 1e-4)


@pytest.mark.parametrize("L,nq", [(1, 1), (2, 2), (64, 64), (65, 2), (129, 129), (300, 37), (700, 700)])
@pytest.mark.parametrize("shape", SHAPES + [(9, 96, 96, 64, 128), (1, 160, 96, 16, 64)])
def test_latent_prefill(hip, pkg, shape, L, nq):
    t = Latent(pkg, L, nq, *shape, False)
    t.check(t.prefill(hip), 1.5e-2 if L > 1 else 4e-2)  # (one key: its rounded score decides its share against the sink)


@pytest.mark.parametrize("spike", [0, 1, 63, 64, 127, 128, 500, 639])
def test_latent_attention_finds_one_key(hip, pkg, spike):
    """one key takes nearly all of the weight, wherever it lies"""
    t = Latent(pkg, 640, 1, *SHAPES[0], False, seed=spike, spike=spike)
    v = np.abs(t.want).max()
    assert v < 0.2  # (its value vector is zero: a kernel that misses it returns an average of the others)
    assert np.abs(t.decode(hip)[:, :, :t.vdim] - t.want).max() < 1e-3
    assert np.abs(t.prefill(hip)[:, :, :t.vdim] - t.want).max() < 5e-3


@pytest.mark.parametrize("f32", [True, False])
def test_latent_rows(hip, pkg, f32):
    g = rng(5)
    m, qr, kr, rot, pos0, eps = 7, 56, 72, 16, 61, 1e-2
    ldq, ldc, ldr, cap = 64, 128, 32, 128
    z, qw, kw = g.standard_normal((m, qr + kr + rot)).astype(np.float32), g.standard_normal(qr).astype(np.float32), g.standard_normal(kr).astype(np.float32)
    spec = {"dims": rot, "base": 300.0}
    f, _ = so.rotary_frequencies(spec)
    ang = np.arange(cap)[:, None] * f
    new = u.zeros_f32 if f32 else u.zeros_bf16
    cq, c, r = new(m, ldq), new(cap, ldc), new(cap, ldr)
    keep = [u.dev_f32(v) for v in (z, qw, kw, np.cos(ang), np.sin(ang))] + [u.dev(np.array([pos0], np.int32))]
    a = [t.data_ptr() for t in keep]
    rows = pkg.LatentRows(a[0], z.shape[1], qr, kr, rot, a[1], a[2], eps, cq.data_ptr(), ldq, c.data_ptr(), r.data_ptr(), ldc, ldr, a[3], a[4], a[5])
    hip.latent_rows_dev(rows, m, f32)
    z64, tol = z.astype(np.float64), F32_TOL if f32 else BF_TOL
    assert u.rms_error(u.host(cq)[:, :qr], so.norm_plain(z64[:, :qr], qw, eps)) < tol and not u.host(cq)[:, qr:].any()
    assert u.rms_error(u.host(c)[pos0:pos0 + m, :kr], so.norm_plain(z64[:, qr:qr + kr], kw, eps)) < tol
    assert u.rms_error(u.host(r)[pos0:pos0 + m, :rot], so.rotate(z64[:, qr + kr:], range(pos0, pos0 + m), spec)) < tol
    got = u.host(c)
    assert not got[:pos0].any() and not got[pos0 + m:].any() and not got[:, kr:].any()


# ---- linear attention --------------------------------------------------------------------------------------------------
def linear_case(n, heads, dim, vdim, decay, seed=0):
    g = rng(n, heads, dim, seed)
    dimp, vdimp = u.up_to(dim, 32), u.up_to(vdim, 32)
    q, k, v = u.rounded(g.standard_normal((n, heads, dim))), u.rounded(g.standard_normal((n, heads, dim))), u.rounded(g.standard_normal((n, heads, vdim)))
    S = g.standard_normal((heads, dim, vdim))
    state = np.zeros((heads, vdimp, dimp), np.float32)
    state[:, :vdim, :dim] = S.transpose(0, 2, 1)
    S = state[:, :vdim, :dim].transpose(0, 2, 1).astype(np.float64)
    out = np.zeros((n, heads, vdim))
    for t in range(n):
        S = np.array(decay)[:, None, None] * S + k[t].astype(np.float64)[:, :, None] * v[t].astype(np.float64)[:, None, :]
        out[t] = np.einsum("hdv,hd->hv", S, q[t].astype(np.float64))
    qkv = np.concatenate([u.padded(q, dimp).reshape(n, -1), u.padded(k, dimp).reshape(n, -1), u.padded(v, vdimp).reshape(n, -1)], axis=1)
    pw = np.array([[d ** i for i in range(129)] for d in decay], np.float32)
    return dimp, vdimp, qkv, state, pw, out, S


LINEAR = [(1, 3, 40, 24), (2, 2, 64, 64), (127, 2, 32, 96), (128, 6, 64, 64), (129, 2, 128, 128), (300, 1, 200, 160), (521, 2, 96, 32)]


@pytest.mark.parametrize("n,heads,dim,vdim", LINEAR)
@pytest.mark.parametrize("form", ["recurrent", "chunked"])
def test_linear_attention(hip, form, n, heads, dim, vdim):
    decay = [0.5, 0.999, 1.0, 0.0, 0.9, 0.97][:heads]
    dimp, vdimp, qkv, state, pw, want, S = linear_case(n, heads, dim, vdim, decay)
    st, out, pd = u.dev_f32(state), u.zeros_f32(n, heads, vdimp), u.dev_f32(pw)
    if form == "recurrent":
        hip.linear_recurrent_dev(u.dev_f32(qkv), qkv.shape[1], n, heads, dimp, vdimp, pd, st, out, heads * vdimp)
    else:
        nb = hip.linear_workspace_bytes(n, heads, dimp, vdimp)
        hip.linear_chunked_dev(u.dev_bf16(qkv), qkv.shape[1], n, heads, dimp, vdimp, pd, st, out, heads * vdimp, u.zeros_f32(nb // 4), nb)
    got, gs = u.host(out), u.host(st)
    tol = 1e-5 if form == "recurrent" else 1e-4
    for h in range(heads):
        assert u.rms_error(got[:, h, :vdim], want[:, h]) < tol, (h, decay[h])
        assert u.rms_error(gs[h, :vdim, :dim].T, S[h]) < tol, (h, decay[h])
    assert not got[:, :, vdim:].any()


def test_linear_attention_forms_hand_the_state_over(hip):
    """portions of every size through both forms: the state carries"""
    heads, dim, vdim, n = 2, 64, 32, 400
    dimp, vdimp, qkv, state, pw, want, _ = linear_case(n, heads, dim, vdim, [0.95, 0.999])
    st, pd, got, at = u.dev_f32(state), u.dev_f32(pw), [], 0
    for size in (2, 1, 130, 3, 128, 1, 127, 8):
        out, part = u.zeros_f32(size, heads, vdimp), qkv[at:at + size]
        if size == 1:
            hip.linear_recurrent_dev(u.dev_f32(part), qkv.shape[1], size, heads, dimp, vdimp, pd, st, out, heads * vdimp)
        else:
            nb = hip.linear_workspace_bytes(size, heads, dimp, vdimp)
            hip.linear_chunked_dev(u.dev_bf16(part), qkv.shape[1], size, heads, dimp, vdimp, pd, st, out, heads * vdimp, u.zeros_f32(nb // 4), nb)
        got.append(u.host(out))
        at += size
    assert at == n and u.rms_error(np.concatenate(got)[:, :, :vdim], want) < 1e-4


@pytest.mark.parametrize("dim,vdim", [(32, 128), (96, 160), (160, 96)])
def test_linear_attention_in_shares_of_value_columns(hip, dim, vdim):
    """Many workgroups take all of a head's value columns each, few of them 64 columns: the same outputs, bit for bit."""
    n, heads = 129, 129
    dimp, vdimp, qkv, state, pw, want, S = linear_case(n, heads, dim, vdim, [0.5 + 0.49 * h / heads for h in range(heads)])

    def run(h0, count):
        cut = [qkv[:, o + h0 * w:o + (h0 + count) * w] for o, w in ((0, dimp), (heads * dimp, dimp), (2 * heads * dimp, vdimp))]
        part = np.ascontiguousarray(np.concatenate(cut, axis=1))
        out, nb = u.zeros_f32(n, count, vdimp), hip.linear_workspace_bytes(n, count, dimp, vdimp)
        hip.linear_chunked_dev(u.dev_bf16(part), part.shape[1], n, count, dimp, vdimp, u.dev_f32(pw[h0:h0 + count]), u.dev_f32(state[h0:h0 + count]), out, count * vdimp, u.zeros_f32(nb // 4), nb)
        return u.host(out)

    got = run(0, heads)
    assert all(u.rms_error(got[:, h, :vdim], want[:, h]) < 1e-4 for h in (0, 64, 128))
    assert np.array_equal(got[:, 3:5], run(3, 2)) and np.array_equal(got[:, 128:], run(128, 1))


def test_gated_norm_rows(hip):
    g = rng(3)
    m, n, mean_n, ldh, eps = 4, 96, 80, 128, 1e-2
    o, w, gate = g.standard_normal((m, n)).astype(np.float32), g.standard_normal(n).astype(np.float32), g.standard_normal((m, 200)).astype(np.float32)
    h = u.zeros_f32(m, ldh) + 1
    hip.gated_norm_rows_dev(u.dev_f32(o), n, u.dev_f32(w), u.dev_f32(gate), 200, eps, True, m, n, mean_n, h, ldh, True)
    o64 = o.astype(np.float64)
    want = o64 / np.sqrt((o64 ** 2).sum(1, keepdims=True) / mean_n + eps) * w * gate[:, :n]
    assert u.rms_error(u.host(h)[:, :n], want) < F32_TOL and not u.host(h)[:, n:].any()


@pytest.mark.parametrize("n,width", [(0, 0), (1, 0), (255, 256), (257, 1), (3000, 2560)])
def test_sequence_update(hip, n, width):
    import torch

    history, scalars, x = torch.full((4000,), 9, dtype=torch.int32, device="cuda"), torch.tensor([5, 6], dtype=torch.int32, device="cuda"), torch.full((width + 2,), 3.0, device="cuda")
    tokens, row = torch.arange(n + 1, dtype=torch.int32).pin_memory(), torch.randn(width + 1, device="cuda")
    P = lambda t, at=0: C.c_void_p(t.data_ptr() + 4 * at)
    call = lambda *a: hip._call("sequence_update_dev", *a, C.c_void_p(torch.cuda.current_stream().cuda_stream))
    call(P(history), C.c_size_t(7), C.c_size_t(n), P(tokens), P(scalars), C.c_int32(11), None, C.c_int32(0), P(row), P(x, 1), C.c_size_t(width))
    torch.cuda.synchronize()
    want = torch.full((4000,), 9, dtype=torch.int32)
    want[7:7 + n] = tokens[:n]
    assert torch.equal(history.cpu(), want) and scalars.tolist() == [11, 6]
    assert torch.equal(x[1:1 + width], row[:width]) and x[0] == 3 and x[-1] == 3
    call(P(history), C.c_size_t(8), C.c_size_t(n), None, None, C.c_int32(1), P(scalars, 1), C.c_int32(12), None, None, C.c_size_t(0))
    torch.cuda.synchronize()
    want[8:8 + n] = 0
    assert torch.equal(history.cpu(), want) and scalars.tolist() == [11, 12]
    with pytest.raises(Exception):
        call(None, C.c_size_t(0), C.c_size_t(1), P(tokens), None, C.c_int32(0), None, C.c_int32(0), None, None, C.c_size_t(0))


@pytest.mark.parametrize("shift", [0, 1])  # rows that start off their alignment go column by column
@pytest.mark.parametrize("width", [4, 1024, 1028, 2048, 2052, 3072, 3076, 3073, 4100])
def test_row_norms_at_register_edges(hip, width, shift):
    g = rng(width, shift)
    m, ldh, eps = 3, u.up_to(width, 64) + 4, 1e-2
    x, y = (g.standard_normal((m, width)).astype(np.float32) for _ in range(2))
    pw, nw = (g.standard_normal(width).astype(np.float32) for _ in range(2))
    gate = u.rounded(g.standard_normal((m, width)))
    y64, gate_ld = y.astype(np.float64), u.up_to(width, 4)

    def off(a, zeros):  # a device tensor whose first element lies `shift` past an aligned place
        d = zeros(a.size + 8)
        d[shift:shift + a.size] = (u.dev_f32(a) if zeros is u.zeros_f32 else u.dev_bf16(a)).reshape(-1)
        return d[shift:shift + a.size]

    for f32, tol in ((True, F32_TOL), (False, BF_TOL)):
        h, xd = (u.zeros_f32 if f32 else u.zeros_bf16)(m, ldh) + 7, off(x, u.zeros_f32)
        hip.residual_norm_rows_dev(xd, m, width, eps, 0.5, y=off(y, u.zeros_f32), ldy=width, post_weight=off(pw, u.zeros_f32), next_weight=u.dev_f32(nw), h=h, ldh=ldh, h_f32=f32)
        want = x + y64 / np.sqrt((y64 ** 2).mean(1, keepdims=True) + eps) * (0.5 + pw)
        assert u.rms_error(u.host(xd).reshape(m, width), want) < F32_TOL
        want = want / np.sqrt((want ** 2).mean(1, keepdims=True) + eps) * (0.5 + nw)
        assert u.rms_error(u.host(h)[:, :width], want) < tol and not u.host(h)[:, width:].any()

        h = (u.zeros_f32 if f32 else u.zeros_bf16)(m, ldh) + 7
        hip.gated_norm_rows_dev(off(y, u.zeros_f32), width, u.dev_f32(pw), (u.dev_f32 if f32 else u.dev_bf16)(u.padded(gate, gate_ld)), gate_ld, eps, f32, m, width, width, h, ldh, f32)
        want = y64 / np.sqrt((y64 ** 2).mean(1, keepdims=True) + eps) * pw * gate
        assert u.rms_error(u.host(h)[:, :width], want) < tol and not u.host(h)[:, width:].any()


@pytest.mark.parametrize("width", [64, 252, 256, 260, 508, 512, 516])
def test_row_norms_of_narrow_rows(hip, width):
    test_row_norms_at_register_edges(hip, width, 0)


@pytest.mark.parametrize("width,shift", [(255, 0), (3, 0), (1024, 1), (4095, 0), (4096, 1), (4097, 0), (4100, 1), (8192, 0)])
def test_row_norms_of_single_columns(hip, width, shift):
    test_row_norms_at_register_edges(hip, width, shift)


@pytest.mark.parametrize("q_rank,kv_rank", [(0, 1024), (2048, 0), (2049, 1025), (257, 1), (1536, 512)])
def test_latent_rows_at_register_edges(hip, pkg, q_rank, kv_rank):
    import torch

    g = rng(q_rank, kv_rank)
    m, rot, pos, eps, cap = 5, 8, 3, 1e-2, 16
    rd = rot if kv_rank else 0
    ldz, ldcq = q_rank + kv_rank + rd, q_rank + 3
    z = g.standard_normal((m, ldz)).astype(np.float32)
    qw, kw = g.standard_normal(max(q_rank, 1)).astype(np.float32), g.standard_normal(max(kv_rank, 1)).astype(np.float32)
    angle = g.standard_normal((cap, rot // 2)).astype(np.float32)
    dev = dict(z=u.dev_f32(z), qw=u.dev_f32(qw), kw=u.dev_f32(kw), cs=u.dev_f32(np.cos(angle)), sn=u.dev_f32(np.sin(angle)), cq=u.zeros_f32(m, ldcq) + 7, c=u.zeros_f32(cap, max(kv_rank, 1)),
               r=u.zeros_f32(cap, rot), pos=torch.tensor([pos], dtype=torch.int32, device="cuda"))
    P = {k: v.data_ptr() for k, v in dev.items()}
    fields = dict(z=P["z"], ldz=ldz, q_rank=q_rank, eps=eps, pos=P["pos"])
    if q_rank:
        fields.update(q_weight=P["qw"], cq=P["cq"], ldcq=ldcq)
    if kv_rank:
        fields.update(kv_rank=kv_rank, rot_dim=rd, kv_weight=P["kw"], ccache=P["c"], rcache=P["r"], ldc=kv_rank, ldr=rot, rope_cos=P["cs"], rope_sin=P["sn"])
    hip.latent_rows_dev(pkg.LatentRows(**fields), m, True)
    z64 = z.astype(np.float64)
    unit = lambda a: a / np.sqrt((a ** 2).mean(1, keepdims=True) + eps)
    if q_rank:
        assert u.rms_error(u.host(dev["cq"])[:, :q_rank], unit(z64[:, :q_rank]) * qw) < F32_TOL and not u.host(dev["cq"])[:, q_rank:].any()
    if kv_rank:
        assert u.rms_error(u.host(dev["c"])[pos:pos + m], unit(z64[:, q_rank:q_rank + kv_rank]) * kw) < F32_TOL
        a, b, cs, sn = z64[:, ldz - rot:ldz - rot // 2], z64[:, ldz - rot // 2:], np.cos(angle[pos:pos + m]), np.sin(angle[pos:pos + m])
        assert u.rms_error(u.host(dev["r"])[pos:pos + m], np.concatenate([a * cs - b * sn, b * cs + a * sn], 1)) < F32_TOL

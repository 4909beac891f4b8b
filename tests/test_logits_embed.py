"""Logits, greedy token and the next position's embedding row in one go (include/bitnet_hip.h section 5: dense_logits_embed), rows as they are, normed and of token pairs, tokens chosen and forced,
tables of fewer rows than there are logits: the same, bit for bit, as the two calls one behind the other."""
import ctypes as C

import numpy as np
import pytest

from tests import stack_util as u

pytestmark = pytest.mark.gpu


class Embedding(C.Structure):
    _fields_ = [("table", C.c_void_p), ("ld", C.c_size_t), ("width", C.c_size_t), ("vocab", C.c_size_t), ("scale", C.c_float), ("eps", C.c_float), ("norm_weight", C.c_void_p), ("pairs", C.c_void_p),
                ("ld_pairs", C.c_size_t), ("buckets", C.c_size_t), ("mul_prev", C.c_uint64), ("mul_cur", C.c_uint64), ("out", C.c_void_p)]


@pytest.mark.parametrize("kind", ["plain", "norm", "pairs"])
@pytest.mark.parametrize("width,rows", [(64, 700), (64, 500), (1540, 651), (4096, 650), (132, 1)])
@pytest.mark.parametrize("forced", [False, True])
def test_logits_and_next_row(hip, pkg, kind, width, rows, forced):
    g, vocab, best, at, buckets = np.random.default_rng([width, rows]), 700, 650, 3, 97
    ld, cols = u.up_to(width, 64), 64
    x = g.standard_normal(cols).astype(np.float32)
    w = u.rounded(g.standard_normal((vocab, cols)))
    w[best] = u.rounded(8 * x)
    table, pairs = u.dev_bf16(u.padded(u.rounded(g.standard_normal((rows, width))), ld)), u.dev_bf16(u.padded(u.rounded(g.standard_normal((buckets + 1, width))), ld))
    norm, xd, wd = u.dev_f32(g.standard_normal(width)), u.dev_f32(x), u.dev_bf16(w)
    history = np.arange(20, 30).astype(np.int32)
    got = []
    for together in (False, True):
        logits, scratch, token, out = u.zeros_f32(vocab), u.zeros_f32(2048), u.dev(np.array([-1], np.int32)), u.zeros_f32(width)
        pos, past, n_forced = u.dev(np.array([at], np.int32)), u.dev(history), u.dev(np.array([at + 1 + forced], np.int32))
        p = [C.c_void_p(t.data_ptr()) for t in (xd, wd, logits, scratch, token, pos, past, n_forced)]
        vi = pkg.VectorInput(x=p[0].value, kind=pkg.IN_PLAIN)
        args = [C.byref(vi), p[1], C.c_size_t(vocab), C.c_size_t(cols), C.c_size_t(cols), *p[2:]]
        if together:
            e = Embedding(table.data_ptr(), ld, width, rows, 0.75, 1e-5, norm.data_ptr() if kind == "norm" else None, pairs.data_ptr() if kind == "pairs" else None, ld, buckets, 31, 17, out.data_ptr())
            assert hip.c.bitnet_hip_embedding_follows(C.byref(e))
            hip._call("dense_logits_embed_dev", *args, C.byref(e), None)
        else:
            hip._call("dense_logits_dev", *args, None)
            if kind == "plain":
                hip.embed_bf16_dev(table, ld, past, out, 1, width, rows, offset=pos, scale=0.75)
            elif kind == "norm":
                hip.embed_norm_bf16_dev(table, ld, past, norm, 1e-5, out, 1, width, rows, offset=pos, scale=0.75)
            else:
                hip.embed_pairs_bf16_dev(table, ld, pairs, ld, buckets, 31, 17, past, out, 1, width, rows, offset=pos, scale=0.75)
        got.append([u.host(t) for t in (logits, token, pos, past, out)])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert got[1][1][0] == best and got[1][2][0] == at + 1 and got[1][3][at + 1] == (history[at + 1] if forced else best)

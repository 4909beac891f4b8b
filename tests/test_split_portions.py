"""A portion's queries behind many keys, the keys of a block shared out to several workgroups (include/bitnet_hip.h section 5: gqa_prefill_scratch): against the same portion with its keys together,
and the definition."""
import pytest

from tests import stack_util as u
from tests.test_mixer_ops import Attention, ChunkAttention, pos_dev

pytestmark = pytest.mark.gpu


def both(hip, t, rows, ld, n, nq):
    outs = [t.new(nq, t.heads * t.vdimp), t.new(nq, t.heads * t.vdimp)]
    size = hip.gqa_prefill_scratch_bytes(t.attn, n, nq)
    scratch = u.zeros_f32(size // 4) + float("nan")
    hip.gqa_prefill_dev(t.attn, rows, ld, n, nq, outs[0], t.heads * t.vdimp)
    hip.gqa_prefill_scratch_dev(t.attn, rows, ld, n, nq, outs[1], t.heads * t.vdimp, scratch, size)
    return outs, size // (4 * nq * t.heads * t.attn.maps * (4 + t.vdimp))


# stretches: two at least, as many as there are CUs for, a last one that is short, none of its own for the first queries of a block, no more than pays
@pytest.mark.parametrize("shape,n,nq,parts", [((4, 2, 24, 40, 2), 300, 1, 3), ((4, 2, 24, 40, 2), 700, 130, 6), ((12, 3, 128, 128, 1), 520, 20, 5), ((20, 1, 64, 100, 2), 640, 64, 5), ((2, 1, 200, 256, 2), 450, 65, 4),
                                              ((8, 2, 96, 64, 1), 400, 300, 4), ((1, 1, 32, 32, 1), 900, 900, 4), ((34, 2, 16, 24, 2), 500, 70, 1), ((8, 2, 96, 64, 1), 128, 3, 1)])
def test_portion_in_stretches(hip, pkg, shape, n, nq, parts):
    t = Attention(pkg, n, *shape, False)
    t.fill(hip, 0, n)
    rows = t.put(t.rows[n - nq:])
    hip.gqa_rows_dev(t.attn, rows, t.ld, False, False, pos_dev(n - nq), nq)
    outs, got = both(hip, t, rows, t.ld, n, nq)
    assert got == (parts if parts > 1 else 0)
    t.check(outs[1], n - nq, 2e-2)
    assert u.rms_error(u.host(outs[1]), u.host(outs[0])) < 4e-3  # one rounding to bf16 each


# heads, kv heads, columns, rotated ones, chunk: chunks that begin inside a stretch, a sink that counts once, gates behind
@pytest.mark.parametrize("shape", [(4, 2, 24, 16, 0), (4, 2, 24, 16, 300), (5, 1, 40, 0, 410), (2, 1, 200, 64, 0)])
@pytest.mark.parametrize("n,nq", [(430, 20), (620, 150)])
def test_chunked_portion_in_stretches(hip, pkg, shape, n, nq):
    t = ChunkAttention(pkg, n, *shape, False)
    t.fill(hip, 0, n)
    rows = t.put(t.rows[n - nq:])
    hip.gqa_rows_dev(t.attn, rows, t.ld, False, False, pos_dev(n - nq), nq)
    t.gated(rows)
    outs, _ = both(hip, t, rows, t.ld, n, nq)
    t.check(outs[1], n - nq, 2e-2)
    assert u.rms_error(u.host(outs[1]), u.host(outs[0])) < 4e-3


def test_room_is_wanted_where_there_are_stretches(hip, pkg):
    """no room, too little of it or room off sixteen bytes is refused where keys are shared out, and none is needed where they are not"""
    t = Attention(pkg, 700, 4, 2, 24, 40, 2, False)
    t.fill(hip, 0, 700)
    rows, out = t.put(t.rows[570:]), t.new(130, 4 * t.vdimp)
    size = hip.gqa_prefill_scratch_bytes(t.attn, 700, 130)
    room = u.zeros_f32(size // 4 + 4)
    for scratch, n in ((None, 0), (None, size), (room, size - 1), (room[1:], size)):
        with pytest.raises(pkg.BitNetHipError, match="scratch of"):
            hip.gqa_prefill_scratch_dev(t.attn, rows, t.ld, 700, 130, out, 4 * t.vdimp, scratch, n)
    assert not u.host(out).any()
    hip.gqa_rows_dev(t.attn, rows, t.ld, False, False, pos_dev(570), 130)
    assert hip.gqa_prefill_scratch_bytes(t.attn, 130, 130) == 0
    hip.gqa_prefill_scratch_dev(t.attn, rows, t.ld, 130, 130, out, 4 * t.vdimp, None, 0)
    want = t.new(130, 4 * t.vdimp)
    hip.gqa_prefill_dev(t.attn, rows, t.ld, 130, 130, want, 4 * t.vdimp)
    assert u.host(want).any() and (u.host(out) == u.host(want)).all()

"""Prompt attention by tiles of 64 keys in one buffer (two maps of 128 columns, 256 columns of two) and in two: one tile to seven, whole and one key past, against the definition in 64 bits."""
import pytest

from test_mixer_ops import Attention, pos_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 65, 128, 129, 192, 256, 257, 449])
@pytest.mark.parametrize("shape", [(3, 1, 128, 128, 2), (2, 1, 256, 256, 2), (2, 1, 256, 256, 1), (4, 2, 128, 128, 1), (4, 2, 96, 112, 1), (4, 2, 64, 128, 2), (4, 2, 32, 48, 2), (4, 2, 64, 64, 1)])
@pytest.mark.parametrize("last", [False, True])
def test_portion_of_tiles(hip, pkg, shape, n, last):
    t = Attention(pkg, n, *shape, False)
    t.fill(hip, 0, n)
    nq = min(n, 17) if last else n
    rows = t.put(t.rows[n - nq:])
    hip.gqa_rows_dev(t.attn, rows, t.ld, False, False, pos_dev(n - nq), nq)
    out = t.new(nq, t.heads * t.vdimp)
    hip.gqa_prefill_dev(t.attn, rows, t.ld, n, nq, out, t.heads * t.vdimp)
    t.check(out, n - nq, 2e-2)  # (rounded queries, keys and outputs, 8 bits each; the weights are pairs)

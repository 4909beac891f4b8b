"""Prompt attention over latent keys: the queries' rotated part by eight elements and one by one (halves that are no multiple of eight, tables off sixteen bytes), tiles around their edges,
against the definition in 64 bits."""
import pytest

import stack_util as u
from test_stack_ops import Latent

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,nq", [(1, 1), (63, 63), (65, 65), (130, 130), (257, 40)])
@pytest.mark.parametrize("shape", [(5, 128, 64, 128, 128), (3, 64, 16, 64, 64), (3, 64, 24, 64, 64), (2, 32, 96, 32, 64), (2, 32, 8, 160, 64), (2, 192, 48, 256, 64)])
@pytest.mark.parametrize("off", [0, 1])
def test_latent_prefill_turns(hip, pkg, shape, L, nq, off):
    t = Latent(pkg, L, nq, *shape, False)
    cos, sin = (u.zeros_f32(a.numel() + off) for a in (t.cos, t.sin))
    cos[off:], sin[off:] = t.cos.flatten(), t.sin.flatten()
    t.attn.rope_cos, t.attn.rope_sin = cos.data_ptr() + 4 * off, sin.data_ptr() + 4 * off
    t.check(t.prefill(hip), 1.5e-2 if L > 1 else 4e-2)  # (rounded queries, keys and outputs, 8 bits each; one key: its rounded score decides its share against the sink)

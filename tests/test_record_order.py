"""Decode attention whose workgroups lie in the order of the records: eight of all heads and queries at a time, up to 32 of those on an XCD.  Members and records around both edges
(records of the capacity that are no multiple of eight, members that fill no chunk), against the definition in 64 bits."""
import numpy as np
import pytest

import stack_util as u
from test_mixer_ops import Attention, pos_dev
from test_stack_ops import Latent

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [60, 64 * 7, 64 * 8 + 1, 64 * 17])
@pytest.mark.parametrize("heads,nq", [(31, 1), (33, 1), (16, 2), (11, 3), (49, 7)])
@pytest.mark.parametrize("f32", [True, False])
def test_latent_records_in_any_order(hip, pkg, heads, nq, L, f32):
    t = Latent(pkg, L, nq, heads, 32, 32, 32, 64, f32)
    t.check(t.decode(hip), 1e-5 if f32 else 1e-4)  # (the f32 sums of 64 + 32 products and of L weights, 24 bits; the query's pairs of bf16, 16 bits)


@pytest.mark.parametrize("n", [100, 128 * 7, 128 * 8 + 1, 128 * 9])
@pytest.mark.parametrize("heads,kv,maps,nq", [(31, 1, 1, 1), (33, 11, 1, 1), (8, 2, 2, 2), (11, 11, 1, 3), (24, 6, 2, 7)])
@pytest.mark.parametrize("f32", [True, False])
def test_records_of_any_size_in_any_order(hip, pkg, heads, kv, maps, nq, n, f32):
    t = Attention(pkg, n, heads, kv, 24, 40, maps, f32)
    rows = t.fill(hip, 0, n)
    scratch = u.zeros_f32(hip.gqa_scratch_bytes(heads, maps, t.vdimp, nq) // 4)
    out = u.zeros_f32(nq, heads * t.vdimp)
    hip.gqa_any_dev(t.attn, rows[n - nq:].contiguous(), t.ld, f32, f32, pos_dev(n - nq), 0, nq, scratch)
    hip.gqa_merge_dev(t.attn, pos_dev(n - nq), 0, nq, scratch, out, heads * t.vdimp, False)
    t.check(out, n - nq, 1e-5 if f32 else 2e-2)  # (bf16: keys and values are rounded to 8 bits behind their norms)


@pytest.mark.parametrize("capacity", [128, 128 * 7, 8192])
@pytest.mark.parametrize("heads,kv,maps", [(24, 6, 1), (40, 2, 1), (16, 8, 2)])
def test_steps_with_records_to_end_at_once(hip, pkg, heads, kv, maps, capacity):
    n = 100
    t = Attention(pkg, n, heads, kv, 64, 64, maps, False)
    t.fill(hip, 0, n - 1)
    k, v = (u.zeros_bf16(*s) for s in ((kv, maps, capacity, t.dimp), (kv, t.vdimp, capacity)))
    k[:, :, :t.cap], v[:, :, :t.cap] = t.keep[3], t.keep[4]
    factor = u.zeros_f32(capacity)
    factor[:t.cap] = t.keep[2]
    t.attn.kcache, t.attn.vcache, t.attn.q_factor, t.attn.capacity = k.data_ptr(), v.data_ptr(), factor.data_ptr(), capacity
    scratch = u.zeros_f32(hip.gqa_scratch_bytes(heads, maps, t.vdimp, 1) // 4)
    scratch.fill_(np.nan)  # (what no workgroup writes is read by none)
    out = u.zeros_f32(1, heads * t.vdimp)
    hip.gqa_step_dev(t.attn, u.dev_f32(t.rows[n - 1]), pos_dev(n - 1), scratch)
    hip.gqa_merge_dev(t.attn, pos_dev(n - 1), 0, 1, scratch, out, heads * t.vdimp, False)
    t.check(out, n - 1, 2e-2)

"""The attention's records merged by the product behind it, lane by lane (include/bitnet_hip.h section 5: gqa_project) and the forms that a
model's steps take by their position: against the merge's own launch, a 64-bit product and steps by themselves."""
import numpy as np
import pytest

from tests import stack_util as u
from tests.test_mixer_ops import pos_dev

pytestmark = pytest.mark.gpu
F32_TOL = 3e-6


# heads, columns of one, rows of the product, extra columns of its matrix; position, chunk, window; records asked for
@pytest.mark.parametrize("heads,vdimp,rows,extra", [(1, 32, 5, 0), (12, 128, 1536, 0), (20, 128, 1030, 64), (3, 160, 70, 32), (4, 1024, 9, 0), (7, 96, 2050, 32), (2, 96, 16500, 0)])
@pytest.mark.parametrize("pos,chunk,window,records", [(0, 0, 0, 1), (127, 0, 0, 2), (128, 0, 0, 2), (511, 0, 0, 4), (512, 0, 0, 5), (1023, 0, 0, 8), (900, 0, 200, 3), (1024, 0, 0, 9),
                                                      (1535, 0, 0, 12), (1500, 1024, 0, 4), (2900, 0, 1100, 10)])
@pytest.mark.parametrize("sink,gate", [(False, None), (True, "head"), (False, "column")])
def test_records_merged_by_lanes(hip, pkg, heads, vdimp, rows, extra, pos, chunk, window, records, sink, gate):
    """what lies in the slots past the position's records is never used"""
    g = np.random.default_rng([heads, vdimp, rows, pos])
    n, first = heads * vdimp, max(pos // chunk * chunk if chunk else 0, pos - window + 1 if window else 0)
    used = (pos - first // 128 * 128) // 128 + 1
    assert used <= records
    rec = np.full((heads, 128, 4 + vdimp), np.nan, np.float32)
    rec[:, :used, 0], rec[:, :used, 1] = 3 * g.standard_normal((heads, used)), g.uniform(0.5, 60.0, (heads, used))
    rec[:, :used, 4:] = g.standard_normal((heads, used, vdimp))
    scratch = u.dev_f32(rec.reshape(-1))
    keep = [u.zeros_f32(64), u.dev_f32(g.standard_normal(heads)), u.dev_f32(g.standard_normal(n))]
    p = [t.data_ptr() for t in keep]
    kw = dict(chunk=chunk, window=window)
    if sink:
        kw["sink"] = p[1]
    if gate:
        kw.update(gate=p[2], ldgate=n, gate_f32=1, gate_columns=int(gate == "column"))
    attn = pkg.Gqa(heads, 1, 1, 32, 32, vdimp, vdimp, 4096, 1e-5, 0.0, 1.0, 0, 0, p[0], p[0], p[0], **kw)
    cols = u.up_to(n, 64) + extra
    ld = u.up_to(cols, 64)
    w, bias, y = u.rounded(g.standard_normal((rows, cols)) / np.sqrt(n)), g.standard_normal(rows).astype(np.float32), u.zeros_f32(rows)
    assert hip.gqa_project_records(attn, cols) == 12
    hip.gqa_project_dev(attn, pos_dev(pos), records, scratch, u.dev_bf16(u.padded(w, ld)), rows, cols, ld, y, bias=u.dev_f32(bias))
    m, l, v = (rec[:, :used, 0].astype(np.float64), rec[:, :used, 1].astype(np.float64), rec[:, :used, 4:].astype(np.float64))
    s = u.host(keep[1]).astype(np.float64) * np.log2(np.e) if sink else np.full(heads, -np.inf)
    top = np.maximum(m.max(1), s)
    e = np.exp2(m - top[:, None])
    out = (e[..., None] * v).sum(1) / ((e * l).sum(1) + np.exp2(s - top))[:, None]
    if gate:
        z = u.host(keep[2]).astype(np.float64)
        out /= 1 + np.exp(-(z.reshape(heads, vdimp) if gate == "column" else z[:heads, None]))
    assert u.rms_error(u.host(y), w[:, :n].astype(np.float64) @ out.reshape(-1) + bias) < F32_TOL


@pytest.mark.parametrize("heads,vdimp,rows,extra,pos", [(1, 32, 5, 0, 0), (12, 128, 1536, 0, 200), (3, 160, 70, 32, 511), (4, 1024, 9, 0, 300), (7, 96, 3100, 32, 130)])
def test_weights_off_sixteen_bytes(hip, pkg, heads, vdimp, rows, extra, pos):
    """gqa_out's own kernel (weights off four bytes), and the lanes' product of weights on eight: as of the same weights on sixteen bytes, up to the order of sums"""
    g = np.random.default_rng([heads, vdimp, rows])
    n, used = heads * vdimp, pos // 128 + 1
    rec = np.full((heads, 128, 4 + vdimp), np.nan, np.float32)
    rec[:, :used, 0], rec[:, :used, 1] = 3 * g.standard_normal((heads, used)), g.uniform(0.5, 60.0, (heads, used))
    rec[:, :used, 4:] = g.standard_normal((heads, used, vdimp))
    scratch, some, gate = u.dev_f32(rec.reshape(-1)), u.zeros_f32(64), u.dev_f32(g.standard_normal(n))
    attn = pkg.Gqa(heads, 1, 1, 32, 32, vdimp, vdimp, 1024, 1e-5, 0.0, 1.0, 0, 0, *[some.data_ptr()] * 3, gate=gate.data_ptr(), ldgate=n, gate_f32=1, gate_columns=1)
    cols = u.up_to(n, 64) + extra
    ld = u.up_to(cols, 64)
    w = u.bf16_bits(u.padded(u.rounded(g.standard_normal((rows, cols)) / np.sqrt(n)), ld)).view(np.int16).reshape(-1)
    on, eight, off = (u.dev(np.concatenate([np.zeros(k, np.int16), w]))[k:] for k in (0, 4, 1))
    assert off.data_ptr() % 16 == 2
    got = []
    for weights in (on, eight, off):
        y = u.zeros_f32(rows)
        hip.gqa_out_dev(attn, pos_dev(pos), used, scratch, weights, rows, cols, ld, y)
        got.append(u.host(y))
    assert np.array_equal(got[1], got[0]) and u.rms_error(got[2], got[0]) < F32_TOL
    with pytest.raises(pkg.BitNetHipError, match="bad arguments"):
        hip.gqa_project_dev(attn, pos_dev(pos), used, scratch, eight, rows, cols, ld, u.zeros_f32(rows))


def test_steps_across_the_forms(pkg, tmp_path):
    """a Lurepel model's steps around 128, 256, 512, 1024 and 1536 keys: as a prompt of all tokens gives them"""
    import importlib

    synth = importlib.import_module("bitnet-rs_amd.synth")
    config = synth.lurepel_config("1b", 2)
    config["vocab"] = 512
    synth.write_lurepel(str(tmp_path), config)
    m = pkg.open_model(str(tmp_path), max_pos=2048)
    tokens = np.random.default_rng(5).integers(0, 512, 1550).astype(np.int32)
    for at in (126, 254, 510, 1022, 1534):
        m.reset()
        m.feed(tokens[:at + 5])
        m.prefill(at, with_logits=False, digits=2)
        m.run(5)
        got = m.last_logits().copy()
        m.reset()
        m.feed(tokens[:at + 5])
        m.prefill(at + 5, with_logits=True, digits=2)
        assert u.rms_error(got, m.last_logits()) < 2e-2, at


@pytest.mark.parametrize("heads,kv_heads,dim", [(3, 1, 288), (28, 7, 128)])
def test_steps_of_other_heads_across_the_forms(pkg, tmp_path, heads, kv_heads, dim):
    """heads of 288 columns, whose records come from gqa_any, and 3584 columns, whose records past eight take a launch of their own: the same, a prompt of the last five tokens against steps"""
    config = u.lurepel([u.chunk_layer(heads=heads, kv_heads=kv_heads, dim=dim, scale=0.05, chunk=4096, dims=64)], width=112, vocab=150)
    path = u.save_model(str(tmp_path), config, u.random_tensors(config, 8))
    m = pkg.open_model(path, max_pos=2048)
    tokens = np.random.default_rng(6).integers(0, 150, 1550).astype(np.int32)
    for at in (126, 254, 510, 1022, 1534):
        m.reset()
        m.feed(tokens[:at + 5])
        m.prefill(at, with_logits=False, digits=2)
        m.run(5)
        got = m.last_logits().copy()
        m.reset()
        m.feed(tokens[:at + 5])
        m.prefill(at + 5, with_logits=True, digits=2)
        assert u.rms_error(got, m.last_logits()) < 2e-2, at

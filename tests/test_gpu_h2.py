"""The encoder's products on split fp16 activations (csrc/gemm_h2.hip) at the
edges of their tiles, against the float64 restatement of the encoder: one row
(the few-row kernel), row counts around 32, 64 and 128, a batch in
micro-batches, widths that leave the column tiles partly empty; and models
whose weights or gains keep them on the three-term products."""
import numpy as np
import pytest

from ai_amd import _native as N
from ai_amd import gemma as G
from ai_amd import synth as S
from test_oracle import f64_encoder

pytestmark = pytest.mark.gpu

# float32 sums of at most 512 terms through two layers: every other layer
# test of this suite holds hidden rows to 1e-5
REL = 1e-5


def shape(hidden, ffn):
    return S.ModelShape(hidden_size=hidden, num_hidden_layers=2, num_attention_heads=2, num_key_value_heads=1,
                        intermediate_size=ffn, vocab_size=300, sliding_window=64, sliding_window_pattern=2,
                        max_tokens=512, dense_out=[])


def weights(sh, edit=None):
    ws = {}
    for name, shp, kind in S.weight_specs(sh):
        w = S.make_weight(name, shp, kind, 77)
        ws[name] = S.bf16_to_f32(w) if kind == "m" else w
    if edit:
        edit(ws)
    return ws


def check(sh, ws, lengths):
    lengths = np.array(lengths, np.int32)
    r = np.random.default_rng(5)
    ids = np.zeros((len(lengths), int(lengths.max())), np.int32)
    for b, n in enumerate(lengths):
        ids[b, :n] = r.integers(3, sh.vocab_size, n)
    with N.Context(0) as ctx:
        m = G.Model(sh, ctx)
        for name, w in ws.items():
            m.set_weight(name, w)
        m.finalize()
        got = m.encode_ids(ids, lengths)
        m.close()
    states = []
    f64_encoder(sh, ws, ids, lengths, states=states)
    want = np.concatenate([s[-1] for s in states])
    rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert rel.max() <= REL, rel.max()


@pytest.mark.parametrize("hidden,ffn", [(256, 96), (512, 288)])
@pytest.mark.parametrize("lengths", [[1], [31], [33], [64, 1], [129], [300, 7, 210], [257] * 9])
def test_split_products_at_tile_edges(hidden, ffn, lengths):
    sh = shape(hidden, ffn)
    check(sh, weights(sh), lengths)


def tiny_weight(ws):  # 2^-60 beside values near 0.1: no power of two makes both exact in fp16
    ws["layers.0.self_attn.o_proj.weight"][3, 5] = 2.0 ** -60


def outlier_gain(ws):  # one gain 1 000 times the others
    ws["layers.1.pre_feedforward_layernorm.weight"][7] = 1000.0


@pytest.mark.parametrize("edit", [tiny_weight, outlier_gain])
def test_models_outside_the_split_range(edit):
    sh = shape(256, 96)
    check(sh, weights(sh, edit), [40, 3])

"""The dtype=f32 path (the reference's BackendOptions::f32, runtime/crates/laya-core/src/backend.rs:
25-27, checked upstream by laya-mlx/tests/parity.rs:54-65) against the oracle, which is f32 too.

Both sides hold f32 weights and sum in f32, so the gates here are tighter than the 16-bit path's:
hidden states within 1e-3 relative per position, logits within 1e-3 absolute, pooled rows within
1e-3 relative, answer probabilities within 1e-4, every decision identical. The differences left
are the products' operands (each a pair of f16, to 2^-23 of its value, without the product of the
two low parts, 2^-22 of a term), summation order and the erf and exp implementations.
test_f32_tile_edges holds blocks of layers to float64 at 2e-6.
"""
from __future__ import annotations

import json
from pathlib import Path

import numpy as np
import pytest

from oracle import oracle as O
from oracle.torch_ref import TorchOracle
from sys1rust_amd.backend import DEFAULT_TUNING, HipBackend, synth_checkpoint
from sys1rust_amd.decode import ActHead, decode_answers
from sys1rust_amd.workloads import AGENT, MODERNBERT_LARGE, Batch, workload

from gates import decisive_checkpoint, hidden_rel, random_batch, say

pytestmark = pytest.mark.gpu

GOLDEN = Path(__file__).resolve().parent / "golden"
HIDDEN_REL_F32 = 1e-3
LOGIT_ABS_F32 = 1e-3
POOLED_REL_F32 = 1e-3
PROB_ABS_F32 = 1e-4


def gate_f32(m, b, ref_hidden, lg_ref, pl_ref, act, tag, padding=True):
    hid = m.encoder_hidden(b).reshape(b.n, b.len, -1)
    rel = hidden_rel(hid, ref_hidden, b, padding=padding)
    out = m.forward(b)
    dl = float(np.abs(out.logits - lg_ref).max()) if b.kmax else 0.0
    pg, pr = out.pooled.reshape(b.n, -1), pl_ref.reshape(b.n, -1)
    dp = float((np.linalg.norm(pg - pr, axis=-1) / np.linalg.norm(pr, axis=-1)).max())
    dprob = dact = 0.0
    same = True
    if b.kmax:  # answers need answer slots
        a = decode_answers(out.logits, b.kmax, b.marker_count, b.qtype, pooled=out.pooled, act_head=act)
        r = decode_answers(lg_ref, b.kmax, b.marker_count, b.qtype, pooled=pl_ref, act_head=act)
        dprob = max((float(np.abs(x["probabilities"] - y["probabilities"]).max()) for x, y in zip(a, r)
                     if len(y["probabilities"])), default=0.0)
        dact = max(abs(x["act_probability"] - y["act_probability"]) for x, y in zip(a, r))
        same = all(x.get("choice") == y.get("choice") for x, y in zip(a, r))
    say(f"{tag}: hidden rel {rel:.2e}, logits {dl:.2e}, pooled rel {dp:.2e}, probabilities {dprob:.2e}, "
        f"act {dact:.2e}, choices identical {same}")
    assert rel <= HIDDEN_REL_F32, (tag, rel)
    assert dl <= LOGIT_ABS_F32, (tag, dl)
    assert dp <= POOLED_REL_F32, (tag, dp)
    assert dprob <= PROB_ABS_F32 and dact <= PROB_ABS_F32, (tag, dprob, dact)
    assert same, tag


@pytest.fixture(scope="module")
def small():
    z = np.load(GOLDEN / "golden_small.npz")
    cfg = json.loads(str(z["encoder_config"]))
    agent = json.loads(str(z["agent_config"]))
    st = synth_checkpoint(json.dumps(cfg), json.dumps(agent), int(z["seed"]), int(z["scorer_width"]), 2, True)
    b = Batch(int(z["n"]), int(z["len"]), int(z["kmax"]), z["input_ids"], z["attention_mask"], z["seq_lens"],
              z["marker_pos"], z["marker_count"], z["qtype"])
    return cfg, agent, st, b


@pytest.mark.parametrize("settings", ["", "mask=bool,dense_upto=0", "band=1,fuserope", DEFAULT_TUNING])
def test_f32_small_model_matches_the_oracle(small, settings):
    """The golden batch (3 ragged rows, window 16) at every position, padding included, and the
    forward's logits, pooled rows and answers, under several mask paths."""
    cfg, agent, st, b = small
    spec = ",".join(x for x in [settings, "dtype=f32"] if x)
    m = HipBackend(st, json.dumps(cfg), json.dumps(agent), settings=spec)
    assert m.name() == "hip(gfx950,f32)"
    assert m.active_kernels() == []  # the plain f32 kernels only
    o = O.Oracle(st, cfg, agent, settings=settings)
    ref = o.encoder_hidden(b)
    lg, pl = o.forward(b, ref)
    gate_f32(m, b, ref, lg, pl, ActHead.from_weights(o.w), f"f32 small {settings[:30]!r}")
    m.close()


def test_f32_short_rows_and_no_markers(small):
    """Rows of 1, 3 and 9 tokens, and a batch without answer markers (kmax 0)."""
    cfg, agent, st, _ = small
    lens, L = [1, 3, 9], 9
    rng = np.random.default_rng(7)
    ids = rng.integers(5, 1000, size=(3, L)).astype(np.uint32)
    am = np.zeros((3, L), np.uint32)
    for r, n in enumerate(lens):
        am[r, :n] = 1
        ids[r, n:] = 1002
    o = O.Oracle(st, cfg, agent)
    act = ActHead.from_weights(o.w)
    m = HipBackend(st, json.dumps(cfg), json.dumps(agent), settings="dtype=f32")
    for kmax, mp, mc in [(2, [[0, 0], [2, 0], [4, 8]], [0, 1, 2]), (0, None, [0, 0, 0])]:
        b = Batch(3, L, kmax, ids.reshape(-1), am.reshape(-1), np.array(lens, np.uint64),
                  np.array(mp, np.uint32).reshape(-1) if mp else np.zeros(0, np.uint32), np.array(mc, np.uint64),
                  np.array([0, 1, 2], np.uint32))
        ref = o.encoder_hidden(b)
        lg, pl = o.forward(b, ref)
        gate_f32(m, b, ref, lg, pl, act, f"f32 short rows kmax={kmax}")
    m.close()


@pytest.mark.parametrize("layers", [0, 1])
def test_f32_encoder_depths(small, layers):
    """An encoder without layers (the embeddings, the final norm and the head), and one with one."""
    cfg, agent, _, b = small
    cfg = dict(cfg, num_hidden_layers=layers)
    st = synth_checkpoint(json.dumps(cfg), json.dumps(agent), 9, 256, 2, True)
    o = O.Oracle(st, cfg, agent)
    ref = o.encoder_hidden(b)
    lg, pl = o.forward(b, ref)
    for settings in ("dtype=f32", DEFAULT_TUNING + ",dtype=f32"):
        m = HipBackend(st, json.dumps(cfg), json.dumps(agent), settings=settings)
        gate_f32(m, b, ref, lg, pl, ActHead.from_weights(o.w), f"f32 layers={layers} {settings[-30:]!r}")
        m.close()


def test_f32_modernbert_large_512_tokens():
    """The 28-layer ModernBERT-large shape over a 512-token state with one question, and a padded
    600-position batch at every position (chunked local attention for the padding), against the
    oracle's torch f32 restatement on the GPU."""
    st = synth_checkpoint(json.dumps(MODERNBERT_LARGE), json.dumps(AGENT), seed=2024, scorer_width=1024)
    m = HipBackend(st, json.dumps(MODERNBERT_LARGE), json.dumps(AGENT), settings="dtype=f32")
    o = O.Oracle(st, MODERNBERT_LARGE, AGENT)
    t = TorchOracle(o, "cuda")
    act = ActHead.from_weights(o.w)
    b = workload("state512_1q", seed=5)
    say(f"f32 large: n={b.n} len={b.len} T={b.total_tokens()}")
    ref = t.encoder_hidden(b)
    lg, pl = t.forward(b, ref)
    gate_f32(m, b, ref, lg, pl, act, "f32 large state512_1q")
    lens, L = [600, 300, 20], 600
    rng = np.random.default_rng(17)
    ids = rng.integers(5, 50000, size=(3, L)).astype(np.uint32)
    am = np.zeros((3, L), np.uint32)
    for r, n in enumerate(lens):
        am[r, :n] = 1
        ids[r, n:] = 50283
    bp = Batch(3, L, 0, ids.reshape(-1), am.reshape(-1), np.array(lens, np.uint64), np.zeros(0, np.uint32),
               np.zeros(3, np.uint64), np.zeros(3, np.uint32))
    rel = hidden_rel(m.encoder_hidden(bp).reshape(3, L, -1), t.encoder_hidden(bp), bp, padding=True)
    say(f"f32 large padded 600: hidden rel at every position {rel:.2e}")
    assert rel <= HIDDEN_REL_F32, rel
    m.close()


def test_f32_mmbert_golden_batch():
    """The mmBERT-base shape (hidden 768, 12 heads, GeGLU 1152) on its golden fixture's batch,
    against the oracle at every position, padding included."""
    z = np.load(GOLDEN / "golden_mmbert.npz")
    cfg = json.loads(str(z["encoder_config"]))
    agent = json.loads(str(z["agent_config"]))
    st = synth_checkpoint(json.dumps(cfg), json.dumps(agent), int(z["seed"]), int(z["scorer_width"]), 2, True)
    b = Batch(int(z["n"]), int(z["len"]), int(z["kmax"]), z["input_ids"], z["attention_mask"], z["seq_lens"],
              z["marker_pos"], z["marker_count"], z["qtype"])
    m = HipBackend(st, json.dumps(cfg), json.dumps(agent), settings="dtype=f32")
    o = O.Oracle(st, cfg, agent)
    ref = o.encoder_hidden(b)
    lg, pl = o.forward(b, ref)
    gate_f32(m, b, ref, lg, pl, ActHead.from_weights(o.w), "f32 mmbert golden")
    m.close()


@pytest.mark.parametrize("case", ["golden_small", "golden_large", "golden_mmbert"])
def test_f32_against_the_independent_fixtures(case):
    """The f32 option straight against the golden fixtures written by transformers'
    ModernBertModel (hidden states) and torch's TransformerEncoderLayer head and scorer (logits,
    pooled rows), at the tolerances the oracle itself meets against them."""
    z = np.load(GOLDEN / f"{case}.npz")
    cfg = json.loads(str(z["encoder_config"]))
    agent = json.loads(str(z["agent_config"]))
    st = synth_checkpoint(json.dumps(cfg), json.dumps(agent), int(z["seed"]), int(z["scorer_width"]), 2, True)
    b = Batch(int(z["n"]), int(z["len"]), int(z["kmax"]), z["input_ids"], z["attention_mask"], z["seq_lens"],
              z["marker_pos"], z["marker_count"], z["qtype"])
    m = HipBackend(st, json.dumps(cfg), json.dumps(agent), settings="dtype=f32")
    hid = m.encoder_hidden(b).reshape(b.n, b.len, -1)
    sel = z["hidden_sel"]
    g = hid[sel[:, 0], sel[:, 1]]
    rel = float((np.linalg.norm(g - z["hidden"], axis=-1) / np.linalg.norm(z["hidden"], axis=-1)).max())
    out = m.forward(b)
    dl = float(np.abs(out.logits - z["logits"]).max())
    pg, pr = out.pooled.reshape(b.n, -1), z["pooled"].reshape(b.n, -1)
    dp = float((np.linalg.norm(pg - pr, axis=-1) / np.linalg.norm(pr, axis=-1)).max())
    say(f"f32 {case} against the fixture: hidden rel {rel:.2e}, logits {dl:.2e}, pooled rel {dp:.2e}")
    assert rel < 1e-4 and dl < 1e-5 and dp < 1e-4, (rel, dl, dp)
    m.close()


def test_f32_random_batches(small):
    """Six of the seeded random batches (ragged rows of 1-300 tokens, 0-6 answer slots) on the
    decisive-scorer checkpoint, every position of encoder_hidden included."""
    cfg, agent, st, _ = small
    st = decisive_checkpoint(st)
    m = HipBackend(st, json.dumps(cfg), json.dumps(agent), settings="dtype=f32")
    o = O.Oracle(st, cfg, agent)
    act = ActHead.from_weights(o.w)
    rng = np.random.default_rng(20261202)
    for case in range(6):
        b = random_batch(rng, cfg["vocab_size"], cfg["pad_token_id"])
        ref = o.encoder_hidden(b)
        lg, pl = o.forward(b, ref)
        gate_f32(m, b, ref, lg, pl, act, f"f32 random {case} n={b.n} len={b.len} kmax={b.kmax}")
    m.close()


# Rows at the edges of the f32 kernels' tiles, alone and in batches: 32, 64 and 128 rows of a product,
# 32-key tiles and 32- to 128-query tiles of attention; a window of 32 keys on each side; more answer
# slots than tokens. 90 tiles of 128 queries (x 8 heads) take one wave per 32 queries, and 8990 rows
# 64 x 128 tiles in every product, the residual ones of width 512 among them; the last tiles hold 1, 33, 97
# and 128 queries. 600 rows of 9 take 64-query tiles.
EDGES = [([1], 0), ([31], 1), ([33, 64], 2), ([65, 1, 32], 3), ([127, 129, 128], 2), ([193], 3), ([600] * 9 + [37], 4),
         ([3, 5], 9), ([129, 161, 225, 256, 128] * 10, 2)]
# A product of K terms is off by at most 1.7e-7 of its result's norm (K up to 2048 here: operands to 2^-23,
# products to 2^-21, f32 sums); twenty of them in quadrature 8e-7, and the worst of some thousand rows
# about twice that. One weight matrix of one layer cut to a single f16 moves a row by 8e-6 or more.
REL_F64 = 2e-6


@pytest.mark.parametrize("lens,kmax", EDGES)
def test_f32_tile_edges(lens, kmax):
    """Every position, pooled row and logit against float64, with weights of 24 significant bits."""
    from gates import f32_checkpoint
    from oracle.oracle import Oracle
    from sys1rust_amd.workloads import collate, small_config

    cfg = small_config(layers=3, vocab=1024, local_attention=64)
    cfg["pad_token_id"] = 1002
    rng = np.random.default_rng(sum(lens) + kmax)
    items = []
    for L in lens:
        markers = sorted(rng.integers(0, L, kmax).tolist())
        items.append((rng.integers(0, 1000, L).tolist(), markers, int(rng.integers(0, 3))))
    b = collate(items, pad_id=1002)
    st = f32_checkpoint(synth_checkpoint(json.dumps(cfg), json.dumps(AGENT), seed=5, scorer_width=256), cfg, AGENT)
    settings = DEFAULT_TUNING + ",dtype=f32"
    m = HipBackend(st, json.dumps(cfg), json.dumps(AGENT), settings=settings, device=0)
    o = TorchOracle(Oracle(st, cfg, AGENT, settings=DEFAULT_TUNING), "cuda").double()
    ref = o.encoder_hidden(b)
    lg, pl = o.forward(b, ref)
    hid = m.encoder_hidden(b).reshape(b.n, b.len, -1)
    out = m.forward(b)
    m.close()
    rel = [hidden_rel(hid, ref, b, padding=True), 0.0]
    pg, pr = out.pooled.reshape(b.n, -1), pl.reshape(b.n, -1)
    rel[1] = float((np.linalg.norm(pg - pr, axis=-1) / np.linalg.norm(pr, axis=-1)).max())
    real = (np.arange(max(kmax, 1))[None, :kmax] < np.asarray(b.marker_count).astype(int)[:, None]).reshape(-1)
    dl = float(np.abs(out.logits - lg)[real].max()) if real.any() else 0.0
    say(f"f32 rows {lens[:5]} x {len(lens)} slots {kmax}: hidden, pooled rel {rel}, logits {dl:.2e} of {np.abs(lg[real]).max() if real.any() else 0:.2f}")
    assert max(rel) <= REL_F64 and dl <= REL_F64, (rel, dl)  # logits are below 1


def _rescaled(st: bytes, cfg: dict, span: int, norm: int, gate: int) -> bytes:
    """The same model in exact arithmetic, its operands spread over 2 * span powers of two around 2^norm
    and 2^gate: channel k of mlp_norm times 2^e_k and column k of Wi divided by it, gate row j of Wi times
    2^f_j and column j of Wo divided by it."""
    import struct

    n = struct.unpack("<Q", st[:8])[0]
    header, out = json.loads(st[8:8 + n]), bytearray(st)
    rng = np.random.default_rng(8)

    def scale(name, s):
        a, z = (8 + n + o for o in header[name]["data_offsets"])
        assert header[name]["dtype"] == "BF16"
        w = (np.frombuffer(bytes(out[a:z]), np.uint16).astype(np.uint32) << 16).view(np.float32)
        w = (w.reshape(header[name]["shape"]) * s.astype(np.float32)).reshape(-1)
        out[a:z] = (w.view(np.uint32) >> 16).astype(np.uint16).tobytes()

    inter = cfg["intermediate_size"]
    for l in range(cfg["num_hidden_layers"]):
        p = f"encoder.layers.{l}.mlp"
        e = 2.0 ** (norm + rng.integers(-span, span + 1, cfg["hidden_size"]))
        f = 2.0 ** (gate + rng.integers(-span, span + 1, inter))
        scale(p + "_norm.weight", e)
        scale(p + ".Wi.weight", np.concatenate([np.ones(inter), f])[:, None] / e[None, :])
        scale(p + ".Wo.weight", 1.0 / f[None, :])
    return bytes(out)


@pytest.mark.parametrize("span,norm,gate", [(6, 0, 0), (10, 0, 0), (6, -100, 0), (6, 70, 0), (6, 0, 80), (6, 0, -100)])
def test_f32_wide_operand_range(span, norm, gate):
    """The split operands keep their precision over a wide range of magnitudes: a model whose MLP
    operands are spread over 2^12 and 2^20, or lie around a far power of two, gives the plain model's results. Each operand is held to 2^-23
    of its value either way, a product of two to 2^-21 (5e-7), and a sum of K = 1024 rounds to at most
    K 2^-24, typically its root (2e-6); three layers of two such products, doubled for the two models:
    2e-5 relative. An operand rounded to one f16 would be off by 2e-4 or more."""
    from sys1rust_amd.workloads import collate, small_config

    cfg = small_config(layers=3, vocab=1024)
    cfg["pad_token_id"] = 1002
    rng = np.random.default_rng(3)
    b = collate([(rng.integers(0, 1000, L).tolist(), [1, L // 2], 0) for L in (70, 200, 33)], pad_id=1002)
    st = synth_checkpoint(json.dumps(cfg), json.dumps(AGENT), seed=6, scorer_width=256)
    outs = []
    for image in (st, _rescaled(st, cfg, span, norm, gate)):
        m = HipBackend(image, json.dumps(cfg), json.dumps(AGENT), settings=DEFAULT_TUNING + ",dtype=f32", device=0)
        outs.append((m.encoder_hidden(b), m.forward(b)))
        m.close()
    rel = [float(np.linalg.norm(x - y) / np.linalg.norm(x)) for x, y in
           ((outs[0][0], outs[1][0]), (outs[0][1].pooled, outs[1][1].pooled), (outs[0][1].logits, outs[1][1].logits))]
    say(f"f32 operands over 2^{2 * span} around 2^{norm}, 2^{gate}: hidden, pooled, logits rel {rel}")
    assert max(rel) <= 2e-5, rel


@pytest.mark.parametrize("rows,length", [(3, 33), (6, 97), (24, 97), (70, 130)])
def test_f32_nonfinite_keys_stay_in_their_window(rows, length):
    """A token whose value is NaN, within and at both sides of the 32-key tiles (one local layer, window
    16; 32-, 64- and 128-query work tiles): the queries that see it get no finite result, and every
    other one the same bits as with any other token in its place."""
    from gates import local_model, with_embedding
    from sys1rust_amd.workloads import Batch

    cfg, agent, st = local_model()
    W = cfg["local_attention"] // 2
    rng = np.random.default_rng(rows)
    ids = rng.integers(10, 1000, (rows, length)).astype(np.uint32)
    at = rng.integers(0, length, rows)
    at[:3] = (0, min(31, length - 1), length - 1)

    def batch(token):
        x = ids.copy()
        x[np.arange(rows), at] = token
        return Batch(rows, length, 0, x.reshape(-1), np.ones(x.size, np.uint32), np.full(rows, length, np.uint64),
                     np.zeros(0, np.uint32), np.zeros(rows, np.uint64), np.zeros(rows, np.uint32))

    m = HipBackend(with_embedding(st, 7, np.nan), json.dumps(cfg), json.dumps(agent), settings="dtype=f32", device=0)
    say(f"f32 NaN keys in {rows} rows of {length}")
    plain, nan = (m.encoder_hidden(batch(t)).reshape(rows, length, -1) for t in (8, 7))
    sees = np.abs(np.arange(length)[None, :] - at[:, None]) <= W
    changed = (plain != nan).any(-1)
    assert int((changed & ~sees).sum()) == 0
    assert int((np.isfinite(nan).all(-1) & sees).sum()) == 0
    m.close()

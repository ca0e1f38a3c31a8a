"""Layered models (Nerenex; for whole models Safolorn, Segetar and Fororax too, see test_safolorn_gpu.py, test_segetar_gpu.py and
test_fororax_gpu.py for their mechanisms) on the device against the plain oracle of tests/layered_oracle.py: every mechanism alone, prompts,
portions and decoding, unequal batches, reuse of pages and slots, window edges with a key that stands out, and greedy generation
through the engine loop.  Models are small and random; none of their numbers come from a checkpoint."""
import json
import os
import subprocess

import numpy as np
import pytest

from tests import layered_gen as G
from tests import layered_oracle as L
from tests.tile_sizes import FEW_ROWS, SIZES, sizes_that_ran

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BIN = os.path.join(ROOT, "ferrum-infer-rs_amd", "bin")
# rms over the vocabulary of the difference, relative to the rms of the logits: rounding only
TOL = {"float32": 3e-5, "bfloat16": 4e-2}
DTYPES = ["float32", "bfloat16"]


@pytest.fixture(scope="module")
def pkg():
    import torch  # noqa: F401  (ahead of the library: imported later, torch finds no device, and other modules' tests need it)
    import __graft_entry__ as ge
    p = ge.load_package()
    p.load_library()
    return p


@pytest.fixture(scope="module")
def cases(tmp_path_factory):
    """name → (config, weights, checkpoint directory)"""
    made = {}

    def get(name):
        if name not in made:
            cfg = G.CONFIGS[name]
            w = G.weights(cfg, G.SEEDS.get(name, 11 + len(made)))
            made[name] = (cfg, w, G.write_checkpoint(tmp_path_factory.mktemp(name), cfg, w))
        return made[name]
    return get


def load(pkg, path, dtype, tokens=512, seqs=4, slots=0, blocks=None, max_len=None):
    return pkg.HipModel.from_checkpoint(path, kv_num_blocks=blocks or (tokens + 15) // 16 + seqs, max_seqs=seqs, max_tokens=max(tokens, seqs),
                                        max_seq_len=max_len or tokens, dtype=dtype, state_slots=slots)


def rel(got, want):
    """Worst row: rms difference over rms of all wanted rows."""
    want = np.asarray(want, np.float64)
    d = np.sqrt(np.mean((np.asarray(got, np.float64) - want) ** 2, axis=-1))
    return float(np.max(d) / np.sqrt(np.mean(want ** 2)))


def feed(m, seq, tokens, cuts):
    """Logits of every token of one sequence fed in portions of the given sizes (the last size repeats)."""
    out, at, i = [], 0, 0
    while at < len(tokens):
        n = min(cuts[min(i, len(cuts) - 1)], len(tokens) - at)
        out.append(m.forward_rows([(seq, tokens[at:at + n], at)], list(range(n))))
        at += n
        i += 1
    return np.concatenate(out)


def toks(cfg, n, seed):
    return np.random.default_rng(seed).integers(0, cfg["vocab"], n).astype(np.uint32)


# ── each mechanism alone ──────────────────────────────────────────────────────────────────────────────────────────────────
def one_layer(layer, width=72, vocab=50, mult=1.0, **kw):
    return G.config(width, vocab, [layer], mult=mult, **kw)


def taps_of(pkg, tmp_path, cfg, w, dtype, tokens):
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype, tokens=max(512, len(tokens)))
    m.enable_taps()
    m.forward_rows([(1, tokens, 0)], [len(tokens) - 1])
    return m.read_taps(len(tokens))


@pytest.mark.parametrize("dtype", DTYPES)
def test_pair_embedding_across_portions(pkg, tmp_path, dtype):
    """With residual factor 0 the stream stays the embedding: the pair's row for every token, the extra row for the first one, and the
    previous token carried over portion borders, decode steps and a released sequence."""
    cfg = one_layer(G.recurrent(24, 2, 2), mult=0.0, buckets=89, mul_prev=1000003, mul_cur=77)
    w = G.weights(cfg, 3)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype)
    m.enable_taps()
    t = toks(cfg, 23, 5)
    want = L.embed(t, w["embed"].astype(np.float64), w["bigram"].astype(np.float64), 89, 1000003, 77)
    for seq, cuts in ((1, [23]), (2, [1, 2, 7, 1]), (3, [5, 1, 1, 4, 1])):
        at = 0
        while at < len(t):
            n = min(cuts.pop(0) if cuts else 3, len(t) - at)
            m.forward_rows([(seq, t[at:at + n], at)], [])
            assert np.abs(m.read_taps(n)[0] - want[at:at + n]).max() < 1e-6
            at += n
        m.release(seq)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,n", [(1030, 9), (1056, 40), (2044, 17), (2052, 520), (4100, 5)])
def test_rows_of_several_quads_a_thread(pkg, tmp_path, dtype, width, n):
    """Gated branches, normed and added, in rows that a thread holds two or four pieces of, or none."""
    cfg = G.config(width, 50, [G.attention(2, 8, 4, 8, 16, 24, 7, ff=20), G.recurrent(24, 2, 2, ff=33)])
    t, taps = toks(cfg, n, 6), []
    w = G.weights(cfg, 19)
    L.forward(cfg, w, t, taps)
    assert rel(taps_of(pkg, tmp_path, cfg, w, dtype, t), taps) < TOL[dtype]


ENDS = {"nerenex": lambda w: G.config(w, 50, [G.recurrent(24, 2, 2, ff=33), G.attention(2, 8, 4, 8, 16, 24, 7)]),
        "nerenex with a feed-forward": lambda w: G.config(w, 50, [G.attention(2, 8, 4, 8, 16, 24, 7), G.recurrent(24, 2, 2, ff=33)]),
        "safolorn": lambda w: G.safolorn(w, 50, 12, [G.sink_attention(2, 8, 4, 8, 24, mlp=G.glu(30, 0.7))]),
        "segetar": lambda w: G.segetar(w, 50, [G.scan(24, 2, 1, 2, mlp=G.dense(30))]),
        "a loop behind a layer": lambda w: G.segetar(w, 50, [G.scan(24, 2, 1, 2, mlp=G.dense(30)), G.scan(16, 2, 1, 2)], (1, 2, 2)),
        "a loop": lambda w: G.segetar(w, 50, [G.scan(24, 2, 1, 2, mlp=G.dense(30)), G.scan(16, 2, 1, 2)], (0, 1, 2)),
        "fororax": lambda w: G.fororax(w, 50, [G.far_attention(2, 1, 8, 8, mlp=G.identity_experts(3, 1, 2, 9, 33))])}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [72, 45, 2056])
@pytest.mark.parametrize("name", list(ENDS))
def test_norms_of_the_first_layer_and_of_the_head(pkg, tmp_path, name, width, dtype):
    """Steps whose rows all go to the head, which the last update norms, against the same steps with listed rows, which the head norms itself: numbers of the format that differ
    by their last place where 32-bit sums do, so logits by no more than two of its roundings; and both against the oracle.  Rows of one piece a thread, of none and of several."""
    cfg = ENDS[name](width)
    w, t = G.weights(cfg, 23), toks(cfg, 9, 8)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype)
    got = [np.concatenate([m.unified_forward([(s, t[i:i + 1], i, True) for s in (1, 2)], want_logits=True)[1] for i in range(len(t))])]
    got.append(np.concatenate([m.forward_rows([(s, t[i:i + 1], i) for s in (3, 4)], [0, 1]) for i in range(len(t))]))
    assert rel(got[0], got[1]) < {"float32": 2e-6, "bfloat16": 2.0 ** -7}[dtype]
    assert rel(got[0], np.repeat(L.forward(cfg, w, t), 2, axis=0)) < TOL[dtype]


ATTN = [G.attention(3, 20, 6, 36, 44, 52, 9, base=300.0), G.attention(16, 32, 16, 32, 32, 64, 40), G.attention(5, 64, 34, 17, 33, 130, 25, scale=0.3),
        G.attention(1, 5, 2, 3, 4, 7, 2), G.attention(33, 16, 8, 24, 20, 385, 64), G.attention(2, 130, 70, 140, 16, 520, 30)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("i", range(len(ATTN)))
def test_latent_attention_alone(pkg, tmp_path, dtype, i):
    cfg = one_layer(ATTN[i])
    w, t = G.weights(cfg, 20 + i), toks(cfg, 70, 6)
    taps = []
    L.forward(cfg, w, t, taps)
    assert rel(taps_of(pkg, tmp_path, cfg, w, dtype, t), taps) < (1e-5 if dtype == "float32" else 3e-2)


REC = [G.recurrent(66, 3, 3), G.recurrent(64, 1, 4), G.recurrent(40, 5, 1), G.recurrent(96, 2, 7)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("i", range(len(REC)))
def test_recurrence_alone(pkg, tmp_path, dtype, i):
    """200 tokens: several scan chunks, decays from near 0 to near 1."""
    cfg = one_layer(REC[i])
    w, t = G.weights(cfg, 30 + i), toks(cfg, 200, 7)
    taps = []
    L.forward(cfg, w, t, taps)
    assert rel(taps_of(pkg, tmp_path, cfg, w, dtype, t), taps) < (1e-5 if dtype == "float32" else 2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,blocks,conv,rows", [(96, 3, 1, 1), (128, 1, 2, 15), (256, 2, 4, 16), (200, 2, 3, 17), (129, 1, 4, 33), (32, 1, 5, 17)])
def test_recurrence_a_token_at_a_time(pkg, tmp_path, dtype, width, blocks, conv, rows):
    """Sequences from their first token on, longer than the convolution and at unequal positions: blocks of 32, 64 and 128 channels (one launch) and of more, 1 to 4 taps and 5,
    rows that end on either side of a tile.  Logits round as those of whole models do; the slots were used before."""
    cfg = one_layer(G.recurrent(width, blocks, conv))
    w, n = G.weights(cfg, 34), 7
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype, seqs=rows)
    for turn in range(2):
        t = [toks(cfg, n, 40 + 64 * turn + i) for i in range(rows)]
        got = [[] for _ in t]
        for s in range(n + 2):
            on = [i for i in range(rows) if 0 <= s - i % 3 < n]
            for i, lg in zip(on, m.forward_rows([(i, t[i][s - i % 3:s - i % 3 + 1], s - i % 3) for i in on], list(range(len(on)))) if on else []):
                got[i].append(lg)
        assert all(rel(got[i], L.forward(cfg, w, t[i])) < TOL[dtype] for i in range(rows))
        for i in range(rows):
            m.release(i)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("ff", [41, 160])
def test_feed_forward_alone(pkg, tmp_path, dtype, ff):
    """norm1 = −1 erases the mixer's contribution: what remains is the gated, normed feed-forward with its piecewise activation."""
    cfg = one_layer(G.recurrent(24, 2, 2, ff=ff), mult=0.7)
    w, t = G.weights(cfg, 41), toks(cfg, 33, 8)
    w["l0.norm1"][:] = -1.0
    x = L.embed(t, w["embed"].astype(np.float64), w["bigram"].astype(np.float64), 97, 31, 5)
    f = {k: v.astype(np.float64) for k, v in w.items()}
    want = L.add_sublayer(x, L.dense_ff(x, L.group(f, "l0.mlp.")), f["l0.rg2"], f["l0.rg2.b"], f["l0.norm2"], 0.7, 1e-5)
    assert rel(taps_of(pkg, tmp_path, cfg, w, dtype, t)[0], want) < (1e-5 if dtype == "float32" else 2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
def test_large_gate_and_activation_inputs_stay_finite(pkg, tmp_path, dtype):
    cfg = one_layer(G.recurrent(32, 2, 3, ff=64))
    w, t = G.weights(cfg, 43), toks(cfg, 20, 9)
    for k in ("l0.mlp.up", "l0.rg1", "l0.rg2", "l0.mix.ra", "l0.mix.y"):
        w[k] *= 64.0
    taps = []
    L.forward(cfg, w, t, taps)
    assert rel(taps_of(pkg, tmp_path, cfg, w, dtype, t), taps) < (1e-4 if dtype == "float32" else 0.1)


# ── whole models: prompts, portions, decoding ─────────────────────────────────────────────────────────────────────────────
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(G.CONFIGS))
def test_prompt_portions_and_decoding_agree_with_the_oracle(pkg, cases, name, dtype):
    cfg, w, path = cases(name)
    t = toks(cfg, 301, 1)
    want = L.forward(cfg, w, t)
    m = load(pkg, path, dtype)
    errs = {}
    for seq, (label, cuts) in enumerate({"whole": [301], "portions": [2, 3, 64, 17, 65, 2, 129], "twos": [100, 2], "sixteens": [16],
                                         "decode": [240, 1], "from the first token": [1, 1, 1, 1, 1, 33]}.items()):
        errs[label] = rel(feed(m, seq, t, cuts), want)
        m.release(seq)
    assert max(errs.values()) < TOL[dtype], errs


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["wide", "shared", "loop", "talks"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6])
def test_first_tokens(pkg, cases, n, name, dtype):
    """Sequences shorter than the convolution, in a slot and blocks that another sequence has just left."""
    cfg, w, path = cases(name)
    m = load(pkg, path, dtype, seqs=1, blocks=10, tokens=160)
    m.forward_rows([(1, toks(cfg, 150, 2), 0)], [])
    m.release(1)
    t = toks(cfg, n, 50 + n)
    assert rel(feed(m, 2, t, [n]), L.forward(cfg, w, t)) < TOL[dtype]
    m.release(2)
    assert rel(feed(m, 3, t, [1]), L.forward(cfg, w, t)) < TOL[dtype]


@pytest.mark.parametrize("tiles", [0, 2])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "wide", "deep", "sinks", "shared", "loop", "all", "far", "talks"])
def test_unequal_batch_against_each_request_alone(pkg, cases, knobs, name, dtype, tiles):
    """Portions of some requests beside single decoded tokens of others, members coming and going; rows against the oracle, and against
    the same rows computed alone to rounding."""
    cfg, w, path = cases(name)
    knobs.set(LATENT_TILES=tiles)
    m = load(pkg, path, dtype, tokens=400, seqs=4)
    seqs = {i: toks(cfg, n, 60 + i) for i, n in enumerate((190, 37, 140, 75))}
    want = {i: L.forward(cfg, w, t) for i, t in seqs.items()}
    plan = [{0: 100, 1: 5}, {0: 1, 1: 1, 2: 70}, {2: 66, 0: 2, 3: 3, 1: 1}, {0: 64, 3: 69, 1: 2}, {0: 1, 2: 1, 3: 1, 1: 1}, {1: 27, 0: 22, 2: 3, 3: 2}]
    at = {i: 0 for i in seqs}
    got = {i: [] for i in seqs}
    for step in plan:
        items = [(i, seqs[i][at[i]:at[i] + n], at[i]) for i, n in step.items()]
        total = sum(step.values())
        rows = m.forward_rows(items, list(range(total)))
        r = 0
        for i, n in step.items():
            got[i].append(rows[r:r + n])
            r += n
            at[i] += n
    alone = load(pkg, path, dtype, tokens=400, seqs=4)
    for i, t in seqs.items():
        g = np.concatenate(got[i])
        assert at[i] == len(t)
        assert rel(g, want[i]) < TOL[dtype]
        assert rel(g, feed(alone, 10 + i, t, [len(t)])) < TOL[dtype]
        alone.release(10 + i)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "loop"])
def test_pages_and_slots_are_used_again(pkg, cases, name, dtype):
    """A pool that holds two short requests, two state slots, twelve requests one after the other with different lengths: every one must
    be what it is alone; exhaustion is refused without side effects."""
    cfg, w, path = cases(name)
    m = load(pkg, path, dtype, tokens=96, seqs=2, slots=2, blocks=6)
    assert m.state_slots() == (2, 2)
    live = {}
    for i in range(12):
        n = [33, 7, 48, 20][i % 4]
        t = toks(cfg, n, 100 + i)
        if len(live) == 2:
            m.release(live.pop(min(live)))
        g = feed(m, 200 + i, t, [[n], [5, 1], [2]][i % 3])
        live[i] = 200 + i
        assert rel(g, L.forward(cfg, w, t)) < TOL[dtype] * (1.5 if (name, dtype) == ("loop", "bfloat16") else 1), i      # (norms of small results, eight layers)
    assert m.state_slots() == (2, 0)
    with pytest.raises(RuntimeError, match="state slots"):
        m.forward_rows([(999, toks(cfg, 3, 1), 0)], [])
    before = m.kv_slot_capacity_snapshot()
    for s in live.values():
        m.release(s)
    assert m.state_slots() == (2, 2) and before["free_blocks"] < 6 and m.kv_slot_capacity_snapshot()["free_blocks"] == 6
    # recurrent state is not kept per block: the prefix cache must never splice such a sequence
    t = toks(cfg, 40, 9)
    feed(m, 500, t, [40])
    m.prefix_cache_register(500, t, 0)
    m.reserve_kv_slots([(501, 40)])
    assert m.prefix_cache_acquire(501, t) == 0


@pytest.mark.parametrize("name", ["deep", "shared", "far"])
def test_prefix_cache_of_an_attention_only_model(pkg, cases, name):
    """Without recurrent layers a cached prefix is spliced in, including the previous token of the pair embedding."""
    cfg, w, path = cases(name)
    m = load(pkg, path, "float32", tokens=160, seqs=2)
    t = toks(cfg, 70, 19)
    feed(m, 1, t[:48], [48])
    m.prefix_cache_register(1, t[:48], 0)
    m.reserve_kv_slots([(2, 70)])
    n = m.prefix_cache_acquire(2, t)
    assert n == 48
    g = m.forward_rows([(2, t[48:], 48)], list(range(22)))
    assert rel(g, L.forward(cfg, w, t)[48:]) < TOL["float32"]


# ── window edges: one key stands out ──────────────────────────────────────────────────────────────────────────────────────
def standout(window, seed=5, kv_rank=64, dim=32, rot=8, vdim=32, heads=4):
    """One attention layer in which token 1's query scores token 0's key far above every other key, wherever they are: the query
    projection of the plain part is α·(direction of token 0's key) ⊗ (token 1's query latent)."""
    cfg = one_layer(G.attention(heads, dim, rot, vdim, 40, kv_rank, window, scale=1.0), width=72, vocab=60)
    w = G.weights(cfg, seed)
    w["bigram"][:] = 0.0
    p = "l0.mix."
    f = {k: v.astype(np.float64) for k, v in w.items()}
    cq = lambda x: L.unit_rms(x @ f[p + "dq"].T, 1e-5) * f[p + "dq.norm"]
    lat = lambda x: L.unit_rms(x @ f[p + "dkv"][:kv_rank].T, 1e-5) * f[p + "dkv.norm"]
    ask, key = cq(f["embed"][1]), lat(f["embed"][0])
    for h in range(heads):
        k = f[p + "uk"][h * dim:(h + 1) * dim] @ key
        uq = np.zeros((dim + rot, 40))
        uq[:dim] = np.outer(k / (k @ k) * 14.0, ask / (ask @ ask))
        w[p + "uq"][h * (dim + rot):(h + 1) * (dim + rot)] = G.bf16(uq)
    return cfg, w


@pytest.mark.parametrize("form,dtype", [("plain", "float32")] + [(f, "bfloat16") for f in ("latent", "pair", "split", "pair split", "expanded", "plain")])
@pytest.mark.parametrize("window", [1, 2, 16, 17, 64, 100])
def test_window_edge(pkg, tmp_path, knobs, forms, window, form, dtype):
    """Token 0 stands exactly on the last visible place, or one further back, for query token 1 — in a prompt, in a portion and decoded,
    with the window's edge at every kind of place within a page.  The oracle with a window one off must be far away."""
    knobs.set(LATENT_PLAIN=int(form == "plain"), LATENT_SPLITS=4 if "split" in form else 1, LATENT_TILES=2 if "pair" in form else 1,
              LATENT_EXPAND_MIN_ROWS=2 if form == "expanded" else 0)
    cfg, w = standout(window)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype)
    forms.reset()
    wrong = json.loads(json.dumps(cfg))
    wrong["layers"][0]["mixer"]["mask"]["size"] = window + 1
    seq = 0
    for at in (0, 3, 15, 16):
        for back in (window - 1, window):
            t = np.full(at + back + 1, 7, np.uint32)
            t[2:] = toks(cfg, max(0, len(t) - 2), 70)[:max(0, len(t) - 2)] % 50 + 5
            t[:2] = t[:2] if len(t) < 2 else 9
            t[at] = 0 if back else 1
            t[at + back] = 1
            want = L.forward(cfg, w, t)[-1:]
            if back == window:                                       # a window one larger would see it
                assert rel(L.forward(wrong, w, t)[-1:], want) > 3 * TOL["bfloat16"]
            whole = feed(m, seq, t, [len(t)])[-1:]
            step = feed(m, seq + 1, t, [max(1, len(t) - 1), 1])[-1:]
            parts = feed(m, seq + 2, t, [max(1, len(t) - 2), 2])[-1:]
            for s in range(3):
                m.release(seq + s)
            seq += 3
            assert max(rel(g, want) for g in (whole, step, parts)) < TOL[dtype], (at, back)
    h = forms.hits()
    if form == "plain":
        assert h.get("latent_attn_plain") and not h.get("latent_attn") and not h.get("latent_attn_expanded")
    elif "split" in form or "pair" in form:
        assert bool(h.get("latent_attn_split")) == ("split" in form) and bool(h.get("latent_attn_pair")) == ("pair" in form)
    elif form == "expanded":
        assert h.get("latent_attn_expanded") or window == 1
    else:
        assert h.get("latent_attn") and not h.get("latent_attn_expanded")


@pytest.mark.parametrize("dtype", DTYPES)
def test_far_key_among_hundreds_at_page_borders(pkg, tmp_path, dtype):
    """The key that stands out sits 290 tokens back, around a page border, in a prompt, decoded, and seen from a long later portion."""
    cfg, w = standout(600)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype, tokens=512)
    far = json.loads(json.dumps(cfg))
    far["layers"][0]["mixer"]["mask"]["size"] = 250
    for i, at in enumerate((14, 15, 16, 17, 31, 32)):
        t = toks(cfg, at + 291, 80) % 50 + 5
        t[at], t[-1] = 0, 1
        want = L.forward(cfg, w, t)[-1:]
        assert rel(L.forward(far, w, t)[-1:], want) > 3 * TOL["bfloat16"]
        for j, cuts in enumerate(([len(t)], [len(t) - 1, 1], [40, 200, 100], [64, 3])):
            assert rel(feed(m, 10 * i + j, t, cuts)[-1:], want) < TOL[dtype], (at, cuts)
            m.release(10 * i + j)


# ── decoding loop, graph, sampling ────────────────────────────────────────────────────────────────────────────────────────
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("splits", [1, 4])
@pytest.mark.parametrize("name", ["all", "loop", "bare", "far", "uneven"])
def test_grouped_steps_prepare_their_rows(pkg, cases, knobs, forms, name, splits, dtype):
    """Single tokens from the first one on, over the starts of blocks, at unequal positions, then a portion that reads what they cached: heads of 1 to 4 pieces of 32, one norm
    for all heads and one each, more heads than a tile holds, another layer's cache.  Against a launch of its own: the roots' sums run in another order, so numbers of the
    format differ by a place now and then, logits by no more than four of its roundings; and against the oracle."""
    cfg, w, path = cases(name)
    t = toks(cfg, 41, 14)
    got = []
    knobs.set(GROUPED_SPLITS=splits)
    for off in (None, 1):
        knobs.set(NO_GROUPED_STEP=off)
        forms.reset()
        m = load(pkg, path, dtype)
        rows = []
        for i in range(36):
            now = [(1, t[i:i + 1], i)] + ([(2, t[i - 5:i - 4], i - 5)] if i >= 5 else [])
            rows.append(m.forward_rows(now, list(range(len(now)))))
        rows.append(m.forward_rows([(1, t[36:], 36)], list(range(5))))
        got.append(np.concatenate(rows))
        assert bool(forms.hits().get("grouped_attn_step")) == (not off)
    want = L.forward(cfg, w, t)
    wanted = np.concatenate([np.stack([want[i]] + ([want[i - 5]] if i >= 5 else [])) for i in range(36)] + [want[36:]])
    assert rel(got[0], got[1]) < {"float32": 2e-6, "bfloat16": 2.0 ** -6}[dtype]
    # (in 16 bits 36 steps of these tokens take either way to the edge of TOL, 0.04 of the oracle: there the two errors have to be alike, by as much as the results may differ)
    err = [rel(g, wanted) for g in got]
    assert err[0] < TOL[dtype] if dtype == "float32" else err[0] < err[1] + 2.0 ** -6, err


@pytest.mark.parametrize("name,dtype,rows,keys,form", [("grouped", "bfloat16", 1, 512, "grouped_attn_keys"), ("grouped", "bfloat16", 1, 513, "grouped_attn_split"),
                                                       ("grouped", "bfloat16", 1, 1025, "grouped_attn_split"), ("grouped", "bfloat16", 33, 1025, "grouped_attn_keys"),
                                                       ("grouped", "bfloat16", 33, 1537, "grouped_attn_split"), ("latent", "float32", 1, 127, "latent_attn"),
                                                       ("latent", "float32", 1, 128, "latent_attn_split"), ("latent", "bfloat16", 1, 256, "latent_attn"),
                                                       ("latent", "bfloat16", 1, 257, "latent_attn_split")])
def test_keys_of_a_step_on_both_sides_of_a_split(pkg, tmp_path, name, dtype, rows, keys, form, forms):
    """A step over as many keys as one split takes, and over one more, against the oracle; with 66 workgroups a split takes more.  (Of several rows the others are of one token.)"""
    cfg = G.segetar(72, 50, [G.gated_pair(8, 4 if rows == 1 else 2, 24, 32, 2000, 2, 16, 16)]) if name == "grouped" else one_layer(G.attention(8, 32, 16, 32, 32, 64, 2000))
    w, t = G.weights(cfg, 37), toks(cfg, keys, 15)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype, seqs=max(rows, 4), tokens=1600)
    m.forward_rows([(1, t[:-1], 0)], [])
    forms.reset()
    got = m.forward_rows([(1, t[-1:], keys - 1)] + [(2 + i, t[i:i + 1], 0) for i in range(rows - 1)], [0])
    assert forms.hits().get(form) == 1, forms.hits()
    assert rel(got, L.forward(cfg, w, t)[-1:]) < TOL[dtype]


@pytest.mark.parametrize("dtype,rows,alone", [("float32", 64, False), ("float32", 65, True), ("bfloat16", 65, False)])
def test_rows_of_a_round_of_workgroups_prepare_themselves(pkg, tmp_path, dtype, rows, alone, forms):
    """32 bits, 4 heads of keys: 256 workgroups run at once, and with more of them a launch of its own prepares the rows.  Second tokens, against the oracle."""
    cfg = G.segetar(72, 50, [G.gated_pair(8, 4, 24, 32, 40, 2, 16, 16)])
    w = G.weights(cfg, 43)
    t = [toks(cfg, 2, 50 + i) for i in range(rows)]
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype, seqs=rows)
    m.forward_rows([(i, t[i][:1], 0) for i in range(rows)], [])
    forms.reset()
    got = m.forward_rows([(i, t[i][1:], 1) for i in range(rows)], list(range(rows)))
    assert bool(forms.hits().get("grouped_attn_step")) != alone, forms.hits()
    assert rel(got, np.stack([L.forward(cfg, w, t[i])[1] for i in range(rows)])) < TOL[dtype]


def near_greedy(cfg, w, prompt, out, slack):
    """Every generated token's oracle logit is within `slack` (relative to the logits' rms) of the best one."""
    full = np.concatenate([prompt, out]).astype(np.uint32)
    lg = L.forward(cfg, w, full[:-1])[len(prompt) - 1:]
    gap = lg.max(axis=1) - lg[np.arange(len(out)), out]
    return float(gap.max() / np.sqrt(np.mean(lg ** 2))) <= slack


@pytest.mark.parametrize("n,max_len", [(1, 48), (3, 1600), (20, 1600), (65, 272)])
def test_what_a_decode_call_hands_over(pkg, cases, n, max_len):
    """Calls of one step, in which positions, previous tokens and block tables (up to 2000 words) travel each time, against one long call, whose
    later steps the device feeds itself; tables that get a block in between, a number of sequences that changes."""
    cfg, _, path = cases("shared")
    lens = [max_len - 40 - (7 * i) % 33 if i % 5 == 0 else 1 + (11 * i) % 30 for i in range(n)]
    prompts = [toks(cfg, k if max_len > 48 else 5, 70 + i) for i, k in enumerate(lens)]
    got = []
    for calls in ([1] * 20, [20], [3, 1, 16]):
        m = load(pkg, path, "float32", tokens=2048, seqs=n, max_len=max_len, blocks=n * ((max_len + 15) // 16) + 1)
        nxt = np.concatenate([m.unified_forward([(i, p, 0, True)])[0] for i, p in enumerate(prompts)])
        if n > 1:
            m.decode_steps([n - 1], nxt[-1:], 1)
            m.release(n - 1)
            m.unified_forward([(n - 1, prompts[-1], 0, True)])
        out = []
        for steps in calls:
            out.append(m.decode_steps(range(n), nxt, steps))
            nxt = out[-1][-1]
        got.append(np.concatenate(out))
        assert [m.block_table(i)[1] for i in range(n)] == [len(p) + 20 for p in prompts]
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "wide", "sinks", "shared", "loop", "all", "far", "talks"])
def test_long_decoding_through_the_graph(pkg, cases, forms, name, dtype):
    """Three sequences of different lengths decode 150 tokens past their windows in one captured step (several replays with eager
    forwards between them); the same ids as eager single steps, and the oracle's choices up to rounding."""
    cfg, w, path = cases(name)
    m = load(pkg, path, dtype, tokens=3 * 260, seqs=4, max_len=260)
    prompts = [toks(cfg, n, 90 + n) for n in (5, 61, 33)]
    first, _ = m.unified_forward([(i, p, 0, True) for i, p in enumerate(prompts)])
    forms.reset()
    ids, out, nxt = [0, 1, 2], [first[None]], first
    for steps in (1, 60, 2, 40):
        out.append(m.decode_steps(ids, nxt, steps))
        nxt = out[-1][-1]
        # eager work between replays: an unrelated sequence comes and goes
        m.unified_forward([(7, toks(cfg, 9, steps), 0, True)])
        m.release(7)
    gen = np.concatenate(out)
    assert forms.hits().get("graph_replay", 0) >= 100
    # eager, one mixed forward per token, continuing from the state the graph left
    for _ in range(46):
        lens = [m.block_table(i)[1] for i in ids]
        nxt, _ = m.unified_forward([(i, [int(t)], n, True) for i, t, n in zip(ids, nxt, lens)])
        gen = np.concatenate([gen, nxt[None]])
    for i, p in enumerate(prompts):
        assert near_greedy(cfg, w, p, gen[:, i], 2e-4 if dtype == "float32" else 0.25)
    # the whole generation again, eagerly, in another model
    e = load(pkg, path, dtype, tokens=3 * 260, seqs=4, max_len=260)
    nxt, _ = e.unified_forward([(i, p, 0, True) for i, p in enumerate(prompts)])
    again = [nxt]
    for s in range(len(gen) - 1):
        nxt, _ = e.unified_forward([(i, [int(t)], len(p) + s, True) for i, (t, p) in enumerate(zip(nxt, prompts))])
        again.append(nxt)
    if dtype == "float32":
        assert np.array_equal(np.stack(again), gen)


@pytest.mark.parametrize("name", ["tiny", "one", "bare", "lone"])
def test_masked_and_penalised_greedy_choice(pkg, cases, name):
    cfg, w, path = cases(name)
    m = load(pkg, path, "float32")
    t = toks(cfg, 20, 4)
    lg = L.forward(cfg, w, t)[-1]
    best = int(np.argmax(lg))
    mask = np.ones(cfg["vocab"], np.uint8)
    mask[best] = 0
    assert int(m.unified_forward([(1, t, 0, True)], token_mask=mask)[0][0]) == int(np.argmax(np.where(mask, lg, -np.inf)))
    pen = np.where(np.arange(len(lg)) == best, lg / 50.0 if lg[best] > 0 else lg * 50.0, lg)
    assert int(m.unified_forward([(2, t, 0, True)], repetition_penalties=[(50.0, [best])])[0][0]) == int(np.argmax(pen))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "sinks", "loop", "far"])
def test_generation_through_the_engine_loop(cases, name, dtype):
    """The command line: admission bounded by two state slots and a small pool, prompts cut by a 24-token budget beside decoding
    sequences, graph decoding in between; greedy ids against the oracle."""
    cfg, w, path = cases(name)
    prompts = [toks(cfg, n, 300 + n) for n in (30, 3, 57, 12, 1, 41)]
    text = ";".join(",".join(str(int(x)) for x in p) for p in prompts)
    cmd = [os.path.join(BIN, "ferrum_hip_serve"), "--model", path, "--dtype", dtype, "--prompt-ids", text, "--concurrency", "4", "--state-slots", "2",
           "--out-len", "20", "--max-batched-tokens", "24", "--kv-blocks", "9", "--dump-tokens"]
    p = subprocess.run(cmd, capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stderr[-2000:]
    lines = p.stdout.strip().splitlines()
    head = json.loads(lines[0])
    assert head["model"] == cfg["architecture"] and head["output_tokens"] == 6 * 20 and head["kv_blocks_free_at_exit"] == head["kv_blocks_total"] == 9
    out = {int(l.split(":")[0].split()[1]): np.array(l.split(":")[1].split(), np.int64) for l in lines[1:]}
    for i, pr in enumerate(prompts):
        assert near_greedy(cfg, w, pr, out[i + 1], 2e-4 if dtype == "float32" else 0.25), i


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["wide", "shared", "all", "talks"])
def test_trace_replay(cases, tmp_path, name, dtype):
    """bin/trace_run: portions beside decoded tokens, requests that pause, end and make room; logits against the oracle."""
    cfg, w, path = cases(name)
    seqs = {f"q{i}": toks(cfg, n, 400 + n) for i, n in enumerate((150, 20, 90, 64, 33))}
    want = {k: L.forward(cfg, w, t) for k, t in seqs.items()}
    plan = [{"q0": 100, "q1": 2}, {"q1": 17, "q2": 30}, {"q0": 1, "q1": 1, "q2": 2, "q3": 64}, {"q0": 49, "q2": 58, "q4": 31}, {"q4": 2}]
    p = subprocess.Popen([os.path.join(ROOT, "bin", "trace_run"), "--model", path, "--dtype", dtype, "--out", str(tmp_path), "--max-tokens", "384"],
                         stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
    at = {k: 0 for k in seqs}
    for s, step in enumerate(plan):
        entries, end, rows = [], [], []
        for k, n in step.items():
            pick = sorted({0, n // 2, n - 1}) if not (s == 1 and k == "q2") else []
            entries.append({"id": k, "tokens": [int(x) for x in seqs[k][at[k]:at[k] + n]], "want": pick})
            rows += [want[k][at[k] + j] for j in pick]
            at[k] += n
            if at[k] == len(seqs[k]):
                end.append(k)
        p.stdin.write(json.dumps({"step": s, "entries": entries, "end": end}) + "\n")
        p.stdin.flush()
        assert p.stdout.readline().strip() == f"done {s}"
        got = np.fromfile(tmp_path / f"{s}.f32", "<f4").reshape(-1, cfg["vocab"])
        assert got.shape[0] == len(rows) and rel(got, rows) < TOL[dtype]
    p.stdin.close()
    assert p.wait(timeout=30) == 0


@pytest.mark.parametrize("splits", [1, 4])
@pytest.mark.parametrize("heads,dim,rot,vdim,rank,window", [(3, 20, 6, 36, 30, 700), (17, 16, 10, 8, 60, 33), (5, 24, 40, 12, 100, 64), (2, 8, 6, 8, 128, 1), (16, 32, 64, 16, 250, 90),
                                                            (4, 16, 2, 16, 384, 700), (6, 8, 34, 10, 512, 130), (1, 8, 4, 8, 520, 50), (2, 8, 70, 8, 40, 20)])
def test_latent_attention_in_32_bits(pkg, tmp_path, knobs, forms, heads, dim, rot, vdim, rank, window, splits):
    """Every padded size of the latent, one head and more heads than a row tile, windows inside a step of keys and across several; whole prompts,
    portions and single tokens, keys in one piece and split.  Latents of more than 512 and rotated parts of more than 64 take the plain form."""
    knobs.set(LATENT_SPLITS=splits)
    cfg = G.config(64, 80, [G.attention(heads, dim, rot, vdim, 40, rank, window)], buckets=13)
    w, t = G.weights(cfg, rank), toks(cfg, 170, 9)
    want = L.forward(cfg, w, t)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), "float32")
    forms.reset()
    for seq, cuts in enumerate(([170], [100, 1, 1, 47, 20, 1], [1, 15, 16, 17, 121])):
        assert rel(feed(m, seq, t, cuts), want) < TOL["float32"]
        m.release(seq)
    h, plain = forms.hits(), rank > 512 or rot > 64
    assert bool(h.get("latent_attn_plain")) == plain and bool(h.get("latent_attn_split" if splits > 1 else "latent_attn")) != plain


@pytest.mark.parametrize("name", ["wide", "shared", "sinks", "loop", "talks"])
def test_few_row_and_tile_projections_agree(pkg, cases, knobs, forms, name):
    """The 16-bit tile kernel in each of its sizes and the few-row kernel on the same portions."""
    cfg, w, path = cases(name)
    t = toks(cfg, 200, 12)
    want = L.forward(cfg, w, t)
    for size, set_to in (*SIZES.items(), (None, FEW_ROWS)):
        knobs.set(**set_to)
        m = load(pkg, path, "bfloat16")
        forms.reset()
        assert rel(feed(m, 1, t, [200]), want) < TOL["bfloat16"]
        h = forms.hits()
        if size:
            assert h.get("tiled_gemm_big") and sizes_that_ran(h) == {size}
        else:                                                              # (blocks of an expert's rows have a rule of their own)
            assert h.get("tiled_gemm") and not h.get("tiled_gemm_big")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("j", [3, 4])
@pytest.mark.parametrize("name", ["wide", "shared", "loop", "all", "talks"])
def test_sections_within_a_wave_s_columns(pkg, cases, knobs, forms, name, j, dtype):
    """48 and 64 columns a wave where the projection's parts, of 32 columns and of more, each have an activation of their own, and the last wave's columns do not all exist."""
    cfg, w, path = cases(name)
    t = toks(cfg, 29, 13)
    knobs.set(TILED_J=j, TILED_MIN_TILES=-1, TILED_BIG_MIN_TILES=10 ** 6)
    m = load(pkg, path, dtype)
    forms.reset()
    assert rel(feed(m, 1, t, [29]), L.forward(cfg, w, t)) < TOL[dtype]
    assert forms.hits().get(f"tiled_gemm_cols{16 * j}")


@pytest.mark.parametrize("layer,width", [(G.attention(20, 32, 16, 32, 32, 512, 40), 72), (G.attention(24, 32, 16, 32, 32, 512, 40), 72), (G.recurrent(24, 2, 2, ff=8192), 3104)])
def test_groups_and_slabs_past_a_round_of_workgroups(pkg, tmp_path, layer, width, forms):
    """As many 16-column tiles as make a wave of one projection take 48 or 64 columns, but in groups (the heads' own projections to 512 latents) or in four slabs of K: 32 columns,
    the faster form there."""
    cfg = one_layer(layer, width=width)
    w, t = G.weights(cfg, 41), toks(cfg, 24, 16)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), "bfloat16", seqs=24)
    forms.reset()
    got = m.forward_rows([(i, t[i:i + 1], 0) for i in range(24)], list(range(24)))
    assert not forms.hits().get("tiled_gemm_cols48" if width == 72 else "tiled_gemm_cols64"), forms.hits()
    assert rel(got, np.concatenate([L.forward(cfg, w, t[i:i + 1]) for i in range(24)])) < TOL["bfloat16"]


EVEN = {"nerenex": lambda: G.config(256, 260, [G.recurrent(256, 2, 3, ff=384), G.attention(20, 64, 32, 48, 128, 256, 130, ff=640), G.recurrent(640, 5, 2, ff=128)], mult=0.6),
        "safolorn": lambda: G.safolorn(128, 260, 40, [G.sink_attention(8, 64, 32, 64, 256, 1e5, G.LONG, mlp=G.glu(384, 1.5)), G.sink_attention(4, 64, 32, 32, 256, 1e5, G.LONG, mlp=G.experts(5, 2, 256))]),
        "segetar": lambda: G.segetar(256, 260, [G.scan(256, 16, 128, 4, mlp=G.dense(384)), G.gated_pair(8, 2, 64, 64, 130, 4, 64, 64, mlp=G.grouped_experts(6, 2, 128, 2, 1))]),
        "fororax": lambda: G.fororax(128, 260, [G.talk_attention(8, 2, 64, 32, mlp=G.identity_experts(6, 2, 2, 128, 160)), G.far_attention(4, 2, 64, 96, mlp=G.identity_experts(3, 1, 1, 384, 96))])}


@pytest.mark.parametrize("name", EVEN)
def test_projections_in_tiles_of_256_x_256(pkg, tmp_path, knobs, forms, name):
    """K of whole rounds of four steps: sections that begin within a wave's columns and between two, gated and rare activations among them, biases, experts' blocks of
    256 rows with experts that receive few."""
    cfg = EVEN[name]()
    w, t = G.weights(cfg, 31), toks(cfg, 420, 12)
    path, want = G.write_checkpoint(tmp_path, cfg, w), L.forward(cfg, w, t)
    knobs.set(TILED_256=1, TILED_BIG_MIN_TILES=1, MOE_ROWS_BLOCK=256)
    m = load(pkg, path, "bfloat16")
    forms.reset()
    assert rel(feed(m, 1, t, [420]), want) < TOL["bfloat16"]
    h = forms.hits()
    assert h.get("tiled_gemm_256x256") and bool(h.get("tiled_gemm_grouped_big")) == (name != "nerenex")


@pytest.mark.parametrize("ff,n,forced,taken", [(2048, 32, None, 1), (2048, 31, None, 0), (256, 32, None, 0), (2048, 32, 257, 0)])
def test_blocks_of_256_sorted_rows(pkg, tmp_path, knobs, forms, ff, n, forced, taken):
    """Two experts of which each token takes one: blocks of 256 rows from a mean of 2048 (128 tokens a sequence, and one more), where one of the two projections runs in
    tiles of as many rows (2048 columns of K 2048), not where neither does (256 columns, K of 256) or another size is asked for; against blocks of 128."""
    cfg = G.safolorn(2048, 260, 40, [G.sink_attention(4, 64, 32, 32, 256, 1e5, G.LONG, mlp=G.experts(2, 1, ff))])
    path = G.write_checkpoint(tmp_path, cfg, G.weights(cfg, 33))
    items = [(i, toks(cfg, 129, i), 0) for i in range(n)]
    at = [129 * i + j for i in range(n) for j in (0, 64, 128)]
    out = {}
    for block in (None, 128):
        knobs.set(TILED_WIDE_MIN_TILES=forced, MOE_ROWS_BLOCK=block)
        m = load(pkg, path, "bfloat16", tokens=129 * n, seqs=n, blocks=9 * n + 2, max_len=256)
        forms.reset()
        out[block] = m.forward_rows(items, at)
        if block is None:
            assert forms.hits().get("moe_rows_256", 0) == taken, forms.hits()
        del m
    assert rel(out[None], out[128]) < 4e-3        # (both sum K in steps of 32 in fp32: equal but for the order, 16-bit results of one layer)


def test_columns_of_several_kinds_in_one_round(pkg, tmp_path, knobs, forms):
    """An input projection of one round of 256 x 256 whose sections begin within a wave's columns: those are finished slowly there, so it runs in tiles of 128 x 256."""
    cfg = G.safolorn(1152, 260, 40, [G.sink_attention(16, 64, 32, 32, 256, 1e5, G.LONG, mlp=G.glu(1552, 1.5))])
    path = G.write_checkpoint(tmp_path, cfg, G.weights(cfg, 35))
    items = [(i, toks(cfg, 128, i), 0) for i in range(13)]
    out = {}
    for forced in (None, 1):
        knobs.set(TILED_256=forced)
        m = load(pkg, path, "bfloat16", tokens=128 * 13, seqs=13, blocks=8 * 13 + 2, max_len=256)
        forms.reset()
        out[forced] = m.forward_rows(items, [128 * i + 127 for i in range(13)])
        h = forms.hits()
        assert bool(h.get("tiled_gemm_256x256")) == bool(forced) and bool(h.get("tiled_gemm_128x256")) != bool(forced), h
        del m
    assert rel(out[None], out[1]) < 4e-3


@pytest.mark.parametrize("name", ["wide", "shared", "sinks", "loop", "talks"])
@pytest.mark.parametrize("big", [1, 10 ** 6])
def test_32_bit_projections_of_prompts(pkg, cases, knobs, forms, name, big):
    """The tiles that so few rows take, mostly of 64 × 64, and the few-row kernel, whatever the projections' sizes."""
    cfg, w, path = cases(name)
    t = toks(cfg, 200, 12)
    knobs.set(TILED_BIG_MIN_TILES=big)
    m = load(pkg, path, "float32")
    forms.reset()
    assert rel(feed(m, 1, t, [200]), L.forward(cfg, w, t)) < TOL["float32"]
    assert bool(forms.hits().get("tiled_gemm_big")) == (big == 1)


@pytest.mark.parametrize("tokens,width,ff,size", [(700, 64, 1024, "64x64"), (700, 64, 1025, "64x64"), (700, 200, 1400, "128x64"), (641, 64, 1500, "128x64"),
                                                  (656, 330, 1300, "128x64"), (2000, 64, 1500, "128x128"), (1921, 200, 1400, "128x128"), (2047, 130, 1601, "128x128")])
def test_32_bit_tile_sizes(pkg, tmp_path, forms, tokens, width, ff, size):
    """Every tile of a 32-bit prompt's up-projection: rows and columns past the last tile, K of 4, 10, 14 and 22 steps of 16 (fewer than the ring of rows holds, and
    past the 128 products that are summed apart)."""
    cfg = G.config(width, 80, [G.attention(2, 8, 6, 8, 20, 16, 40, ff=ff)], buckets=13)
    w, t = G.weights(cfg, 31), toks(cfg, tokens, 9)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), "float32", tokens=2048)
    forms.reset()
    assert rel(feed(m, 1, t, [tokens]), L.forward(cfg, w, t)) < TOL["float32"]
    assert size in sizes_that_ran(forms.hits())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["wide", "odd", "shared", "sinks", "loop", "uneven", "talks", "far"])
def test_pages_that_held_no_numbers(pkg, tmp_path, name, dtype):
    """A sequence whose embedding is infinite leaves its pages to the next one, whose blocks end anywhere: nothing of it is seen in a prompt, in portions or a token at a
    time over the edge of a block."""
    cfg = G.CONFIGS[name]
    w = dict(G.weights(cfg, 5))
    w["embed"] = w["embed"].copy()
    w["embed"][3] = np.inf
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype, tokens=64, seqs=2, blocks=4)
    t = toks(cfg, 40, 9)
    t[t == 3] = 4
    for seq, cuts in enumerate(([21], [5, 1, 1], [15, 3, 1], [16, 16, 8])):
        assert not np.isfinite(feed(m, 9, np.full(40, 3, np.uint32), [40])).any()
        m.release(9)
        got = feed(m, seq, t[:40 if cuts[-1] == 8 else 21], cuts)
        assert np.isfinite(np.delete(got, 3, axis=1)).all()                     # (the column of that token, where the embedding serves as the head, is infinite)
        m.release(seq)


def test_missing_and_misshapen_weights_are_named(pkg, tmp_path):
    cfg = G.CONFIGS["tiny"]
    w = G.weights(cfg, 1)
    for name, new in (("l0.mix.ra", None), ("l1.mix.o", np.zeros((40, 15), np.float32)), ("l2.rg1.b", np.zeros(3, np.float32))):
        bad = {k: v for k, v in w.items() if k != name}
        if new is not None:
            bad[name] = new
        with pytest.raises(RuntimeError, match=name.replace(".", r"\.")):
            load(pkg, G.write_checkpoint(tmp_path / name, cfg, bad), "bfloat16")

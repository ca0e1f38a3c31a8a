"""Segetar's mechanisms on the device against the plain oracle of tests/layered_oracle.py: each alone through the taps of small models,
with mistakes planted in the oracle where random weights would hide them; whole models, batches and the engine loop are covered with
the other layered architectures in test_layered_gpu.py."""
import json

import numpy as np
import pytest

from tests import layered_gen as G
from tests import layered_oracle as L
from tests.test_layered_gpu import DTYPES, TOL, cases, feed, load, pkg, rel, taps_of, toks  # noqa: F401  (two are fixtures)

pytestmark = pytest.mark.gpu
ALONE = {"float32": 1e-5, "bfloat16": 2e-2}


def model(layers, width=72, vocab=50, loop=None, **kw):
    return G.segetar(width, vocab, layers, loop, **kw)


def changed(cfg, edit):
    c = json.loads(json.dumps(cfg))
    edit(c)
    return c


def silence(w, *what):
    """Takes an output ("left.o", "right.out", …) of every layer's mixer out."""
    for k in w:
        if k.split(".mix.")[-1] in what:
            w[k][:] = 0.0


def left_only(w):
    silence(w, "right.o", "right.out")
    return w


def right_only(w):
    silence(w, "left.o", "left.out")
    return w


def agree(pkg, tmp_path, cfg, w, dtype, n=70, tol=None, seed=6):
    t, taps = toks(cfg, n, seed), []
    L.forward(cfg, w, t, taps)
    assert rel(taps_of(pkg, tmp_path, cfg, w, dtype, t), taps) < (tol or ALONE[dtype])
    return t, taps


def differs(cfg, w, t, taps, bound=1e-3):
    other = []
    L.forward(cfg, w, t, other)
    return rel(other, taps) > bound


def portions_agree(pkg, tmp_path, cfg, w, dtype, n, cuts, seed=6):
    t = toks(cfg, n, seed)
    want = L.forward(cfg, w, t)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype, tokens=max(512, n + 16))
    for i, c in enumerate(cuts):
        assert rel(feed(m, i, t, c), want) < TOL[dtype], c
        m.release(i)
    return t, want


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,n", [(1030, 9), (1056, 40), (2044, 17), (2052, 520), (4100, 5)])
def test_rows_of_several_quads_a_thread(pkg, tmp_path, dtype, width, n):
    """Both branches of a layer normed and joined, experts' rows added, in rows that a thread holds two or four pieces of, or none."""
    cfg = model([G.gated_pair(2, 1, 8, 8, 9, 1, 8, 8), G.scan(24, 3, 5, 2, mlp=G.grouped_experts(4, 2, 12))], width=width)
    agree(pkg, tmp_path, cfg, G.weights(cfg, 19), dtype, n=n, tol=2 * ALONE[dtype])


# ── grouped attention ─────────────────────────────────────────────────────────────────────────────────────────────────────
ATTN = [(6, 2, 20, 28, 9, 6), (4, 4, 32, 32, 40, 32), (24, 1, 64, 64, 25, 40), (1, 1, 5, 3, 1, 2), (8, 4, 96, 70, 64, 0), (35, 7, 128, 128, 33, 128), (3, 3, 200, 190, 50, 100),
        (2, 1, 256, 256, 30, 256), (2, 2, 300, 40, 20, 300)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", ["gated", "plain"])
@pytest.mark.parametrize("i", range(len(ATTN)))
def test_grouped_attention_alone(pkg, tmp_path, dtype, kind, i):
    """With biases, rotation and head gates; without all three and behind a norm of its result."""
    H, kv, dim, vdim, window, rot = ATTN[i]
    if kind == "gated":
        layer = G.gated_pair(H, kv, dim, vdim, window, 1, 4, 4, rot=rot, base=300.0, left=1.7)
    else:
        layer = G.retention_pair(H, kv, dim, vdim, window, (0.5,), 4, 4)
    cfg = model([layer])
    w = left_only(G.weights(cfg, 20 + i))
    t, taps = agree(pkg, tmp_path, cfg, w, dtype, tol=ALONE[dtype] * (1 if dtype == "float32" else 2))
    assert differs(changed(cfg, lambda c: c["layers"][0]["mixer"]["left"]["mask"].update(size=window + 1)), w, t, taps)
    if H > kv > 1:                                                            # heads dealt out in turn would show
        swap = dict(w)
        for n, d in (("k", dim), ("v", vdim)):
            swap[f"l0.mix.left.{n}"] = w[f"l0.mix.left.{n}"].reshape(kv, d, -1)[::-1].reshape(kv * d, -1)
        assert differs(cfg, swap, t, taps)


def test_rotation_pairs_neighbours_in_attention(pkg, tmp_path, monkeypatch):
    cfg = model([G.gated_pair(2, 1, 24, 24, 40, 1, 4, 4, rot=16, base=50.0, scale=0.6)])
    w = left_only(G.weights(cfg, 31))
    t, taps = agree(pkg, tmp_path, cfg, w, "float32")
    monkeypatch.setattr(L, "rotate_interleaved", L.rotated_halves)
    assert differs(cfg, w, t, taps)


def test_queries_and_keys_are_normed_over_all_heads(pkg, tmp_path, monkeypatch):
    """One head's rows are much larger than the others': a norm per head would show."""
    cfg = model([G.retention_pair(4, 2, 16, 16, 30, (0.5,), 4, 4)])
    w = left_only(G.weights(cfg, 32))
    w["l0.mix.left.q"][:16] *= 4.0
    w["l0.mix.left.k"][16:] *= 4.0
    t, taps = agree(pkg, tmp_path, cfg, w, "float32")
    unit = L.unit_rms
    monkeypatch.setattr(L, "unit_rms", lambda x, eps: unit(x.reshape(len(x), -1, 16), eps).reshape(x.shape) if x.shape[-1] in (64, 32) else unit(x, eps))
    assert differs(cfg, w, t, taps)


# one key stands out
FORMS = [("plain", "float32")] + [(f, "bfloat16") for f in ("plain", "keys", "split", "tile")]


def set_form(knobs, form):
    knobs.set(GROUPED_PLAIN=int(form == "plain"), GROUPED_SPLITS={"keys": 1, "split": 4}.get(form, 0), GROUPED_TILE_MIN_ROWS=1 if form == "tile" else 10 ** 6)


def standout(window, kind, seed=5, heads=6, kv=2, dim=32, rot=8):
    """One attention layer in which token 1's query scores token 0's key far above every other key, wherever they are (the rotated
    dimensions take no part)."""
    if kind == "gated":
        layer = G.gated_pair(heads, kv, dim, dim, window, 1, 4, 4, rot=rot, scale=0.6, left=2.0)
    else:
        layer, rot = G.retention_pair(heads, kv, dim, dim, window, (0.5,), 4, 4, scale=0.6), 0
    cfg = model([layer], vocab=60)
    w = left_only(G.weights(cfg, seed, clear_routes=False))
    p, f = "l0.mix.left.", {k: np.asarray(v, np.float64) for k, v in w.items()}
    h = lambda t: L.unit_rms(f["embed"][t], 1e-5) * f["l0.norm1"]
    if kind == "gated":
        w[p + "q.b"] = G.bf16(0.1 * w[p + "q.b"])
    key = (L.unit_rms(f[p + "k"] @ h(0) + f.get(p + "k.b", 0.0), 1e-5) * f[p + "k.norm"]).reshape(kv, dim)
    key[:, :rot] = 0.0
    w[p + "q.norm"][:] = 1.0
    ask = h(1)
    want = np.repeat(key, heads // kv, axis=0).reshape(-1)
    w[p + "q"] = G.bf16(np.outer(want, ask / (ask @ ask)) * 4.0 + 0.3 * w[p + "q"])
    return cfg, w


@pytest.mark.parametrize("form,dtype", FORMS)
@pytest.mark.parametrize("kind", ["gated", "plain"])
@pytest.mark.parametrize("window", [1, 2, 16, 17, 64, 100])
def test_window_edge(pkg, tmp_path, knobs, forms, window, kind, form, dtype):
    """Token 0 stands on the last visible place, or one further back, for query token 1 — in a prompt, in a portion and decoded, with
    the window's edge at every kind of place within a page.  The oracle with a window one off must be far away."""
    set_form(knobs, form)
    cfg, w = standout(window, kind)
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype)
    forms.reset()
    wrong = changed(cfg, lambda c: c["layers"][0]["mixer"]["left"]["mask"].update(size=window + 1))
    seq = 0
    for at in (0, 3, 15, 16):
        for back in (window - 1, window):
            t = toks(cfg, at + back + 1, 70) % 50 + 5
            t[at] = 0 if back else 1
            t[at + back] = 1
            want = L.forward(cfg, w, t)[-1:]
            if back == window:
                assert rel(L.forward(wrong, w, t)[-1:], want) > 3 * TOL["bfloat16"]
            for cuts in ([len(t)], [max(1, len(t) - 1), 1], [max(1, len(t) - 2), 2], [max(1, len(t) - 3), 2, 1]):
                assert rel(feed(m, seq, t, cuts)[-1:], want) < TOL[dtype], (at, back, cuts)
                m.release(seq)
                seq += 1
    h = forms.hits()
    assert h.get({"plain": "grouped_attn_plain", "keys": "grouped_attn_keys", "split": "grouped_attn_split", "tile": "grouped_attn_tile"}[form])


@pytest.mark.parametrize("form,dtype", FORMS)
def test_far_key_and_future_key(pkg, tmp_path, knobs, form, dtype):
    """The key that stands out sits hundreds of tokens back, at a page border; standing right behind the query it must not be seen."""
    set_form(knobs, form)
    cfg, w = standout(600, "gated")
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), dtype, tokens=512)
    seq = 0
    for at, back in ((0, 1), (15, 290), (16, 290), (17, 63), (31, 64), (0, 447)):
        t = toks(cfg, at + back + 3, 80) % 50 + 5
        q = at + back
        t[at], t[q], t[q + 1] = 0, 1, 0
        blind = t.copy()
        blind[at] = 7
        want, none = L.forward(cfg, w, t)[q], L.forward(cfg, w, blind)[q]
        assert rel(none[None], want[None]) > 3 * TOL["bfloat16"]
        for tokens, ref in ((t, want), (blind, none)):
            for cuts in ([len(t)], [q, 1, 1], [max(1, q - 1), 2, 1], [40, 100, 65]):
                assert rel(feed(m, seq, tokens, cuts)[q:q + 1], ref[None]) < TOL[dtype], (at, back, cuts)
                m.release(seq)
                seq += 1


# ── linear attention ──────────────────────────────────────────────────────────────────────────────────────────────────────
LIN = [(5, 12, 20), (1, 3, 2), (4, 64, 128), (3, 128, 64), (2, 32, 32), (2, 100, 96), (1, 256, 256), (7, 48, 160)]


def lin_layer(kind, i):
    H, dim, vdim = LIN[i]
    if kind == "gated":
        return G.gated_pair(2, 1, 8, 8, 5, H, dim, vdim, tau=(16.0, 1.0, 3.0)[i % 3], right=-0.6)
    return G.retention_pair(2, 1, 8, 8, 5, [(0.999, 0.5, 0.97, 0.03, 1.0)[(i + h) % 5] for h in range(H)], dim, vdim, rot=(dim // 2 if i % 2 else dim) // 2 * 2, base=40.0)


CHUNKS = [("step", 0), ("chunk", 1)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", ["gated", "retention"])
@pytest.mark.parametrize("form,rows", CHUNKS)
@pytest.mark.parametrize("i", range(len(LIN)))
def test_linear_attention_alone(pkg, tmp_path, knobs, dtype, kind, form, rows, i):
    """Several chunks, decays from 1 to almost 0, every mistake of decay or rotation visible in 32-bit."""
    knobs.set(LINEAR_CHUNK_MIN_ROWS=rows)
    cfg = model([lin_layer(kind, i)])
    w = right_only(G.weights(cfg, 40 + i))
    t, taps = agree(pkg, tmp_path, cfg, w, dtype, n=200, tol=ALONE[dtype] * {"gated": 1, "retention": 2}[kind] * (1 if dtype == "float32" else 2))      # (small results are normed)
    if kind == "gated":
        assert differs(changed(cfg, lambda c: c["layers"][0]["mixer"]["right"].update(tau=c["layers"][0]["mixer"]["right"]["tau"] * 1.5)), w, t, taps, 1e-4)
    else:
        assert differs(changed(cfg, lambda c: c["layers"][0]["mixer"]["right"].update(decay=[0.9 * d for d in c["layers"][0]["mixer"]["right"]["decay"]])), w, t, taps, 1e-4)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", ["gated", "retention"])
@pytest.mark.parametrize("form,rows", CHUNKS)
@pytest.mark.parametrize("i", [0, 2, 5])
def test_linear_attention_in_portions(pkg, tmp_path, knobs, dtype, kind, form, rows, i):
    knobs.set(LINEAR_CHUNK_MIN_ROWS=rows)
    cfg = model([lin_layer(kind, i)])
    w = right_only(G.weights(cfg, 40 + i))
    portions_agree(pkg, tmp_path, cfg, w, dtype, 260, ([260], [64, 64, 65, 2], [1], [200, 1, 2, 3], [63, 2], [128, 1, 130, 1]))


@pytest.mark.parametrize("form,rows", CHUNKS)
def test_state_of_the_first_token_survives(pkg, tmp_path, knobs, form, rows):
    """No decay, and only the first token writes: every later token must read exactly that, over chunks, portions and decoding."""
    knobs.set(LINEAR_CHUNK_MIN_ROWS=rows)
    cfg = model([G.retention_pair(1, 1, 8, 8, 3, (1.0, 1.0), 16, 16, rot=0)], vocab=60, eps=0.05)
    w = right_only(G.weights(cfg, 61))
    f = {k: np.asarray(v, np.float64) for k, v in w.items()}
    h0 = L.unit_rms(f["embed"][0], 0.05) * f["l0.norm1"]
    w["embed"][1:] = G.bf16(w["embed"][1:] - np.outer(w["embed"][1:] @ (w["l0.norm1"] * h0), h0 / (f["l0.norm1"] * h0 @ h0)))
    w["l0.mix.right.v"] = G.bf16(np.outer(np.linspace(1.0, 2.0, 32), h0 / np.sqrt(h0 @ h0)))
    t = toks(cfg, 240, 4) % 55 + 3
    t[0] = 0
    want = L.forward(cfg, w, t)
    other = t.copy()
    other[0] = 5
    assert rel(L.forward(cfg, w, other)[200:], want[200:]) > 3 * TOL["bfloat16"]
    m = load(pkg, G.write_checkpoint(tmp_path, cfg, w), "float32")            # (in 16 bits the other tokens' values are not quite zero)
    for i, cuts in enumerate(([240], [1, 100, 64, 2], [65, 1])):
        assert rel(feed(m, i, t, cuts), want) < TOL["float32"], cuts
        m.release(i)


# ── selective scan ────────────────────────────────────────────────────────────────────────────────────────────────────────
SCAN = [(75, 9, 5, 3), (24, 2, 1, 1), (512, 16, 20, 4), (44, 24, 40, 2), (100, 64, 3, 5), (33, 130, 7, 4), (40, 256, 33, 8), (320, 1, 64, 4)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("i", range(len(SCAN)))
def test_selective_scan_alone(pkg, tmp_path, dtype, i):
    cfg = model([G.scan(*SCAN[i])])
    w = G.weights(cfg, 70 + i)
    t, taps = agree(pkg, tmp_path, cfg, w, dtype, n=200, tol=ALONE[dtype] * (1 if dtype == "float32" else 2))
    for name in ("A_log", "D", "dt.b", "conv.b", "conv"):
        wrong = dict(w)
        wrong["l0.mix." + name] = w["l0.mix." + name][..., ::-1] if name == "conv" else w["l0.mix." + name] + 0.5
        assert name == "conv" and SCAN[i][3] == 1 or differs(cfg, wrong, t, taps, 1e-4), name


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("i", [0, 2, 5])
def test_selective_scan_in_portions(pkg, tmp_path, dtype, i):
    cfg = model([G.scan(*SCAN[i])])
    w = G.weights(cfg, 70 + i)
    portions_agree(pkg, tmp_path, cfg, w, dtype, 260, ([260], [64, 64, 65, 2], [1], [200, 1, 2, 3], [63, 2], [2, 2, 1, 130, 2]))


# ── joins, feed-forwards, loops ───────────────────────────────────────────────────────────────────────────────────────────
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("scales", [(1.0, 1.0), (1.3, -0.4), (0.0, 2.0)])
def test_scaled_sum_of_two_mixers(pkg, tmp_path, dtype, scales):
    cfg = model([G.gated_pair(4, 2, 16, 12, 20, 3, 8, 24, left=scales[0], right=scales[1])])
    w = G.weights(cfg, 81)
    t, taps = agree(pkg, tmp_path, cfg, w, dtype)
    if scales != (1.0, 1.0):
        assert differs(changed(cfg, lambda c: c["layers"][0]["mixer"].update(left_scale=scales[1], right_scale=scales[0])), w, t, taps)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("eps", [1e-6, 0.3])
def test_mean_of_two_normed_mixers(pkg, tmp_path, dtype, eps):
    """Results of very different size count the same; a large epsilon shows where it stands in every norm."""
    cfg = model([G.retention_pair(4, 2, 16, 12, 20, (0.9, 0.99), 8, 24, mlp=G.grouped_experts(6, 2, 20, 3, 2))] * 2, eps=eps)
    w = G.weights(cfg, 82)
    w["l0.mix.left.o"] *= 16.0
    w["l1.mix.right.o"] *= 16.0
    t, taps = agree(pkg, tmp_path, cfg, w, dtype)
    wrong = {k: v[::-1].copy() if k.endswith("left.out") else v for k, v in w.items()}
    assert differs(cfg, wrong, t, taps)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("ff", [1, 41, 160])
def test_dense_feed_forward_alone(pkg, tmp_path, dtype, ff):
    cfg = model([G.scan(8, 2, 2, 2, mlp=G.dense(ff))])
    w = G.weights(cfg, 83)
    silence(w, "o")
    t, taps = agree(pkg, tmp_path, cfg, w, dtype, n=33)
    for name in ("gate.b", "up.b", "down.b"):
        wrong = dict(w)
        wrong["l0.mlp." + name] = w["l0.mlp." + name] * 0.0
        assert differs(cfg, wrong, t, taps), name


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,top,ff,groups,keep,scale", [(12, 3, 41, 3, 2, 1.7), (16, 1, 64, 4, 1, 1.0), (6, 2, 20, 1, 1, 0.5), (2, 1, 33, 2, 1, 1.0), (8, 8, 24, 4, 4, 1.0), (70, 6, 24, 7, 3, 2.5),
                                                        (130, 2, 40, 2, 1, 1.0), (300, 7, 9, 10, 4, 1.2), (5, 2, 17, 5, 2, 3.0), (512, 8, 8, 64, 9, 1.0)])
@pytest.mark.parametrize("tokens", [1, 3, 90, 500])
def test_grouped_experts_alone(pkg, tmp_path, forms, dtype, n, top, ff, groups, keep, scale, tokens):
    """Routing and sorting in one launch and in two, every number of experts per lane; 32-bit: routers that read everything."""
    cfg = model([G.scan(8, 2, 2, 2, mlp=G.grouped_experts(n, top, ff, groups, keep, scale))])
    w = G.weights(cfg, 84, clear_routes=dtype == "bfloat16" and n <= 16)
    silence(w, "o")
    if dtype == "bfloat16" and n > 16:                                        # choices by the correction alone
        w["l0.mlp.correction"] = G.bf16(8.0 * np.random.default_rng(5).permutation(n) - 4.0 * n)
    _, taps = agree(pkg, tmp_path, cfg, w, dtype, n=tokens)
    h = forms.hits()
    assert bool(h.get("moe_route_sort")) == (tokens * top <= 1024) and bool(h.get("route_grouped")) == (tokens * top > 1024)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,n,top,groups,keep,tokens,fused", [(2080, 24, 8, 8, 4, 32, True), (4096, 33, 3, 3, 2, 128, True), (72, 64, 2, 4, 2, 128, True), (1024, 7, 4, 1, 1, 64, True),
                                                                  (1024, 7, 4, 1, 1, 65, False), (4100, 16, 2, 2, 1, 5, False), (512, 66, 2, 6, 3, 9, False)])
def test_update_router_and_sorted_list_in_one_launch(pkg, tmp_path, knobs, forms, dtype, width, n, top, groups, keep, tokens, fused):
    """4 and 16 waves, rows that end inside a step, two and four tiles of experts, as many pairs as threads; against the same in launches of their own.  Choices with a margin, so
    that the logits' order of summation (32-bit sums of `width` products: 1e-6 of their size) decides none; the stream then differs by the rounding of weights."""
    cfg = model([G.scan(8, 2, 2, 2, mlp=G.grouped_experts(n, top, 32, groups, keep, 1.4))], width=width)
    w = G.weights(cfg, 91, clear_routes=False)
    w["l0.mlp.correction"] = G.bf16(8.0 * np.random.default_rng(5).permutation(n) - 4.0 * n)
    taps = []
    for off in (None, 1):
        knobs.set(NO_STREAM_ROUTE=off)
        forms.reset()
        taps.append(taps_of(pkg, tmp_path, cfg, w, dtype, toks(cfg, tokens, 6)))
        assert bool(forms.hits().get("stream_route")) == (fused and not off)
    assert rel(taps[0], taps[1]) < {"float32": 2e-6, "bfloat16": 2.0 ** -9}[dtype]


@pytest.mark.parametrize("width", [1024, 4096])
def test_routers_of_32_bits_sum_in_parts(pkg, tmp_path, knobs, forms, width):
    """A row's two logits are of 12 and nearly alike, their experts' results opposite: what the layer adds is half of their difference, so the errors of the logits' sums are what the
    stream shows.  In one launch with the update and in launches of their own, against 64 bits.  Emulated, relative to the logits: sums of 128 products and sums of those 2.1 to 2.2e-7,
    sums of 256 2.9e-7; the ratio of two such errors over 1024 rows scatters by 0.03, so 1.2 lies four deviations from either."""
    cfg = model([G.scan(8, 2, 2, 2, mlp=G.grouped_experts(2, 2, 32))], width=width, vocab=1024)
    w, rng = G.weights(cfg, 92, clear_routes=False), np.random.default_rng(7)
    silence(w, "o")
    w["l0.norm2"][:], w["l0.mlp.correction"][:] = 1.0, 0.0
    w["l0.mlp.router"] = G.bf16(rng.standard_normal((2, width)) * 17.0 * width ** -0.5)
    r, rows = w["l0.mlp.router"].astype(np.float64), []
    while len(rows) < 1024:
        x = rng.standard_normal(width)
        x = G.bf16(x - (r[0] - r[1]) * ((r[0] - r[1]) @ x / ((r[0] - r[1]) @ (r[0] - r[1]))))
        level = r[0] @ x / np.sqrt(np.mean(x.astype(np.float64) ** 2))
        if 4.0 < abs(level) < 28.0:                                           # (negative, where weights follow the logits)
            rows.append(-x if level > 0 else x)
    w["embed"] = np.array(rows, np.float32)
    for part in ("gate", "up"):
        w["l0.mlp.e1." + part] = w["l0.mlp.e0." + part]
    w["l0.mlp.e1.down"] = -w["l0.mlp.e0.down"]
    x = w["embed"].astype(np.float64)
    h = L.unit_rms(x, cfg["norm"]["eps"])
    y = (L.silu(h @ w["l0.mlp.e0.gate"].T.astype(np.float64)) * (h @ w["l0.mlp.e0.up"].T.astype(np.float64))) @ w["l0.mlp.e0.down"].T.astype(np.float64)
    s = L.sigmoid(h @ r.T)
    want, path, errors = (s[:, 0] - s[:, 1]) / s.sum(axis=1), G.write_checkpoint(tmp_path, cfg, w), []
    for off in (None, 1):
        knobs.set(NO_STREAM_ROUTE=off)
        forms.reset()
        m, got = load(pkg, path, "float32"), []
        m.enable_taps()
        for i in range(0, 1024, 128):
            m.forward_rows([(1, np.arange(i, i + 128, dtype=np.uint32), 0)], [127])
            got.append(m.read_taps(128)[0].astype(np.float64))
            m.release(1)
        assert bool(forms.hits().get("stream_route")) == (not off)
        got = ((np.concatenate(got) - x) * y).sum(axis=1) / (y * y).sum(axis=1)
        errors.append(np.sqrt(np.mean((got - want) ** 2)))
    assert errors[0] < 1.2 * errors[1], errors


MISTAKES = {"weights read the correction": lambda s, c: s + c, "excluded choices are 0": None, "a group counts by its best": None, "choice without the correction": None}


@pytest.mark.parametrize("what", list(MISTAKES))
def test_routing_mistakes_would_show(pkg, tmp_path, monkeypatch, what):
    """All choice scores are negative, groups differ in their second best, corrections differ between the chosen."""
    cfg = model([G.scan(8, 2, 2, 2, mlp=G.grouped_experts(12, 4, 24, 3, 2, 1.3))])
    w = G.weights(cfg, 85, clear_routes=False)
    silence(w, "o")
    w["l0.mlp.correction"] = G.bf16(np.random.default_rng(3).uniform(-2.0, -1.2, 12))
    t, taps = agree(pkg, tmp_path, cfg, w, "float32", n=80)

    def wrong(logits, correction, top, groups, keep, scale):
        s = L.sigmoid(logits)
        base = s if what == "choice without the correction" else s + correction
        choice = base.reshape(groups, -1).copy()
        best = np.sort(choice, axis=1)
        rank = best[:, -1] if what == "a group counts by its best" else best[:, -2:].sum(axis=1)
        drop = np.argsort(-rank, kind="stable")[keep:]
        choice[drop] = 0.0 if what == "excluded choices are 0" else -np.inf
        ids = np.argsort(-choice.reshape(-1), kind="stable")[:top]
        v = (s + correction if what == "weights read the correction" else s)[ids]
        return ids, v / (v.sum() + 1e-20) * scale
    monkeypatch.setattr(L, "grouped_route", wrong)
    assert differs(cfg, w, t, taps)


def test_equal_choices_take_the_first_experts(pkg, tmp_path):
    cfg = model([G.scan(8, 2, 2, 2, mlp=G.grouped_experts(12, 3, 24, 4, 2))])
    w = G.weights(cfg, 86)
    silence(w, "o")
    w["l0.mlp.router"][:] = 0.0
    w["l0.mlp.correction"][:] = 0.0
    agree(pkg, tmp_path, cfg, w, "float32", n=20)


LOOPS = [(0, 3, 2), (0, 1, 3), (1, 3, 2), (2, 3, 4), (1, 2, 1), (0, 3, 1)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("loop", LOOPS)
def test_loops_alone(pkg, tmp_path, dtype, loop):
    """Every place of the loop; the stream after every run, in order; step vectors, the embedding and their place would show."""
    layers = [G.scan(40, 4, 3, 3, mlp=G.dense(30)), G.gated_pair(2, 1, 16, 16, 10, 2, 8, 8), G.retention_pair(2, 2, 8, 8, 12, (0.9,), 8, 8, mlp=G.dense(20))]
    cfg = model(layers, loop=loop)
    w = G.weights(cfg, 87)
    t, taps = agree(pkg, tmp_path, cfg, w, dtype, n=50, tol=ALONE[dtype] * (1 if dtype == "float32" else 2))
    assert len(taps) == 3 + (loop[1] - loop[0]) * (loop[2] - 1)
    edits = (lambda x: x["loop.step"].__setitem__(slice(None), x["loop.step"][::-1] + 0.1), lambda x: x["loop.in"].__setitem__(slice(None), np.roll(x["loop.in"], 72, axis=1)))
    for edit in edits[:1] if loop == (0, 3, 1) else edits:                    # (the only pass opens with x = x0)
        wrong = {k: v.copy() for k, v in w.items()}
        edit(wrong)
        assert differs(cfg, wrong, t, taps, 1e-2)


@pytest.mark.parametrize("dtype", DTYPES)
def test_passes_keep_caches_and_states_of_their_own(pkg, tmp_path, dtype):
    """Portions and single tokens through three passes over every kind of mixer: a pass that read another's cache or state would show at
    the first portion border, as it does between the second and a fourth pass of the oracle."""
    layers = [G.scan(40, 4, 3, 3), G.gated_pair(2, 1, 16, 16, 10, 2, 8, 8), G.retention_pair(2, 2, 8, 8, 12, (0.9, 1.0), 8, 8)]
    cfg = model(layers, loop=(0, 3, 3))
    w = G.weights(cfg, 88)
    w["loop.step"] *= 4.0
    t, want = portions_agree(pkg, tmp_path, cfg, w, dtype, 150, ([150], [1], [2], [40, 1, 3, 70, 2], [65, 2, 1]))


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_do_not_depend_on_batch_mates_or_pages(pkg, cases, dtype):
    """The same prompt in a fresh pool, in scattered pages and another slot, and beside others: equal to rounding."""
    cfg, w, path = cases("all")
    t = toks(cfg, 90, 7)
    m = load(pkg, path, dtype, tokens=400, seqs=4, slots=4)
    alone = feed(m, 1, t, [90])
    m.release(1)
    for s in (2, 3):
        m.forward_rows([(s, toks(cfg, 37, s), 0)], [])
    m.forward_rows([(4, t[:17], 0)], [])
    m.release(2)
    got = [m.forward_rows([(4, t[17:18], 17), (3, toks(cfg, 40, 9), 37)], [0])]
    got.append(m.forward_rows([(5, toks(cfg, 20, 5), 0), (4, t[18:], 18), (3, toks(cfg, 1, 9), 77)], list(range(20, 92))))
    assert rel(np.concatenate(got), alone[17:]) < (5e-6 if dtype == "float32" else 3e-2)


def test_missing_and_misshapen_weights_are_named(pkg, tmp_path):
    cfg = G.SEGETAR["loop"]
    w = G.weights(cfg, 1)
    for name, new in (("l0.norm1", None), ("l0.mix.left.q.norm", np.zeros(100, np.float32)), ("l2.mix.left.q.b", None), ("l2.mix.right.a2", np.zeros((60, 4), np.float32)),
                      ("l0.mlp.correction", np.zeros(11, np.float32)), ("l1.mix.A_log", np.zeros((75, 8), np.float32)), ("loop.step", np.zeros((2, 100), np.float32)),
                      ("loop.in", None), ("l0.mix.right.out", None), ("l1.mlp.down.b", None), ("l3.mlp.e6.gate", None), ("l2.mix.right.a1", None), ("head", None)):
        bad = {k: v for k, v in w.items() if k != name}
        if new is not None:
            bad[name] = new
        with pytest.raises(RuntimeError, match=name.replace(".", r"\.")):
            load(pkg, G.write_checkpoint(tmp_path / name, cfg, bad), "bfloat16")

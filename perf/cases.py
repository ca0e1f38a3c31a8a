"""What is measured: a batch of requests served through the runner, from the first prompt token to the last generated one.

One pass is what a serving program does for a batch: forwards over the prompts (at most `chunk` tokens each), then `steps` tokens per
sequence, one decode call each, with the token that the program's own sampler chose fed back, then the sequences are released.  The
last forward returns its logits, which depend on every token before them through the caches and states.  (The tokens of the greedy
sampler are the maxima of such rows and are not returned beside them: in models of random weights near ties are common.)

Weights are random.  Those of the INT4 models come from the runner's own generator, on the device, from the seed; the others are drawn
here and handed over tensor by tensor, as a checkpoint's are.  The layered models have a few layers of each kind at the benchmark's
sizes, with fewer experts: more of them would only repeat the same calls and make handing over slow.
"""
import os

import numpy as np
import torch

import __graft_entry__ as entry

# The models and sizes that the repository's benchmark names.  The expert model has 8 of its 48 layers: the choice of experts is a step
# function, and over all 48 of random weights two orders of summation come out several percent apart.  The unquantised model has half its
# layers, which are drawn and handed over.
QWEN3_30B = dict(num_layers=8, hidden=2048, num_heads=32, num_kv_heads=4, head_dim=128, vocab=151936, has_qk_norm=1, activation=0,
                 num_experts=128, top_k=8, expert_inter=768, norm_topk_prob=1, rms_eps=1e-6, rope_theta=1e6)
LLAMA_8B = dict(num_layers=32, hidden=4096, num_heads=32, num_kv_heads=8, head_dim=128, intermediate=14336, vocab=128256, has_qk_norm=0,
                activation=0, rms_eps=1e-5, rope_theta=5e5)
GEMMA3_27B = dict(num_layers=62, hidden=5376, num_heads=32, num_kv_heads=16, head_dim=128, intermediate=21504, vocab=262208, has_qk_norm=1,
                  activation=1, rms_eps=1e-6, rope_theta=1e6, rope_scaling_kind=1, rope_p0=8.0, sliding_window=1024, sliding_window_pattern=6,
                  sandwich_norms=1, embed_scale=73.5, rope_local_theta=10000.0)
QWEN3_06B = dict(num_layers=14, hidden=1024, num_heads=16, num_kv_heads=8, head_dim=128, intermediate=3072, vocab=151936, has_qk_norm=1,
                 activation=0, rms_eps=1e-6, rope_theta=1e6)
HOMOGENEOUS = {"qwen3-30b-a3b": QWEN3_30B, "llama31-8b": LLAMA_8B, "gemma3-27b": GEMMA3_27B, "qwen3-0.6b": QWEN3_06B}
LAYERED = dict(width=2048, heads=16, dim=128, rot_dim=64, vdim=128, q_rank=768, kv_rank=512, window=1024, ff=8192, rnn=2048, rnn_blocks=16,
               taps=4, vocab=32768, top=8, expert_ff=1024, side=256, lin_heads=16, lin_dim=64, lin_vdim=128, lin_rank=16, scan_inner=4096,
               scan_state=16, dt_rank=128, experts=24)
BIGRAM = dict(bigram_buckets=16384, bigram_mul_prev=40503, bigram_mul_cur=9973)
YARN = dict(rot_factor=4.0, rot_original=2048.0, rot_fast=32.0, rot_slow=1.0)
EPS = 1e-6                      # of the layered models


def listed():
    def case(name, model, seqs, prompt, steps, ragged=False, chunk=8192, layers=0, dtype=""):
        return dict(name=name, model=model, seqs=seqs, prompt=prompt, steps=steps, ragged=ragged, chunk=chunk, layers=layers, dtype=dtype)
    return [
        # one user of the INT4 expert model, a short question: nothing but latency
        case("int4-moe-one", "qwen3-30b-a3b", 1, 40, 32),
        # the benchmark's batch of 32 requests of 256 tokens
        case("int4-moe-batch", "qwen3-30b-a3b", 32, 256, 16),
        # one long document in a dense INT4 model: prompt attention, then decode over thousands of keys
        case("int4-dense-long", "llama31-8b", 1, 8100, 16),
        # a chat batch of unequal prompts in the same model, mostly decode
        case("int4-dense-chat", "llama31-8b", 12, 150, 32, ragged=True),
        # activation-ordered INT4, windows, norms on both sides of a sublayer
        case("int4-sandwich", "gemma3-27b", 5, 330, 8, ragged=True),
        # unquantised 16-bit projections: prompts of unequal length, in forwards of 2048 tokens
        case("f16-dense-prompts", "qwen3-0.6b", 5, 1500, 0, ragged=True, chunk=2048),
        # the same model decoding
        case("f16-dense-decode", "qwen3-0.6b", 8, 61, 32),
        # latent attention and linear recurrences, bf16: a long prompt and some answer
        case("nerenex-long", "nerenex", 1, 4096, 16, layers=6, dtype="bf16"),
        # the same family in 32 bits, the format that its results are checked in
        case("nerenex-f32", "nerenex", 4, 190, 16, ragged=True, layers=3, dtype="f32"),
        # latent attention with sinks beside dense and expert feed-forwards
        case("safolorn-batch", "safolorn", 8, 1000, 16, ragged=True, layers=2, dtype="bf16"),
        # selective scans, linear attention beside windowed attention, experts by groups, a loop
        case("segetar-batch", "segetar", 32, 256, 16, layers=3, dtype="bf16"),
        # heads mixed behind the softmax, scores by distance, shared experts
        case("fororax-pair", "fororax", 2, 2001, 16, layers=2, dtype="bf16"),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))
    model = rng.choice(["qwen3-30b-a3b", "llama31-8b", "qwen3-0.6b", "nerenex", "safolorn", "segetar", "fororax"])
    layers = {"nerenex": 3, "safolorn": 2, "segetar": 3, "fororax": 2}.get(model, 0)
    dtype = "" if not layers else rng.choice(["bf16", "bf16", "f32"])
    seqs = spread(1, 32)
    prompt = spread(8, max(8, min((1024 if dtype == "f32" else 8192) // seqs, 6000)))
    return dict(model=model, seqs=seqs, prompt=prompt, steps=rng.choice([0, spread(2, 24), spread(2, 24)]), ragged=rng.random() < 0.6,
                chunk=rng.choice([2048, 8192]), layers=layers, dtype=dtype)


# ── shapes of a pass ──

def lengths(case):
    """Prompt tokens of every sequence: unequal ones lie between half of the longest and the longest."""
    p = case["prompt"]
    return [p - (i * 37) % (p // 2 + 1) if case["ragged"] else p for i in range(case["seqs"])]


def portions(case):
    """Prompt forwards as lists of (sequence, first token, end): every forward takes up to `chunk` tokens, in the order of the sequences."""
    out, now, room = [], [], case["chunk"]
    for i, n in enumerate(lengths(case)):
        at = 0
        while at < n:
            take = min(n - at, room)
            now.append((i, at, at + take))
            at, room = at + take, room - take
            if room == 0:
                out, now, room = out + [now], [], case["chunk"]
    return out + [now] if now else out


def tokens_of(case, seed):
    rng = np.random.default_rng(seed)
    vocab = LAYERED["vocab"] if case["layers"] else HOMOGENEOUS[case["model"]]["vocab"]
    return [rng.integers(0, vocab, n + case["steps"]).astype(np.uint32) for n in lengths(case)]


# ── the program's side ──

def prepare(case, seed):
    pkg = entry.load_package()
    n = lengths(case)
    span = (max(n) + case["steps"] + 1 + 15) // 16 * 16
    common = dict(max_seq_len=span, kv_num_blocks=len(n) * span // 16 + 2, max_seqs=len(n),
                  max_tokens=max(len(n), min(case["chunk"], sum(n))))
    if case["layers"]:
        model = layered_model(pkg, case, seed, common)
    else:
        model = pkg.HipModel(group_size=128, **HOMOGENEOUS[case["model"]], **common)
        if case["model"] == "qwen3-0.6b":
            hand_over_dense(model, seed)
        elif case["model"] == "gemma3-27b":
            os.environ["FERRUM_HIP_SYNTH_DESC_ACT"] = "1"       # rows in activation order, as in the pack that the benchmark stands for
            try:
                model.init_synthetic(seed)
            finally:
                del os.environ["FERRUM_HIP_SYNTH_DESC_ACT"]
        else:
            model.init_synthetic(seed)
            if model.cfg.num_experts:
                hand_over_routers(model, seed)
    model.finalize()
    return dict(model=model, case=case, lengths=n, tokens=tokens_of(case, seed), portions=portions(case))


def run(state):
    model, steps, n, toks = state["model"], state["case"]["steps"], state["lengths"], state["tokens"]
    ids = list(range(len(n)))
    logits = []
    for part in state["portions"]:
        items = [(i, toks[i][a:b], a, b == n[i]) for i, a, b in part]
        _, got = model.unified_forward(items, want_logits=steps == 0)
        if steps == 0:
            logits.append(got)
    for s in range(steps - 1):
        model.decode_steps(ids, [toks[i][n[i] + s] for i in ids], 1)
    if steps:
        _, got = model.unified_forward([(i, toks[i][-1:], n[i] + steps - 1, True) for i in ids], want_logits=True)
        logits.append(got)
    for i in ids:
        model.release(i)
    return logits


# ── layered models: layers as the benchmark builds them ──

def layer_kinds(case):
    """The layers in order, as arguments of LayerSpec; the whole-model arguments; the loop."""
    z, fam, count = LAYERED, case["model"], case["layers"]
    if fam == "nerenex":
        rec = dict(mixer=2, ff=1, ff_width=z["ff"], rnn_width=z["rnn"], rnn_blocks=z["rnn_blocks"], conv_taps=z["taps"])
        att = dict(mixer=1, ff=1, ff_width=z["ff"], heads=z["heads"], dim=z["dim"], rot_dim=z["rot_dim"], vdim=z["vdim"], q_rank=z["q_rank"],
                   kv_rank=z["kv_rank"], rot_dims=z["rot_dim"], window=z["window"], scale=(z["dim"] + z["rot_dim"]) ** -0.5, rot_base=1e6)
        return [att if i % 3 == 2 else rec for i in range(count)], dict(residual_mult=0.7, **BIGRAM), {}
    if fam == "safolorn":                                   # every second layer with experts, on the keys of the layer before it
        dense = dict(ff=2, ff_width=z["ff"], ff_limit=7.0, kv_source=0)
        att = dict(mixer=1, heads=z["heads"], dim=z["dim"], rot_dim=z["rot_dim"], vdim=z["vdim"], kv_rank=z["kv_rank"], rot_dims=z["rot_dim"],
                   window=-1, scale=(z["dim"] + z["rot_dim"]) ** -0.5, rot_base=1e6, attn_flags=3, **YARN)
        return ([dict(att, **(dict(ff=3, ff_width=z["expert_ff"], experts=z["experts"], top=z["top"], kv_source=i) if i % 2 else dense))
                 for i in range(count)], dict(residual_mult=1.0, block=1, token_side_dim=z["side"], untied_head=1), {})
    if fam == "segetar":                                    # the two attention layers run twice
        moe = dict(ff=5, ff_width=z["expert_ff"], experts=z["experts"], top=z["top"], route_groups=8, route_keep=4, route_scale=2.5)
        scan = dict(mixer=6, scan_inner=z["scan_inner"], scan_state=z["scan_state"], scan_dt_rank=z["dt_rank"], conv_taps=z["taps"], ff=4,
                    ff_width=z["ff"])
        pair = dict(mixer=3, heads=z["heads"], kv_heads=z["heads"] // 4, dim=z["dim"], vdim=z["vdim"], window=z["window"], scale=z["dim"] ** -0.5,
                    lin_heads=z["lin_heads"], lin_dim=z["lin_dim"], lin_vdim=z["lin_vdim"], **moe)
        gated = dict(pair, mixer2=4, attn_flags=4, rot_dims=z["dim"], rot_base=1e6, lin_rank=z["lin_rank"], lin_tau=16.0, left_scale=1.0,
                     right_scale=1.0)
        retention = dict(pair, mixer2=5, join=1, attn_flags=1, lin_rot_dims=z["lin_dim"], lin_rot_base=1e4)
        return ([[scan, gated, retention][i % 3] for i in range(count)], dict(residual_mult=1.0, block=2, untied_head=1),
                dict(loop_start=1, loop_stop=3, loop_times=2))
    base = dict(mixer=3, heads=z["heads"], kv_heads=z["heads"] // 4, dim=z["dim"], vdim=z["vdim"], window=-1, scale=z["dim"] ** -0.5, ff=6,
                ff_width=z["expert_ff"], ff_limit=7.0, experts=z["experts"], identity_experts=z["experts"] // 4, top=z["top"], route_groups=1,
                route_keep=1, route_scale=1.0, shared_width=z["expert_ff"], shared_limit=7.0)
    talk, far = dict(base, attn_flags=1 | 2 | 4 | 8 | 32 | 64 | 128), dict(base, attn_flags=1 | 8 | 16)
    return ([[talk, far][i % 2] for i in range(count)],
            dict(residual_mult=1.0, block=3, untied_head=1, stream_mult=2.2, embed_scale=1.0, logit_softcap=30.0), {})


def layered_model(pkg, case, seed, common):
    layers, whole, loop = layer_kinds(case)
    if case["model"] == "fororax":
        whole = dict(whole, position_rows=common["max_seq_len"])
    config = pkg.LayeredConfig(dtype=0 if case["dtype"] == "bf16" else 1, state_slots=common["max_seqs"], **whole, **loop)
    model = pkg.HipModel(layered=(config, [pkg.LayerSpec(**k) for k in layers]), num_layers=len(layers), hidden=LAYERED["width"],
                         vocab=LAYERED["vocab"], rms_eps=EPS, **common)
    for name, w in layered_weights(case, seed, common["max_seq_len"]):
        w = w.cpu().numpy()
        if "*" in name:                                     # one tensor per expert
            for e, part in enumerate(w):
                model.set_tensor(name.replace("*", f"e{e}"), part)
        else:
            model.set_tensor(name, w)
    return model


def layered_weights(case, seed, positions=0):
    """Names and float32 tensors, values that 16 bits hold; drawn on the device.  A star in a name: the first axis counts experts."""
    gen = torch.Generator("cuda").manual_seed(seed)

    def mat(*shape, std=None):
        return (torch.randn(shape, generator=gen, device="cuda") * (std or shape[-1] ** -0.5)).bfloat16().float()

    def vec(*shape, mean=0.0, std=0.2):
        return (torch.randn(shape, generator=gen, device="cuda") * std + mean).bfloat16().float()

    def flat(lo, hi, *shape):
        return (torch.rand(shape, generator=gen, device="cuda") * (hi - lo) + lo).bfloat16().float()

    z, fam = LAYERED, case["model"]
    D, V = z["width"], z["vocab"]
    layers, whole, loop = layer_kinds(case)
    yield "embed", mat(V, D, std=1.0)
    if fam == "nerenex":
        yield "bigram", mat(BIGRAM["bigram_buckets"] + 1, D, std=0.7)
        yield "final.norm", vec(D)
    else:
        yield "head", mat(V, D)
        yield "final.norm", flat(0.6, 1.5) if fam == "safolorn" else vec(D, mean=1.0)
    if fam == "safolorn":
        yield "side.embed", mat(V, len(layers) * z["side"], std=1.0)
    if fam == "fororax":
        yield "pos", mat(positions, D, std=0.6)
    if loop:
        eye = torch.eye(D, device="cuda")
        yield "loop.in", (mat(D, 2 * D, std=0.4 * D ** -0.5) + torch.cat([0.8 * eye, 0.3 * eye], 1)).bfloat16().float()
        yield "loop.step", vec(loop["loop_times"], D, std=0.5)
    for i, k in enumerate(layers):
        p, x = f"l{i}.", f"l{i}.mix."
        for s in ("1", "2"):
            yield p + "norm" + s, flat(0.6, 1.5) if fam == "safolorn" else vec(D, mean=0.0 if fam == "nerenex" else 1.0)
        if fam == "nerenex":
            for s in ("1", "2"):
                yield p + "rg" + s, mat(D, D)
                yield p + "rg" + s + ".b", vec(D)
        if k["mixer"] == 1:
            H, R, hd = k["heads"], k["kv_rank"], k["dim"] + k["rot_dim"]
            if k.get("q_rank"):
                yield x + "dq", mat(k["q_rank"], D)
                yield x + "dq.norm", vec(k["q_rank"], mean=1.0)
                yield x + "uq", mat(H * hd, k["q_rank"], std=1.6 * k["q_rank"] ** -0.5)
                yield x + "g", mat(H, D)
            else:
                yield x + "q", mat(H * hd, D, std=1.6 * D ** -0.5)
                yield x + "sink", vec(H, mean=2.0, std=1.5)
            if not k.get("kv_source"):
                yield x + "dkv", mat(R + k["rot_dim"], D)
                yield x + "dkv.norm", vec(R, mean=1.0)
            yield x + "uk", mat(H * k["dim"], R, std=1.6 * R ** -0.5)
            yield x + "uv", mat(H * k["vdim"], R)
            yield x + "o", mat(D, H * k["vdim"])
        elif k["mixer"] == 2:
            W, nb = k["rnn_width"], k["rnn_blocks"]
            for n in ("y", "x"):
                yield x + n, mat(W, D)
                yield x + n + ".b", vec(W)
            yield x + "conv", mat(W, k["conv_taps"], std=0.6)
            yield x + "conv.b", vec(W)
            for n in ("ra", "ri"):
                yield x + n, mat(nb, W // nb, W // nb)
                yield x + n + ".b", vec(nb, W // nb)
            yield x + "lam", flat(-6.0, 1.0, W)             # decays from almost 1 to almost 0
            yield x + "o", mat(D, W)
        elif k["mixer"] == 6:
            W, N, R = k["scan_inner"], k["scan_state"], k["scan_dt_rank"]
            yield x + "in", mat(2 * W, D)
            yield x + "conv", mat(W, k["conv_taps"], std=0.6)
            yield x + "conv.b", vec(W)
            yield x + "x", mat(R + 2 * N, W)
            yield x + "dt", mat(W, R, std=0.7 * R ** -0.5)
            yield x + "dt.b", vec(W, std=1.5, mean=-2.0)
            yield x + "A_log", flat(-3.0, 2.5, W, N)
            yield x + "D", vec(W, mean=1.0)
            yield x + "o", mat(D, W)
        else:
            H, G, flags = k["heads"], k["kv_heads"], k.get("attn_flags", 0)
            left = x + "left." if k.get("mixer2") else x
            for n, rows in (("q", H * k["dim"]), ("k", G * k["dim"]), ("v", G * k["vdim"])):
                yield left + n, mat(rows, D)
                if flags & 4:
                    yield left + n + ".b", vec(rows, std=0.5)
                if n != "v":                                # one gain for every head, or one per number
                    yield left + n + ".norm", vec(k["dim"] if flags & 8 else rows, mean=1.6)
            yield left + "o", mat(D, H * k["vdim"])
            if k.get("mixer2"):
                Hr, kd, vd, right = k["lin_heads"], k["lin_dim"], k["lin_vdim"], x + "right."
                for n, rows in (("q", Hr * kd), ("k", Hr * kd), ("v", Hr * vd), ("g", Hr * vd)):
                    yield right + n, mat(rows, D)
                yield right + "o", mat(D, Hr * vd)
                if k["mixer2"] == 4:
                    yield left + "g", mat(H, D)
                    yield right + "a1", mat(k["lin_rank"], D)
                    yield right + "a2", mat(Hr * kd, k["lin_rank"], std=2.0 * k["lin_rank"] ** -0.5)
                    yield right + "a2.b", vec(Hr * kd, std=3.0)
                    yield right + "norm", vec(vd, mean=1.0)
                else:
                    yield right + "decay", 1.0 - 2.0 ** -torch.linspace(1.0, 10.0, Hr, device="cuda")
                    yield left + "out", vec(D, mean=1.0)
                    yield right + "out", vec(D, mean=1.0)
            elif flags & 32:
                yield x + "sink", vec(H, std=1.0, mean=1.0)
                yield x + "talk", (0.6 * torch.eye(H, device="cuda") + vec(H, H, std=0.7 * H ** -0.5)).bfloat16().float()
                yield x + "g", mat(H * k["vdim"], D)
                yield x + "o.b", vec(D)
            else:
                yield x + "r1", flat(0.2, 1.5, H)
                yield x + "r2", torch.exp(flat(-5.0, 1.0, H)).bfloat16().float()
        if fam == "safolorn":
            yield p + "side.gate", mat(z["side"], D)
            yield p + "side.proj", mat(D, z["side"])
            yield p + "side.norm", vec(D, mean=0.4, std=0.3)
        F, E = k["ff_width"], k.get("experts", 0)
        if k["ff"] == 1:
            yield p + "mlp.up", mat(F, D, std=2.0 * D ** -0.5)
            yield p + "mlp.down", mat(D, F)
            yield p + "mlp.act", flat(-1.0, 1.0, 2)
        elif not E:
            for n in ("gate", "up"):
                yield p + "mlp." + n, mat(F, D)
            yield p + "mlp.down", mat(D, F)
            if k["ff"] == 4:
                for n, rows in (("gate", F), ("up", F), ("down", D)):
                    yield p + f"mlp.{n}.b", vec(rows)
        else:
            choices = E + k.get("identity_experts", 0)
            yield p + "mlp.router", mat(choices, D, std=1.5 * D ** -0.5)
            if k["ff"] == 3:
                yield p + "mlp.router.b", vec(choices, std=0.5)
            else:
                yield p + "mlp.correction", vec(choices, std=0.4 if k["ff"] == 5 else 0.1)
                yield p + "mlp.*.gate", mat(E, F, D)
            yield p + "mlp.*.up", mat(E, F, D)
            # (what experts of nearly equal rank add is kept small beside the stream, as in deep models, where their normalised weights are alike)
            yield p + "mlp.*.down", mat(E, D, F, std=(0.25 if k["ff"] == 5 else 1.0) * F ** -0.5)
            if k.get("shared_width"):
                for n, rows, cols in (("gate", F, D), ("up", F, D), ("down", D, F), ("sg", 1, D)):
                    yield p + "mlp.shared." + n, mat(rows, cols)


# ── a dense model's weights, drawn here ──

def dense_weights(c, seed):
    """(layer or −1, name, float32 tensor): values that fp16 holds."""
    gen = torch.Generator("cuda").manual_seed(seed)

    def mat(n, k, std=None):
        return (torch.randn((n, k), generator=gen, device="cuda") * (std or k ** -0.5)).half().float()

    def gain(n):
        return (1.0 + 0.1 * torch.randn(n, generator=gen, device="cuda")).half().float()

    H, q, kv, F = c["hidden"], c["num_heads"] * c["head_dim"], c["num_kv_heads"] * c["head_dim"], c["intermediate"]
    yield -1, "embed", mat(c["vocab"], H, 0.02)
    yield -1, "final_norm", gain(H)
    for li in range(c["num_layers"]):
        for name in ("input_ln", "post_ln"):
            yield li, name, gain(H)
        for name in ("q_norm", "k_norm"):
            yield li, name, gain(c["head_dim"])
        for name, n, k in (("qkv", q + 2 * kv, H), ("o", H, q), ("gate_up", 2 * F, H), ("down", H, F)):
            yield li, name, mat(n, k)


def hand_over_dense(model, seed):
    for li, name, w in dense_weights(QWEN3_06B, seed):
        w = w.cpu().numpy()
        if li < 0:
            model.set_global(name, w)               # (without an output table of its own the embedding serves as one)
        elif w.ndim == 1:
            model.set_layer_dense(li, name, w)
        else:
            model.set_dense(li, name, w, w.shape[1], w.shape[0])


def hand_over_routers(model, seed):
    """Scores as far apart as a trained router's, so that the last chosen expert weighs little and a near tie for its place does too."""
    rng = np.random.default_rng(seed)
    for li in range(model.cfg.num_layers):
        scores = rng.standard_normal((model.cfg.num_experts, model.cfg.hidden), np.float32) * 4.0 * model.cfg.hidden ** -0.5
        model.set_layer_dense(li, "router", scores)


# ── what a pass cannot do without ──

def model_layers(case):
    """Per layer: weights of every token, weights of an expert, experts, chosen, cached values per token (numbers that decode reads),
    operations per query-key pair, window."""
    if not case["layers"]:
        c = HOMOGENEOUS[case["model"]]
        H, hd, q, kv = c["hidden"], c["head_dim"], c["num_heads"], c["num_kv_heads"]
        attn = H * (q + 2 * kv) * hd + q * hd * H
        E = c.get("num_experts", 0)
        for i in range(c["num_layers"]):
            local = c.get("sliding_window_pattern") and (i + 1) % c["sliding_window_pattern"]
            yield (attn + (E * H if E else 3 * H * c["intermediate"]), 3 * H * c.get("expert_inter", 0), E, c.get("top_k", 0), 2 * kv * hd,
                   4 * q * hd, c["sliding_window"] if local else 0)
        return
    D = LAYERED["width"]
    layers, whole, loop = layer_kinds(case)
    runs = layers + layers[loop["loop_start"]:loop["loop_stop"]] * (loop["loop_times"] - 1) if loop else layers
    for k in runs:
        w, cache, pair, experts = 0, 0, 0, k.get("experts", 0)
        if k["mixer"] == 1:
            H, hd = k["heads"], k["dim"] + k["rot_dim"]
            w += (D * k["q_rank"] + k["q_rank"] * H * hd if k.get("q_rank") else D * H * hd) + D * (k["kv_rank"] + k["rot_dim"])
            w += k["kv_rank"] * H * (k["dim"] + k["vdim"]) + H * k["vdim"] * D
            cache, pair = k["kv_rank"] + k["rot_dim"], 2 * H * (hd + k["vdim"])
        elif k["mixer"] == 2:
            w += 3 * D * k["rnn_width"] + 2 * k["rnn_width"] ** 2 // k["rnn_blocks"]
        elif k["mixer"] == 3:
            H, G = k["heads"], k["kv_heads"]
            w += D * (H + G) * k["dim"] + D * G * k["vdim"] + H * k["vdim"] * D * (2 if k.get("attn_flags", 0) & 64 else 1)
            cache, pair = G * (k["dim"] + k["vdim"]), 2 * H * (k["dim"] + k["vdim"]) + (2 * H * H if k.get("attn_flags", 0) & 32 else 0)
        else:
            w += 3 * D * k["scan_inner"] + k["scan_inner"] * (2 * k["scan_dt_rank"] + 2 * k["scan_state"])
        if k.get("mixer2"):
            w += D * k["lin_heads"] * (2 * k["lin_dim"] + 3 * k["lin_vdim"])
        if case["model"] == "nerenex":
            w += 2 * D * D
        if whole.get("token_side_dim"):
            w += 2 * D * whole["token_side_dim"]
        per = {1: 2, 2: 3, 3: 2, 4: 3, 5: 3, 6: 3}[k["ff"]] * D * k["ff_width"]
        w += D * (experts + k.get("identity_experts", 0)) if experts else per
        if k.get("shared_width"):
            w += 3 * D * k["shared_width"]
        yield w, per if experts else 0, experts, k.get("top", 0), cache, pair, max(k.get("window", 0), 0)


def work(case):
    n, steps = lengths(case), case["steps"]
    c = LAYERED if case["layers"] else HOMOGENEOUS[case["model"]]
    width, number = c.get("width") or c["hidden"], 4.0 if case["dtype"] == "f32" else 2.0
    weight = number if case["layers"] or case["model"] == "qwen3-0.6b" else 0.5 + 2.0 / 128
    forwards = [sum(b - a for _, a, b in part) for part in portions(case)] + [len(n)] * steps
    bytes_, flops = 0.0, 0.0
    for w, expert, experts, top, cache, pair, window in model_layers(case):
        def seen(p):
            return min(p + 1, window) if window else p + 1
        for t in forwards:
            touched = experts * (1.0 - (1.0 - top / experts) ** t) if experts else 0.0
            bytes_ += (w + touched * expert) * weight
            flops += 2.0 * t * (w + top * expert)
        for m in n:
            keys = sum(seen(p) for p in range(m + steps))
            flops += pair * keys
            bytes_ += cache * number * (m + steps + sum(seen(m + s) for s in range(steps)))
    heads = len(n) * (1 + steps)
    bytes_ += (1 + steps) * width * c["vocab"] * number + len(n) * c["vocab"] * 4.0 + sum(forwards) * width * number
    flops += 2.0 * heads * width * c["vocab"]
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times what forwards of another size, whose sums run in another order, differ by.  Measured: 1e-6 in 32 bits; 0.002 to 0.003
    in the dense fp16 models, 0.001 to 0.002 in fororax, 0.0035 in safolorn, 0.007 in nerenex; up to 0.011 where a near tie between experts falls
    the other way (the INT4 expert model, segetar)."""
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": {"llama31-8b": 0.012, "gemma3-27b": 0.008, "qwen3-0.6b": 0.01, "fororax": 0.01, "safolorn": 0.014}.get(case["model"], 0.03)}


# ── the same logits in 64 bits ──

def exact(case, seed):
    """Plain attention over all tokens at once; one row of logits per sequence.  None for the expert models: nearly equal router scores
    choose other experts in another precision, so no nearby value is the only right one; none for the largest dense model, which takes too
    long."""
    if case["model"] == "nerenex":
        rows = nerenex_exact(case, seed)
    elif case["model"] in ("llama31-8b", "qwen3-0.6b"):
        rows = dense_exact(case, seed)
    else:
        return None
    if case["steps"]:
        return [rows]
    n = lengths(case)
    return [rows[[i for i, _, b in part if b == n[i]]] for part in portions(case)]


def unit_rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def causal_softmax(scores, window=0):
    n = scores.shape[-1]
    d = torch.arange(n, device="cuda")[:, None] - torch.arange(n, device="cuda")[None, :]
    return torch.softmax(scores.masked_fill((d < 0) | (d >= (window or n)), float("-inf")), -1)


def dense_exact(case, seed):
    c = HOMOGENEOUS[case["model"]]
    nq, nkv, hd, eps = c["num_heads"], c["num_kv_heads"], c["head_dim"], c["rms_eps"]
    toks = [torch.from_numpy(t.astype(np.int64)).cuda() for t in tokens_of(case, seed)]
    source = given_layers(c, seed) if case["model"] == "qwen3-0.6b" else generated_layers(c, seed)
    table, head, final = next(source)
    xs = [table(t) for t in toks]
    angle = torch.arange(max(map(len, toks)), device="cuda", dtype=torch.float64)[:, None] * (
        c["rope_theta"] ** (-torch.arange(hd // 2, device="cuda", dtype=torch.float64) * 2 / hd))
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def turned(x):
        a, b = x[..., :hd // 2], x[..., hd // 2:]
        co, si = cos[:len(x)], sin[:len(x)]
        return torch.cat([a * co - b * si, b * co + a * si], -1)

    for w in source:
        for i, x in enumerate(xs):
            qkv = (unit_rms(x, eps) * w["input_ln"]) @ w["qkv"].T
            q, k, v = (part.reshape(len(x), -1, hd) for part in qkv.split([nq * hd, nkv * hd, nkv * hd], 1))
            if c["has_qk_norm"]:
                q, k = unit_rms(q, eps) * w["q_norm"], unit_rms(k, eps) * w["k_norm"]
            q, k, out = turned(q), turned(k), torch.empty_like(q)
            for h in range(nq):
                out[:, h] = causal_softmax(q[:, h] @ k[:, h * nkv // nq].T * hd ** -0.5) @ v[:, h * nkv // nq]
            x = x + out.reshape(len(x), -1) @ w["o"].T
            gate, up = ((unit_rms(x, eps) * w["post_ln"]) @ w["gate_up"].T).chunk(2, 1)
            xs[i] = x + (torch.nn.functional.silu(gate) * up) @ w["down"].T
    return (unit_rms(torch.stack([x[-1] for x in xs]), eps) * final) @ head().T


def given_layers(c, seed):
    source = dense_weights(c, seed)
    embed, final = next(source)[2], next(source)[2].double()
    yield lambda t: embed[t].double(), lambda: embed.double(), final
    for _ in range(c["num_layers"]):
        yield {name: w.double() for _, name, w in (next(source) for _ in range(8))}


def mix64(x):
    """The runner's generator: one round of splitmix over int64 tensors (products wrap, shifts are unsigned)."""
    def down(v, s):
        return (v >> s) & ((1 << (64 - s)) - 1)
    x = x - 0x61C8864680B583EB
    x = (x ^ down(x, 30)) * -0x40A7B892E31B1A47
    x = (x ^ down(x, 27)) * -0x6B2FB644ECCEEE15
    return x ^ down(x, 31)


def generated_layers(c, seed):
    """The values that the runner's generator makes for a dense INT4 model."""
    H, hd = c["hidden"], c["head_dim"]
    q, kv, F = c["num_heads"] * hd, c["num_kv_heads"] * hd, c["intermediate"]

    def numbers(count, key, start=0):
        key = (key + (1 << 63)) % (1 << 64) - (1 << 63)
        return mix64(torch.arange(start, start + count, device="cuda") + key)

    def normal(rows, cols, key, pick=None):
        r = numbers(rows * cols, key) if pick is None else mix64(torch.arange(cols, device="cuda") + (pick[:, None] * cols + key))
        u1, u2 = (((r >> 40) & 0xFFFFFF).float() + 0.5) / 16777216.0, ((r >> 16) & 0xFFFFFF).float() / 16777216.0
        return (0.02 * torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(6.2831853 * u2)).half().double().reshape(-1, cols)

    def int4(n, k, key):
        """[n, k]; stored as [n / 64][k / 128][4 tiles of 16 columns][4 × 16 lanes][4 words of 8 codes]."""
        g = k // 128
        word = (numbers(n * k // 8, key) >> 16) & 0xFFFFFFFF
        lo, hi = (torch.tensor([[0, 4, 2, 6], [1, 5, 3, 7]], device="cuda") * 4).unbind()
        code = torch.stack([(word[:, None] >> lo) & 15, (word[:, None] >> hi) & 15], 1).to(torch.int8)     # [word][step of its pair][j]
        code[code == 0] = 8
        code = code.reshape(n // 64, g, 4, 4, 16, 2, 2, 2, 4)              # st, group, tile, a, b, pair of steps, half of j, step, j
        code = code.permute(0, 2, 4, 1, 5, 7, 3, 6, 8).reshape(n, g, 128)
        f = np.float32(1.0) / (np.float32(0.25) * np.sqrt(np.float32(k)))
        low, high = np.float32(0.01) * f, np.float32(0.1) * f
        u = ((numbers(n * g, key ^ 0x5ca1e5) >> 40) & 0xFFFFFF).float() / 16777216.0
        scale = (float(low) + u * float(high - low)).half().double()       # [n / 64][k / 128][16][4 tiles]
        scale = scale.reshape(n // 64, g, 16, 4).permute(0, 3, 2, 1).reshape(n, g, 1)
        return ((code.double() - 8.0) * scale).reshape(n, k)

    yield (lambda t: normal(0, H, seed ^ 0xe0bed, t)), (lambda: normal(c["vocab"], H, seed ^ 0x1a4ead)), 1.0
    for li in range(c["num_layers"]):
        key = seed + 0x1000003 * (li + 1)
        yield dict(input_ln=1.0, post_ln=1.0, q_norm=1.0, k_norm=1.0, qkv=int4(q + 2 * kv, H, key ^ 0x11), o=int4(H, q, key ^ 0x22),
                   gate_up=int4(2 * F, H, key ^ 0x44), down=int4(H, F, key ^ 0x55))


def nerenex_exact(case, seed):
    z = LAYERED
    H, dim, rot, vd, R = z["heads"], z["dim"], z["rot_dim"], z["vdim"], z["kv_rank"]
    source = layered_weights(case, seed)
    embed, bigram, final = (next(source)[1] for _ in range(3))
    xs = []
    for t in tokens_of(case, seed):
        t = t.astype(np.int64)
        rows = np.concatenate([[BIGRAM["bigram_buckets"]], (t[:-1] * BIGRAM["bigram_mul_prev"] + t[1:] * BIGRAM["bigram_mul_cur"])
                               % BIGRAM["bigram_buckets"]])
        xs.append(embed[torch.from_numpy(t).cuda()].double() + bigram[torch.from_numpy(rows).cuda()].double())

    def turned(x):                                          # pairs (2i, 2i + 1) of the last axis
        angle = torch.arange(len(x), device="cuda", dtype=torch.float64)[:, None] * (
            1e6 ** (-torch.arange(rot // 2, device="cuda", dtype=torch.float64) * 2 / rot))
        shape = (len(x),) + (1,) * (x.ndim - 2) + (rot // 2,)
        co, si, u, v = torch.cos(angle).reshape(shape), torch.sin(angle).reshape(shape), x[..., 0::2], x[..., 1::2]
        return torch.stack([u * co - v * si, v * co + u * si], -1).reshape(x.shape)

    def attention(h, w):
        n = len(h)
        q = ((unit_rms(h @ w["dq"].T, EPS) * w["dq.norm"]) @ w["uq"].T).reshape(n, H, dim + rot)
        kv = h @ w["dkv"].T
        latent, key = unit_rms(kv[:, :R], EPS) * w["dkv.norm"], turned(kv[:, R:])
        plain, value, qr = (latent @ w["uk"].T).reshape(n, H, dim), (latent @ w["uv"].T).reshape(n, H, vd), turned(q[..., dim:])
        out = torch.empty(n, H, vd, dtype=torch.float64, device="cuda")
        for a in range(H):
            s = (q[:, a, :dim] @ plain[:, a].T + qr[:, a] @ key.T) * (dim + rot) ** -0.5
            out[:, a] = causal_softmax(s, z["window"]) @ value[:, a]
        return (out * torch.sigmoid(h @ w["g"].T)[:, :, None]).reshape(n, -1) @ w["o"].T

    def recurrence(h, w):
        n, taps = len(h), z["taps"]
        y = torch.nn.functional.gelu(h @ w["y"].T + w["y.b"], approximate="tanh")
        u = h @ w["x"].T + w["x.b"]
        u = torch.cat([u.new_zeros(taps - 1, u.shape[1]), u])
        u = sum(u[j:j + n] * w["conv"][:, j] for j in range(taps)) + w["conv.b"]
        parts = u.reshape(n, z["rnn_blocks"], -1).transpose(0, 1)
        r, i = (torch.sigmoid((parts @ w[g].transpose(1, 2)).transpose(0, 1).reshape(n, -1) + w[g + ".b"].reshape(-1)) for g in ("ra", "ri"))
        log_a = -8.0 * r * torch.nn.functional.softplus(w["lam"])
        a, add = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * i * u
        state, out = torch.zeros_like(add[0]), torch.empty_like(add)
        for t in range(n):
            state = torch.addcmul(add[t], a[t], state)
            out[t] = state
        return (out * y) @ w["o"].T

    for i, k in enumerate(layer_kinds(case)[0]):
        w = {}
        while f"l{i}.mlp.act" not in w:
            name, value = next(source)
            w[name] = value.double()
        layer = {name[len(f"l{i}."):]: v for name, v in w.items()}
        mix = {name[4:]: v for name, v in layer.items() if name.startswith("mix.")}
        p, q = torch.nn.functional.softplus(layer["mlp.act"])

        def feed_forward(h, _):
            s = h @ layer["mlp.up"].T
            neg = s.clamp(max=0.0)
            return (torch.where(s > 0, p * s * s, (0.5 + q) * (torch.expm1(neg) - neg)) + s / 2) @ layer["mlp.down"].T

        for j, x in enumerate(xs):
            for s, sub in (("1", attention if k["mixer"] == 1 else recurrence), ("2", feed_forward)):
                gated = sub(x, mix) * torch.sigmoid(x @ layer["rg" + s].T + layer["rg" + s + ".b"])
                x = x + 0.7 * unit_rms(gated, EPS) * (1.0 + layer["norm" + s])
            xs[j] = x
    return (unit_rms(torch.stack([x[-1] for x in xs]), EPS) * (1.0 + final.double())) @ embed.double().T

"""GPU parity tests: every hot-path op through the C ABI (libferrum_hip.so) vs the CPU oracle on the
same seeded inputs.  Tolerances are the reference's own op_diff buckets
(ferrum-testkit/src/op_diff/mod.rs:46-49: NMSE fp16 1e-6, attention 5e-3, fp16 round-trip 3e-3)
unless a tighter one is written in the test; integer outputs are bit-exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NMSE_FP16_TOL = 1e-6
NMSE_ATTN_TOL = 5e-3


@pytest.fixture(scope="module")
def env():
    import torch
    import __graft_entry__ as ge
    assert torch.cuda.is_available(), "gpu tests need a GPU"
    pkg = ge.load_package()
    pkg.load_library()          # raises if the HIP extension is missing — no fallback
    from oracle import oracle as O
    O.build()
    ctx = pkg.HipBackend.new_context()
    return pkg, pkg.HipBackend, ctx, O, torch


def f16r(a):
    return np.asarray(a, np.float32).astype(np.float16).astype(np.float32)


def nmse(ref, got):
    ref, got = np.asarray(ref, np.float64).ravel(), np.asarray(got, np.float64).ravel()
    return float(((ref - got) ** 2).mean() / max((ref ** 2).mean(), 1e-30))


def dev16(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda").half().contiguous()


def host(t):
    return t.float().cpu().numpy()


# ── norms / elementwise ──────────────────────────────────────────────────────
@pytest.mark.parametrize("tokens,dim", [(1, 768), (7, 1024), (3, 4100), (2, 8192)])
def test_layer_norm_and_gelu_core_ops(env, tokens, dim):
    # Backend::layer_norm / Backend::gelu (required core ops of the trait; CPU cpu.rs:2081-2122) + the event timer
    pkg, B, ctx, O, torch = env
    import ctypes as C
    rng = np.random.default_rng(dim * 3 + tokens)
    x = f16r(rng.standard_normal((tokens, dim)) * 3 + 0.7)
    g, b = f16r(1 + 0.2 * rng.standard_normal(dim)), f16r(0.1 * rng.standard_normal(dim))
    out = torch.empty(tokens, dim, dtype=torch.float16, device="cuda")
    lib = ctx.lib
    e0, e1 = C.c_void_p(), C.c_void_p()
    assert lib.ferrum_hip_event_create(C.byref(e0)) == 0 and lib.ferrum_hip_event_create(C.byref(e1)) == 0
    assert lib.ferrum_hip_event_record(e0, ctx.stream) == 0
    B.layer_norm(ctx, dev16(torch, x), dev16(torch, g), dev16(torch, b), 1e-5, out, tokens, dim)
    assert lib.ferrum_hip_event_record(e1, ctx.stream) == 0
    ms = C.c_float(-1.0)
    assert lib.ferrum_hip_event_elapsed_ms(e0, e1, C.byref(ms)) == 0 and 0.0 <= ms.value < 1000.0
    lib.ferrum_hip_event_destroy(e0); lib.ferrum_hip_event_destroy(e1)
    assert nmse(O.layer_norm(x, g, b, 1e-5), host(out)) < NMSE_FP16_TOL
    B.gelu(ctx, dev16(torch, x), out, tokens * dim)
    assert nmse(O.gelu(x), host(out)) < NMSE_FP16_TOL


@pytest.mark.parametrize("tokens,dim", [(1, 1024), (5, 2048), (32, 4096), (3, 5376), (2, 8192), (7, 128), (256, 2056), (257, 2056), (300, 8192), (260, 16384), (513, 136)])
def test_rms_norm_and_fused_add(env, tokens, dim):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(dim + tokens)
    x = f16r(rng.standard_normal((tokens, dim)) * 2)
    r = f16r(rng.standard_normal((tokens, dim)) * 3)
    w = f16r(1 + 0.2 * rng.standard_normal(dim))
    out = torch.empty(tokens, dim, dtype=torch.float16, device="cuda")
    B.rms_norm(ctx, dev16(torch, x), dev16(torch, w), 1e-6, out, tokens, dim)
    assert nmse(O.rms_norm(x, w, 1e-6), host(out)) < NMSE_FP16_TOL
    rd = dev16(torch, r)
    B.fused_add_rms_norm(ctx, rd, dev16(torch, x), dev16(torch, w), 1e-6, out, tokens, dim)
    r_ref, o_ref = O.fused_add_rms_norm(r, x, w, 1e-6)
    assert nmse(r_ref, host(rd)) < NMSE_FP16_TOL          # residual stored as fp16
    # the fp16 lane norms the ROUNDED residual (fused_add_rms_norm.cu:88-101): compare both ways
    assert nmse(o_ref, host(out)) < 3e-6
    assert nmse(O.rms_norm(host(rd), w, 1e-6), host(out)) < NMSE_FP16_TOL


def test_rms_norm_empty_is_noop(env):
    pkg, B, ctx, O, torch = env
    out = torch.empty(0, 128, dtype=torch.float16, device="cuda")
    B.rms_norm(ctx, out, dev16(torch, np.ones(128)), 1e-6, out, 0, 128)


def test_embedding_silu_gelu_add_scale(env):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(1)
    table = f16r(rng.standard_normal((300, 256)))
    ids = np.array([0, 299, 17, 17, 4], np.uint32)
    out = torch.empty(5, 256, dtype=torch.float16, device="cuda")
    B.embedding_lookup(ctx, dev16(torch, table), torch.from_numpy(ids.astype(np.int32)).cuda(), out, 256)
    assert np.array_equal(host(out), O.embedding_lookup(table, ids))        # a copy: exact
    gu = f16r(rng.standard_normal((6, 2 * 768)) * 3)
    act = torch.empty(6, 768, dtype=torch.float16, device="cuda")
    B.fused_silu_mul_split(ctx, dev16(torch, gu), act, 6, 768)
    assert nmse(O.fused_silu_mul_split(gu, 768), host(act)) < NMSE_FP16_TOL
    B.fused_gelu_tanh_mul_split(ctx, dev16(torch, gu), act, 6, 768)
    assert nmse(O.fused_gelu_tanh_mul_split(gu, 768), host(act)) < NMSE_FP16_TOL
    a, b = f16r(rng.standard_normal(1000)), f16r(rng.standard_normal(1000))
    ad = dev16(torch, a)
    B.add_inplace(ctx, ad, dev16(torch, b), 1000)
    assert np.array_equal(host(ad), f16r(O.add_inplace(a, b)))              # one rounding, exact after fp16
    sd = dev16(torch, np.array([1.0, -2.0, 0.5]))
    B.scale_inplace(ctx, sd, 33.9375, 3)                                    # llama_family.rs:6076-6086 KAT
    assert list(host(sd)) == [33.9375, -67.875, 16.96875]


# ── GPTQ INT4 linear ─────────────────────────────────────────────────────────
def _gptq_case(env, k, n, m, seed, symmetric, g_idx=False, x_fn=None):
    pkg, B, ctx, O, torch = env
    qw, sc, qz = O.make_synthetic_gptq(k, n, 128, seed, symmetric=symmetric)
    sc = f16r(sc)                                          # scales travel as fp16 on the device
    gi = O.make_desc_act_g_idx(k, 128) if g_idx else None
    lin = pkg.GptqLinear.from_raw(qw, sc, qz, gi, None, 4, 128, k, n)
    if x_fn is None:
        x = f16r(np.random.default_rng(seed).standard_normal((m, k)))
    else:
        x = f16r(x_fn(np.arange(m * k, dtype=np.float32)).reshape(m, k))
    out = torch.empty(m, n, dtype=torch.float16, device="cuda")
    lin.forward(ctx, dev16(torch, x), out, m)
    w = O.dequant_gptq(qw, sc, qz, 128, k, n, g_idx=gi)
    ref = O.gemm(x, w, m, n, k)
    return ref, host(out)


def test_gptq_reference_shapes(env):
    # gptq_parity_test.rs:108-145 (K=256,N=128,m=2, sin(0.001 i)) and :329-405 (K=512,N=256,m=2, symmetric,
    # cos(0.003 i) rounded to f16, rel err < 5 %): we hold the fp16 NMSE bucket instead
    ref, got = _gptq_case(env, 256, 128, 2, 0xDEADBEEF, False, x_fn=lambda i: np.sin(i * np.float32(0.001)))
    assert nmse(ref, got) < NMSE_FP16_TOL
    ref, got = _gptq_case(env, 512, 256, 2, 0xC0FFEE, True, x_fn=lambda i: np.cos(i * np.float32(0.003)))
    assert nmse(ref, got) < NMSE_FP16_TOL
    assert np.max(np.abs(ref - got)) / np.max(np.abs(ref)) < 2e-3


@pytest.mark.parametrize("k,n,m", [(2048, 5120, 1), (2048, 5120, 32), (4096, 2048, 4), (4096, 2048, 16),
                                   (1024, 1536, 33), (768, 2048, 64), (512, 264, 100), (256, 72, 7)])
def test_gptq_model_shapes(env, k, n, m):
    ref, got = _gptq_case(env, k, n, m, 0x1234 + k + n + m, True)
    assert nmse(ref, got) < NMSE_FP16_TOL


@pytest.mark.parametrize("k,n,m", [(512, 256, 3), (2048, 640, 17)])
def test_gptq_asymmetric_and_act_order(env, k, n, m):
    ref, got = _gptq_case(env, k, n, m, 0x51A7E5, False)                 # explicit zero points
    assert nmse(ref, got) < NMSE_FP16_TOL
    ref, got = _gptq_case(env, k, n, m, 0x5A170A7, False, g_idx=True)    # desc_act (gptq_parity_test.rs:271)
    assert nmse(ref, got) < NMSE_FP16_TOL


@pytest.mark.parametrize("k,n,m,form", [(8192, 2048, 32, "w4_ldsa"), (2048, 640, 200, "w4_tilep"), (1024, 4096, 2100, "w4_big"),
                                        (4096, 6144, 40, "w4_tilep")])
def test_gptq_act_order_takes_every_dense_kernel_form(env, k, n, m, form, forms):
    """desc_act weights (Gemma-3 GPTQ): the packed rows are in sorted-g_idx order and the activations' columns
    are gathered with the same permutation before the GEMM, so the 17–32-row, 64-row-tile and tall-tile kernels serve them like
    any other weights (round 1 sent every act-order projection of ≥ 17 rows through the per-wave-activation skinny kernel)."""
    forms.reset()
    ref, got = _gptq_case(env, k, n, m, 0xAC70 + m, False, g_idx=True)
    forms.require(form)
    assert nmse(ref, got) < NMSE_FP16_TOL


@pytest.mark.parametrize("k,n,ms,sym", [
    # row-count boundaries of the three dense kernels (≤16 wgsplit, 17–32 LDS-A / wgsplit, ≥64 pipelined tile + split-K, 33–63 wgsplit)
    # on shapes that select each path: deep-K narrow-N (LDS-A with slabs), wide-N, tiny, N not a multiple of 64, asymmetric
    (8192, 2048, (16, 17, 32, 33), True), (1024, 16384, (17, 32, 64, 65), True), (256, 64, (1, 16, 31, 63, 64, 127, 128, 200), True),
    (1536, 1000, (5, 20, 64, 130), True), (2048, 640, (24, 64, 96), False), (14336, 512, (32, 64), True),
    # many row tiles through the pipelined tile kernel — ragged last tile, odd group count (K = 640: 5 groups), split-K
    # (narrow N), columns not a multiple of 256, asymmetric + bias
    (640, 320, (1024, 1100), True), (2048, 512, (1024,), True), (1024, 1000, (1153,), True), (768, 640, (1025,), False),
    # 33–63 rows of the larger projections (K·N ≥ 12 Mi) take the pipelined tile kernel with one ragged 64-row tile
    (4096, 4096, (33, 48, 63), True), (2048, 6144, (40,), False),
    # enough 128- / 256-row tiles to fill the chip: w4_gemm_big_kernel (ragged last tile; asymmetric)
    (2048, 5120, (1664, 3100), True), (1024, 4096, (2100,), False)])
def test_gptq_row_regimes_and_edge_shapes(env, k, n, ms, sym, forms):
    pkg, B, ctx, O, torch = env
    seen = set()
    qw, sc, qz = O.make_synthetic_gptq(k, n, 128, k * 7 + n, symmetric=sym)
    sc = f16r(sc / (0.28 * np.sqrt(k)))
    bias = f16r(np.random.default_rng(n).standard_normal(n)) if n == 640 else None
    lin = pkg.GptqLinear.from_raw(qw, sc, qz, None, bias, 4, 128, k, n)
    w = O.dequant_gptq(qw, sc, qz, 128, k, n)
    for m in ms:
        x = f16r(np.random.default_rng(m).standard_normal((m, k)))
        out = torch.full((m + 1, n), 7.0, dtype=torch.float16, device="cuda")     # guard row: nothing may write past m rows
        forms.reset()
        lin.forward(ctx, dev16(torch, x), out, m)
        ctx.sync()
        # the kernel the row count selects (w4_gemm_dense): ≤ 16 rows K-split skinny; ≥ 64 rows (33 on the larger projections)
        # the pipelined tile kernel; in between the LDS-shared-activation kernel on shapes deep or wide enough for it
        h = forms.hits()
        ran = [f for f in ("w4_wgsplit", "w4_ldsa", "w4_tilep", "w4_big") if h.get(f)]
        assert len(ran) == 1, (k, n, m, h)
        big = k * n >= (12 << 20)
        want = "w4_wgsplit" if m <= 16 else ("w4_tilep" if m >= (33 if big else 64) else None)
        if m >= 1024 and n >= 4096: want = "w4_big"
        assert want is None or ran[0] == want, (k, n, m, h)
        seen.add(ran[0])
        ref = O.gemm(x, w, m, n, k) + (bias[None, :] if bias is not None else 0.0)
        got = host(out)
        assert nmse(ref, got[:m]) < NMSE_FP16_TOL, (k, n, m)
        assert np.all(got[m] == 7.0), (k, n, m)
    if (k, n) in ((8192, 2048), (1024, 16384)):
        assert "w4_ldsa" in seen, seen                     # the 17–32-row cases of these shapes are the LDS-A kernel's


@pytest.mark.parametrize("mt", [6, 8, 16])
@pytest.mark.parametrize("sym", [True, False])
def test_gptq_big_tile_forms(env, mt, sym, knobs, forms):
    """w4_gemm_big_kernel forced on a small projection: 128- and 256-row tiles, ragged last tile, N = 1000 (a partial 256-column
    workgroup and a partial 64-column supertile), bias, symmetric and asymmetric zero points.  Its fp16 weights are
    (q − zero)·scale rounded once — the reference's own dequantisation (`cpu.rs:2283-2315` produces exactly that value in
    f32; Marlin in fp16) — so the oracle comparison holds at the fp16 tolerance."""
    pkg, B, ctx, O, torch = env
    k, n = 1024, 1000
    qw, sc, qz = O.make_synthetic_gptq(k, n, 128, 99 + mt, symmetric=sym)
    sc = f16r(sc / (0.28 * np.sqrt(k)))
    bias = f16r(np.random.default_rng(5).standard_normal(n))
    lin = pkg.GptqLinear.from_raw(qw, sc, qz, None, bias, 4, 128, k, n)
    w = O.dequant_gptq(qw, sc, qz, 128, k, n)
    knobs.set(W4_BIG=mt)
    for m in (16 * mt, 16 * mt + 37, 3 * 16 * mt - 1):
        x = f16r(np.random.default_rng(m).standard_normal((m, k)))
        out = torch.full((m + 1, n), 7.0, dtype=torch.float16, device="cuda")
        forms.reset()
        lin.forward(ctx, dev16(torch, x), out, m)
        ctx.sync()
        forms.require("w4_big", absent=("w4_tilep", "w4_ldsa", "w4_wgsplit"))
        ref = O.gemm(x, w, m, n, k) + bias[None, :]
        got = host(out)
        assert nmse(ref, got[:m]) < NMSE_FP16_TOL, (mt, sym, m)
        assert np.all(got[m] == 7.0), (mt, sym, m)


def test_gptq_linearity(env):
    # size-independent property at a BASELINE shape (Llama-8B o_proj 4096→4096): f(a·x+y) = a·f(x)+f(y)
    pkg, B, ctx, O, torch = env
    k, n, m = 4096, 4096, 8
    qw, sc, qz = O.make_synthetic_gptq(k, n, 128, 99, symmetric=True)
    lin = pkg.GptqLinear.from_raw(qw, f16r(sc), qz, None, None, 4, 128, k, n)
    rng = np.random.default_rng(5)
    x, y = f16r(rng.standard_normal((m, k))), f16r(rng.standard_normal((m, k)))
    z = f16r(2.0 * x + y)                                 # exactly representable inputs are not needed:
    outs = []
    for v in (x, y, z):
        o = torch.empty(m, n, dtype=torch.float16, device="cuda")
        lin.forward(ctx, dev16(torch, v), o, m)
        outs.append(host(o).astype(np.float64))
    lhs = outs[2]
    rhs = None
    # z was rounded to fp16, so compare against f applied to the exact combination in fp64
    w = O.dequant_gptq(qw, f16r(sc), qz, 128, k, n).astype(np.float64)
    rhs = z.astype(np.float64) @ w.T
    assert nmse(rhs, lhs) < NMSE_FP16_TOL
    assert nmse(x.astype(np.float64) @ w.T, outs[0]) < NMSE_FP16_TOL


# ── dense fp16 GEMM (router / lm_head) ───────────────────────────────────────
@pytest.mark.parametrize("m,n,k,f32out", [(1, 128, 2048, True), (32, 128, 2048, True), (5, 1511, 1024, True),
                                          (33, 96, 256, False), (64, 2048, 512, False),
                                          (20, 32768 + 128, 256, True), (32, 32768 + 64, 128, False)])   # the wide-N form of 17–32 rows (lm_head): 64 columns per wave
def test_dense_gemm(env, m, n, k, f32out):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(m * n + k)
    a, b = f16r(rng.standard_normal((m, k))), f16r(rng.standard_normal((n, k)) * 0.1)
    out = torch.empty(m, n, dtype=torch.float32 if f32out else torch.float16, device="cuda")
    B.gemm(ctx, dev16(torch, a), dev16(torch, b), out, m, n, k)
    ref = O.gemm(a, b, m, n, k)
    assert nmse(ref, host(out)) < (1e-10 if f32out else NMSE_FP16_TOL)
    # same product through the load-time fragment-major layout (lm_head / router path)
    bt = B.dense_repack_f16t(ctx, dev16(torch, b), n, k)
    out2 = torch.zeros_like(out)
    B.gemm_f16t(ctx, dev16(torch, a), bt, out2, m, n, k)
    ctx.sync()
    assert nmse(ref, host(out2)) < (1e-10 if f32out else NMSE_FP16_TOL)


@pytest.mark.parametrize("shift", [0, 1, 4])
@pytest.mark.parametrize("n", [328, 640])
@pytest.mark.parametrize("mt", [6, 8, 16])
def test_prefill_tiles_at_any_address(env, mt, n, shift, knobs, forms):
    """Rows and results that begin at a 16-byte piece and not, columns that end within a wave's 64, a last tile of few rows: the same numbers, and nothing beside them."""
    pkg, B, ctx, O, torch = env
    k, m = 256, 16 * mt + 5
    qw, sc, qz = O.make_synthetic_gptq(k, n, 128, 3, symmetric=False)
    sc = f16r(sc / (0.28 * np.sqrt(k)))
    lin = pkg.GptqLinear.from_raw(qw, sc, qz, None, None, 4, 128, k, n)
    knobs.set(W4_BIG=mt)
    x = f16r(np.random.default_rng(m).standard_normal((m, k)))
    src, buf = (torch.full((rows * cols + 16,), 7.0, dtype=torch.float16, device="cuda") for rows, cols in ((m, k), (m, n)))
    src[shift:shift + m * k] = dev16(torch, x).reshape(-1)
    forms.reset()
    lin.forward(ctx, src[shift:shift + m * k], buf[shift:shift + m * n], m)
    ctx.sync()
    forms.require("w4_big")
    got = host(buf)
    assert nmse(O.gemm(x, O.dequant_gptq(qw, sc, qz, 128, k, n), m, n, k), got[shift:shift + m * n].reshape(m, n)) < NMSE_FP16_TOL
    assert np.all(got[:shift] == 7.0) and np.all(got[shift + m * n:] == 7.0)


@pytest.mark.parametrize("blocks,n", [(1, 200), (4, 64), (5, 1480), (6, 520), (9, 264), (13, 712)])
def test_w4_big_tiles_in_bands(env, blocks, n, knobs, forms):
    """Bands of row blocks that divide their number and not, one column tile and several, fewer tiles than XCDs and no multiple of them: each
    tile is taken once."""
    pkg, B, ctx, O, torch = env
    k, m = 256, max(128, 128 * blocks - 3)
    qw, sc, qz = O.make_synthetic_gptq(k, n, 128, 3, symmetric=True)
    sc = f16r(sc / (0.28 * np.sqrt(k)))
    lin = pkg.GptqLinear.from_raw(qw, sc, qz, None, None, 4, 128, k, n)
    knobs.set(W4_BIG=8)
    x = f16r(np.random.default_rng(m).standard_normal((m, k)))
    out = torch.full((m + 1, n), 7.0, dtype=torch.float16, device="cuda")
    forms.reset()
    lin.forward(ctx, dev16(torch, x), out, m)
    ctx.sync()
    forms.require("w4_big")
    ref, got = O.gemm(x, O.dequant_gptq(qw, sc, qz, 128, k, n), m, n, k), host(out)
    for r in range(0, m, 128):
        assert nmse(ref[r:r + 128], got[r:min(r + 128, m)]) < NMSE_FP16_TOL, r
    assert np.all(got[m] == 7.0)


@pytest.mark.parametrize("f32out", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 64, 32), (16, 4096, 1024), (17, 96, 1056), (64, 1024, 3072), (65, 8192, 32), (100, 6176, 96), (200, 2080, 64),
                                   (129, 16416, 160), (300, 4128, 2080), (1100, 1056, 352), (2049, 4096, 128), (3000, 8224, 64), (9, 14400, 2080), (16, 16416, 4128),
                                   (5, 20512, 96), (48, 5152, 256), (33, 8256, 544), (64, 8256, 2080), (64, 10272, 4128)])
def test_dense_gemm_tile_edges(env, m, n, k, f32out):
    """Few rows and every tile size at rows and columns just past a tile, odd and even numbers of 32-column steps, fewer of them than a ring holds;
    also into a result whose address only takes single elements."""
    pkg, B, ctx, O, torch = env
    gen = torch.Generator("cuda").manual_seed(m + n + k)
    a, b = (torch.randn(r, k, generator=gen, device="cuda").half() for r in (m, n))
    bt, want = B.dense_repack_f16t(ctx, b, n, k), a.double() @ b.double().T
    # fp32 sums of exact products in any order, then one rounding to the output's type
    bound = k * 2.0 ** -24 * (a.double().abs() @ b.double().abs().T) + (2.0 ** -24 if f32out else 2.0 ** -11) * want.abs() + 2.0 ** -24
    for shift in (0, 1):
        buf = torch.full((m * n + 64,), 7.0, dtype=torch.float32 if f32out else torch.float16, device="cuda")
        B.gemm_f16t(ctx, a, bt, buf[shift:shift + m * n], m, n, k)
        ctx.sync()
        assert bool(((buf[shift:shift + m * n].view(m, n).double() - want).abs() <= bound).all())
        assert bool((buf[:shift] == 7.0).all()) and bool((buf[shift + m * n:] == 7.0).all())


def test_allocated_memory_is_zero_on_return(env):
    """What another stream writes into new memory stays: no fill is on its way any more (a gigabyte of it takes 0.2 ms, this write a tenth of that)."""
    import ctypes as C
    lib = env[0].load_library()
    stream, p, size = C.c_void_p(), C.c_void_p(), 4 << 30
    want, got = (C.c_uint8 * 64)(*[7] * 64), (C.c_uint8 * 64)()
    assert lib.ferrum_hip_stream_create(C.byref(stream)) == 0
    for _ in range(3):
        assert lib.ferrum_hip_alloc(C.byref(p), C.c_size_t(size)) == 0
        end = C.c_void_p(p.value + size - 128)
        assert lib.ferrum_hip_memcpy_h2d(end, want, C.c_size_t(64), stream) == 0
        assert lib.ferrum_hip_stream_synchronize(None) == 0
        assert lib.ferrum_hip_memcpy_d2h(got, end, C.c_size_t(64), stream) == 0 and bytes(got) == bytes(want)
        assert lib.ferrum_hip_memcpy_d2h(got, C.c_void_p(end.value + 64), C.c_size_t(64), stream) == 0 and not any(got)
        assert lib.ferrum_hip_free(p) == 0
    assert lib.ferrum_hip_stream_destroy(stream) == 0


def test_zeros_of_any_length(env):
    """A range of more 16-byte pieces than a launch has threads, from an odd address to an odd end, its last bytes and those around it."""
    import ctypes as C
    lib, p, size, sevens, got = env[0].load_library(), C.c_void_p(), (1 << 36) + (1 << 20), (C.c_uint8 * 64)(*[7] * 64), (C.c_uint8 * 64)()
    assert lib.ferrum_hip_alloc(C.byref(p), C.c_size_t(size)) == 0
    places = [0, 1 << 34, (1 << 34) + (1 << 20), (1 << 36) - 32, size - 64]
    for at in places:
        assert lib.ferrum_hip_memcpy_h2d(C.c_void_p(p.value + at), sevens, C.c_size_t(64), None) == 0
    assert lib.ferrum_hip_memset_zero(C.c_void_p(p.value + 5), C.c_size_t(size - 5 - 9), None) == 0
    for at in places:
        assert lib.ferrum_hip_memcpy_d2h(got, C.c_void_p(p.value + at), C.c_size_t(64), None) == 0
        assert bytes(got) == bytes(7 if at + i < 5 or at + i >= size - 9 else 0 for i in range(64)), at
    assert lib.ferrum_hip_free(p) == 0


def test_zeros_on_every_replay(env):
    """Ranges that start and end anywhere, alone and on each of several replays of a captured graph with eager work and synchronizations in between."""
    import ctypes as C
    pkg, B, ctx, O, torch = env
    size = 1 << 20
    buf, ranges = torch.zeros(size, dtype=torch.uint8, device="cuda"), [(0, 0), (5, 1), (31, 2), (49, 15), (65, 16), (100, 29), (160, 4096), (5001, 4103), (20003, 900001)]
    want = torch.full((size,), 7, dtype=torch.uint8, device="cuda")
    for at, n in ranges:
        want[at:at + n] = 0
    with torch.cuda.stream(torch.cuda.Stream()):
        c2 = B.new_context()                                       # capture needs a non-default stream

        def zero():
            for at, n in ranges:
                assert c2.lib.ferrum_hip_memset_zero(C.c_void_p(buf.data_ptr() + at), C.c_size_t(n), c2.stream) == 0
        B.begin_graph_capture(c2)
        zero()
        graph = B.end_graph_capture(c2)
        for replay in [False] + [True] * 6:
            buf.fill_(7)
            torch.cuda.synchronize()
            B.replay_graph(c2, graph) if replay else zero()
            c2.sync()
            assert torch.equal(buf, want)
        B.reset_graph(c2, graph)


def _times(env, knobs, call, ways):
    """Best time of a call under every setting of the switches, ms: captured, so that the host does not count, and in turn, so that a slow moment meets all."""
    pkg, B, ctx, O, torch = env
    names, graphs, best = {name for w in ways.values() for name in w}, {}, {}
    with torch.cuda.stream(torch.cuda.Stream()):
        c2 = B.new_context()
        for way, set_to in ways.items():
            knobs.set(**{**dict.fromkeys(names), **set_to})
            call(c2)                                                       # (a kernel's first use sets its LDS size)
            c2.sync()
            B.begin_graph_capture(c2)
            for _ in range(20):
                call(c2)
            graphs[way], best[way] = B.end_graph_capture(c2), float("inf")
        for _ in range(8):
            for way, graph in graphs.items():
                start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                start.record()
                B.replay_graph(c2, graph)
                end.record()
                end.synchronize()
                best[way] = min(best[way], start.elapsed_time(end) / 20)
        for graph in graphs.values():
            B.reset_graph(c2, graph)
    return best


@pytest.mark.parametrize("m,n,k", [(125, 9216, 4096), (456, 8192, 6144), (64, 5120, 256), (64, 8256, 6144), (65, 1024, 4096)])
def test_projections_take_the_faster_side_of_a_line(env, m, n, k, knobs):
    """Shapes at the lines between tile sizes, rows of a workgroup and parts of K where the wrong side costs 12 to 60 %: what is chosen is as fast as any choice, to a
    tenth."""
    from tests.tile_sizes import SIZES
    pkg, B, ctx, O, torch = env
    gen = torch.Generator("cuda").manual_seed(1)
    a, b = (torch.randn(r, k, generator=gen, device="cuda").half() for r in (m, n))
    out, bt = torch.empty(m, n, dtype=torch.float16, device="cuda"), B.dense_repack_f16t(ctx, b, n, k)
    ways = SIZES if m > 65 else {f"{16 * j} columns, K in {w}, rows {t}": dict(TILED_J=j, TILED_KW=w, TILED_MIN_TILES=t) for j in (1, 2) for w in (1, 2, 4) for t in (64, 128)}
    best = _times(env, knobs, lambda c: B.gemm_f16t(c, a, bt, out, m, n, k), {"chosen": {}, **ways})
    assert best["chosen"] < 1.1 * min(best.values()), best


@pytest.mark.parametrize("kw", [0, 1, 2, 4, 8])
@pytest.mark.parametrize("j", [1, 2])
@pytest.mark.parametrize("m,n,k", [(1, 32, 32), (3, 64, 64), (4, 96, 96), (5, 160, 128), (13, 288, 160), (16, 32, 1120), (17, 96, 288), (32, 160, 1024), (33, 64, 544), (49, 96, 4128),
                                   (64, 32, 256), (79, 96, 96)])
def test_few_rows_of_every_count(env, m, n, k, j, kw, knobs, forms):
    """Rows that fill no load and no tile, parts of K of no, one and several chunks that end within one, column groups past the last tile.  Against 64 bits: an fp32 sum
    of K exact products errs by K x 2^-24 of the sum of their magnitudes at most, and fp16 rounds by 2^-11."""
    knobs.set(TILED_J=j, TILED_NW=8 if kw == 8 else 4, TILED_KW=kw, TILED_BIG_MIN_TILES=10 ** 6)
    _few_rows(env, m, n, k)
    forms.require("tiled_gemm")


@pytest.mark.parametrize("kw", [1, 2, 4, 8])
@pytest.mark.parametrize("j", [1, 2, 4])
@pytest.mark.parametrize("m,n,k", [(17, 64, 32), (18, 320, 96), (23, 192, 768), (28, 64, 1120), (29, 576, 1024), (32, 128, 4128), (33, 64, 544), (50, 320, 768), (64, 192, 1056)])
def test_few_rows_of_several_row_tiles(env, m, n, k, j, kw, knobs, forms):
    """The same with two and four row tiles a workgroup, which sizes as small as these would not take, and up to 64 columns a wave; parts of several chunks that are taken in a
    circle and that are not."""
    knobs.set(TILED_J=j, TILED_NW=8 if kw == 8 else 4, TILED_KW=kw, TILED_BIG_MIN_TILES=10 ** 6, TILED_MIN_TILES=-1)
    _few_rows(env, m, n, k)
    forms.require("tiled_gemm", *(["tiled_gemm_cols64"] if j == 4 and m <= 32 else []))


@pytest.mark.parametrize("j", [3, 5, 6])
def test_forced_columns_that_no_form_has(env, j, knobs, forms):
    """A forced number of 16-column tiles for which there is no kernel is 2, as it is with one and four row tiles: every column is written."""
    knobs.set(TILED_J=j, TILED_BIG_MIN_TILES=10 ** 6, TILED_MIN_TILES=-1)
    for m in (10, 20, 50):
        _few_rows(env, m, 320, 96)
    assert bool(forms.hits().get("tiled_gemm_cols48")) == (j == 3)


@pytest.mark.parametrize("m,n,k,form", [(17, 8224, 96, None), (17, 8224, 544, 48), (32, 8256, 2080, 48), (20, 12288, 64, None), (32, 9280, 512, None), (20, 12288, 576, 48), (32, 8192, 2048, None), (32, 12320, 2048, 64), (17, 14336, 4096, 64), (32, 12320, 1024, None),
                                        (32, 14368, 2048, None), (16, 9280, 2048, None)])
def test_columns_past_a_round_of_workgroups(env, m, n, k, form, knobs, forms):
    """48 and 64 columns a wave on both sides of the lines where they begin and end; the last wave's columns there in whole and in parts."""
    _few_rows(env, m, n, k)
    h = forms.hits()
    assert [c for c in (48, 64) if h.get(f"tiled_gemm_cols{c}")] == ([form] if form else []), h


@pytest.mark.parametrize("m,n,k,form", [(30, 65600, 1568, "tiled_gemm_cols64"), (17, 65600, 3104, "tiled_gemm_cols64"), (20, 139328, 1056, None), (32, 139264, 1056, None), (12, 120960, 4128, None),
                                        (12, 120832, 4128, "tiled_gemm"), (32, 139008, 1056, "tiled_gemm"), (10, 65568, 2080, "tiled_gemm"), (15, 32800, 96, "tiled_gemm")])
def test_vocabularies_on_both_sides_of_a_line(env, m, n, k, form, knobs, forms):
    """What is chosen for a wide output: 64 columns a wave, or the kernel that holds no rows in LDS where that is the faster one."""
    _few_rows(env, m, n, k)
    assert form in forms.hits() if form else "tiled_gemm" not in forms.hits(), forms.hits()


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("m,n,k", [(65, 64, 128), (255, 288, 256), (257, 320, 384), (511, 1056, 128), (300, 8256, 512), (2310, 8224, 128), (5000, 4160, 256), (700, 512, 4096)])
def test_tiles_of_256_x_256(env, m, n, k, f32, knobs, forms):
    """Rows and columns on both sides of a tile's end, one round of four steps and several, less than one tile for each workgroup and up to four one after the other."""
    knobs.set(TILED_256=1, TILED_BIG_MIN_TILES=1)
    _few_rows(env, m, n, k, f32)
    forms.require("tiled_gemm_256x256")


@pytest.mark.parametrize("m,n,k,forced,taken", [
    (2001, 8192, 2048, None, True), (2001, 8224, 2048, None, False), (2001, 8192, 2048, 257, False), (2001, 8192, 2048, 256, False), (2001, 8192, 2048, -1, True),
    (2001, 8192, 1024, None, True), (2048, 16384, 1024, None, False), (3072, 16384, 1024, None, False), (4096, 16384, 1024, None, True)])
def test_rule_of_tiles_of_256_x_256(env, m, n, k, forced, taken, knobs, forms):
    """One round of them where two of 128 x 256 fill the card, not two where three do; with K of 1024 one or four, not two or three; a number of the smaller tiles asked for, their own
    line's among them, is what runs."""
    knobs.set(TILED_WIDE_MIN_TILES=forced)
    _few_rows(env, m, n, k)
    hits = forms.hits()
    assert bool(hits.get("tiled_gemm_256x256")) == taken and bool(hits.get("tiled_gemm_128x256")) != taken, hits


@pytest.mark.parametrize("tiles,form", [(0, "tiled_gemm_big"), (2, "tiled_gemm_big"), (3, "tiled_gemm"), (None, "tiled_gemm")])
def test_tile_kernel_from_a_given_number_of_tiles(env, tiles, form, knobs, forms):
    """Two tiles of 64 x 64: a number asked for, 0 among them, or the rule."""
    knobs.set(TILED_BIG_MIN_TILES=tiles)
    _few_rows(env, 65, 64, 64)
    assert set(forms.hits()) & {"tiled_gemm", "tiled_gemm_big"} == {form}


def _few_rows(env, m, n, k, f32=False):
    pkg, B, ctx, O, torch = env
    gen = torch.Generator("cuda").manual_seed(m * n + k)
    a, b = (torch.randn(r, k, generator=gen, device="cuda").half() for r in (m, n))
    buf = torch.full(((m + 2) * n,), 7.0, dtype=torch.float32 if f32 else torch.float16, device="cuda")
    out = buf[n:n + m * n]
    B.gemm_f16t(ctx, a, B.dense_repack_f16t(ctx, b, n, k), out, m, n, k)
    ctx.sync()
    want, size = a.double() @ b.double().T, a.double().abs() @ b.double().abs().T
    assert ((out.reshape(m, n).double() - want).abs() <= (0 if f32 else 2.0 ** -11 * want.abs() + 2.0 ** -25) + k * 2.0 ** -24 * size).all()
    assert (buf[:n] == 7.0).all() and (buf[n + m * n:] == 7.0).all()


@pytest.mark.parametrize("n,k", [(4096, 8192), (8192, 8192), (8192, 4096)])
def test_few_rows_of_a_power_of_two(env, n, k, knobs):
    """A K whose rows of weights all begin at the same place among the memory's channels takes about as long as one that is a little longer; weights from memory, not from
    the caches."""
    pkg, B, ctx, O, torch = env
    took = []
    for kk in (k, k + 160):
        a, out = torch.randn(8, kk, device="cuda").half(), torch.empty(8, n, dtype=torch.float16, device="cuda")
        copies = torch.randn((700 << 20) // (2 * n * kk), n, kk, dtype=torch.float16, device="cuda")          # (tiles of some weights)

        def call(c):
            for w in copies:
                B.gemm_f16t(c, a, w, out, 8, n, kk)
        took.append(_times(env, knobs, call, {"chosen": {}})["chosen"] / len(copies))
        del copies
    assert took[0] < 1.15 * took[1], took


@pytest.mark.parametrize("nq,nkv,tokens,pos,seqs,window", [(32, 4, 64, 700, 24, 0), (14, 2, 4096, 0, 1, 512), (32, 8, 700, 0, 1, 0)])
def test_prompt_attention_takes_the_faster_unit(env, nq, nkv, tokens, pos, seqs, window, knobs):
    """Batches on both sides of the line between units of 64 and 128 rows, where the wrong one costs 12 to 40 %."""
    pkg, B, ctx, O, torch = env
    gen = torch.Generator("cuda").manual_seed(1)
    T, kv, mb = tokens * seqs, pos + tokens, (pos + tokens + 15) // 16
    q, k, v = (torch.randn(n, generator=gen, device="cuda").half() for n in (T * nq * 128, seqs * mb * nkv * 2048, seqs * mb * nkv * 2048))
    out, tables = torch.empty_like(q), torch.arange(seqs * mb, device="cuda", dtype=torch.int32).reshape(seqs, mb)
    cu, po = torch.arange(seqs + 1, device="cuda", dtype=torch.int32) * tokens, torch.full((seqs,), pos, device="cuda", dtype=torch.int32)
    best = _times(env, knobs, lambda c: B.paged_varlen_attention(c, q, k, v, out, cu, po, tables, seqs, T, kv, nq, nkv, 128, window, 16, mb, tokens),
                  {"chosen": {}, "64": dict(ATTN_FLASH_ROWS=64), "128": dict(ATTN_FLASH_ROWS=128)})
    assert best["chosen"] < 1.1 * min(best.values()), best


@pytest.mark.parametrize("hd,tokens", [(256, 1), (256, 40), (128, 8), (128, 2048)])
def test_cache_write_takes_the_faster_form(env, hd, tokens, knobs):
    """A token of four heads a wave, or four tokens of a head."""
    pkg, B, ctx, O, torch = env
    nq, nkv, mb = 32, 8, (tokens + 15) // 16
    qkv, one = torch.randn(tokens, (nq + 2 * nkv) * hd, device="cuda").half(), torch.ones(hd, device="cuda").half()
    cos, q_out, (ck, cv) = torch.ones(tokens, hd // 2, device="cuda"), torch.empty(tokens, nq * hd, device="cuda").half(), (B.alloc_paged_pool(mb, nkv, hd) for _ in range(2))
    tables, cu, po = torch.arange(mb, device="cuda", dtype=torch.int32)[None], torch.tensor([0, tokens], device="cuda", dtype=torch.int32), torch.zeros(1, device="cuda", dtype=torch.int32)
    best = _times(env, knobs, lambda c: B.split_qkv_norm_rope_into_paged_cache_varlen(c, qkv, one, one, cos, cos, q_out, ck, cv, cu, po, tables, 1, tokens, nq, nkv, hd, 1e-6, 1, 16, mb),
                  {"chosen": {}, "quads": dict(ROPE_QUAD_ROWS=0), "heads": dict(ROPE_QUAD_ROWS=10 ** 9)})
    assert best["chosen"] < 1.1 * min(best.values()), best


# ── paged KV write / read ────────────────────────────────────────────────────
def _rope(O, hd, max_seq, theta=1e6):
    return O.build_rope_cache(theta, hd, max_seq)


@pytest.mark.parametrize("quad_rows", [0, 10 ** 9])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("q_lens,pos,nq,nkv", [([1], [0], 1, 1), ([4], [12], 3, 1), ([3, 5], [1, 4], 2, 2), ([16, 0, 8, 0], [0, 3, 4, 0], 5, 3), ([7, 9, 64, 33], [1, 0, 0, 7], 8, 2),
                                               ([4] * 70, [4 * (i % 5) for i in range(70)], 2, 1), ([5] * 66 + [0] * 3, [i % 7 for i in range(69)], 3, 2)])
def test_quads_of_tokens_in_the_paged_cache(env, q_lens, pos, nq, nkv, hd, quad_rows, knobs):
    """Four tokens of a wave at aligned positions and not, across sequences and past the batch, empty sequences in between and at the end, and four heads of a token
    a wave: copies."""
    knobs.set(ROPE_QUAD_ROWS=quad_rows)
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(len(q_lens) + hd)
    S, T, mb = len(q_lens), sum(q_lens), (max(p + n for p, n in zip(pos, q_lens)) + 15) // 16
    qkv = f16r(rng.standard_normal((T, (nq + 2 * nkv) * hd)))
    tables = rng.permutation(S * mb).astype(np.int32).reshape(S, mb)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    ck, cv = B.alloc_paged_pool(S * mb, nkv, hd), B.alloc_paged_pool(S * mb, nkv, hd)
    one, cos, sin = torch.ones(hd, dtype=torch.float16, device="cuda"), torch.ones(512, hd // 2, device="cuda"), torch.zeros(512, hd // 2, device="cuda")
    q_out = torch.full((T + 1, nq * hd), 7.0, dtype=torch.float16, device="cuda")
    B.split_qkv_norm_rope_into_paged_cache_varlen(ctx, dev16(torch, qkv), one, one, cos, sin, q_out, ck, cv, torch.from_numpy(cu).cuda(),
                                                  torch.from_numpy(np.array(pos, np.int32)).cuda(), torch.from_numpy(tables).cuda(), S, T, nq, nkv, hd, 1e-6, 0, 16, mb)
    ctx.sync()
    assert np.array_equal(host(q_out)[:T], qkv[:, :nq * hd]) and np.all(host(q_out)[T] == 7.0)
    left = [ck.float().abs().sum().item(), cv.float().abs().sum().item()]
    for s in range(S):
        kk, vv = B.paged_kv_read(ctx, ck, cv, torch.from_numpy(tables[s]).cuda(), pos[s] + q_lens[s], nkv, hd)
        ctx.sync()
        for got, at in ((kk, nq), (vv, nq + nkv)):
            got = host(got).reshape(-1, nkv * hd)
            assert np.array_equal(got[pos[s]:], qkv[cu[s]:cu[s + 1], at * hd:(at + nkv) * hd]) and not got[:pos[s]].any()
    want = [np.abs(qkv[:, at * hd:(at + nkv) * hd].astype(np.float64)).sum() for at in (nq, nq + nkv)]
    assert np.allclose(left, want, rtol=1e-4)                              # nothing else was written


@pytest.mark.parametrize("qk_mode,hd", [(1, 128), (2, 128), (3, 128), (0, 128), (1, 64), (2, 256)])
def test_split_qkv_norm_rope_into_paged_cache_varlen(env, qk_mode, hd):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(qk_mode * 10 + hd)
    nq, nkv, bs = 8, 2, 16
    q_lens, pos_offs = [5, 1, 19], [3, 40, 0]               # mixed prefill chunks + a decode row
    num_seqs, m_total = len(q_lens), sum(q_lens)
    max_blocks, num_blocks = 8, 32
    cos, sin = _rope(O, hd, 128)
    qkv = f16r(rng.standard_normal((m_total, (nq + 2 * nkv) * hd)))
    qn, kn = f16r(1 + 0.1 * rng.standard_normal(hd)), f16r(1 + 0.1 * rng.standard_normal(hd))
    perm = rng.permutation(num_blocks)
    tables = np.zeros((num_seqs, max_blocks), np.int32)
    used = 0
    for s in range(num_seqs):
        nb = (pos_offs[s] + q_lens[s] + bs - 1) // bs
        tables[s, :nb] = perm[used:used + nb]
        used += nb
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    ck, cv = B.alloc_paged_pool(num_blocks, nkv, hd), B.alloc_paged_pool(num_blocks, nkv, hd)
    q_out = torch.empty(m_total, nq, hd, dtype=torch.float16, device="cuda")
    B.split_qkv_norm_rope_into_paged_cache_varlen(
        ctx, dev16(torch, qkv), dev16(torch, qn), dev16(torch, kn), torch.from_numpy(cos).cuda(),
        torch.from_numpy(sin).cuda(), q_out, ck, cv, torch.from_numpy(cu).cuda(),
        torch.from_numpy(np.array(pos_offs, np.int32)).cuda(), torch.from_numpy(tables).cuda(), num_seqs, m_total, nq,
        nkv, hd, 1e-6, qk_mode, bs, max_blocks)
    ctx.sync()
    for s in range(num_seqs):
        rows = qkv[cu[s]:cu[s + 1]]
        q, k, v = O.split_qkv(rows, nq * hd, nkv * hd)
        T = q_lens[s]
        q_ref = O.qk_norm_rope(q.reshape(T, nq, hd), qn, cos, sin, T, nq, hd, pos_offs[s], 1e-6, qk_mode).transpose(1, 0, 2)
        k_ref = O.qk_norm_rope(k.reshape(T, nkv, hd), kn, cos, sin, T, nkv, hd, pos_offs[s], 1e-6, qk_mode).transpose(1, 0, 2)
        v_ref = v.reshape(T, nkv, hd)
        assert nmse(q_ref, host(q_out[cu[s]:cu[s + 1]])) < NMSE_FP16_TOL
        kv_len = pos_offs[s] + T
        kk, vv = B.paged_kv_read(ctx, ck, cv, torch.from_numpy(tables[s]).cuda(), kv_len, nkv, hd)
        ctx.sync()
        kk, vv = host(kk), host(vv)
        assert nmse(k_ref, kk[pos_offs[s]:]) < NMSE_FP16_TOL
        assert np.array_equal(vv[pos_offs[s]:], v_ref)                     # V is a copy: exact
        assert not kk[:pos_offs[s]].any() and not vv[:pos_offs[s]].any()   # earlier slots untouched
    # bit-exact KV-block indexing: only the blocks named by the tables were written
    written = set(int(b) for s in range(num_seqs) for b in
                  tables[s, pos_offs[s] // bs:(pos_offs[s] + q_lens[s] + bs - 1) // bs])
    pool = host(ck).reshape(num_blocks, -1)
    for blk in range(num_blocks):
        assert bool(pool[blk].any()) == (blk in written)


def test_ragged_batch_of_many_sequences_including_empty_ones(env):
    """150 sequences (more than two 64-wide passes of the in-kernel sequence lookups), a few of them with no query token at
    all: the split/norm/RoPE/paged-write op and the ragged attention grid must place every token with its own sequence."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(2025)
    nq, nkv, hd, bs, S = 4, 2, 64, 16, 150
    q_lens = [int(x) for x in rng.integers(1, 7, size=S)]
    for s in (0, 63, 64, 65, 128, 149):
        q_lens[s] = 0                                           # empty sequences at chunk boundaries and both ends
    q_lens[10], q_lens[100] = 40, 23                            # a few longer chunks
    pos_offs = [int(x) for x in rng.integers(0, 20, size=S)]
    kv_lens = [p + t for p, t in zip(pos_offs, q_lens)]
    max_blocks = (max(kv_lens) + bs - 1) // bs
    num_blocks = sum((n + bs - 1) // bs for n in kv_lens) + 1
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used = 0
    for s, n in enumerate(kv_lens):
        nb = (n + bs - 1) // bs
        tables[s, :nb] = perm[used:used + nb]
        used += nb
    m_total = sum(q_lens)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    cos, sin = _rope(O, hd, 128)
    qkv = f16r(rng.standard_normal((m_total, (nq + 2 * nkv) * hd)))
    qn, kn = f16r(1 + 0.1 * rng.standard_normal(hd)), f16r(1 + 0.1 * rng.standard_normal(hd))
    # context already in the cache: fill it through the same op, one "prefill" of pos_offs[s] tokens per sequence
    ctx_lens = pos_offs
    ctx_total = sum(ctx_lens)
    ccu = np.concatenate([[0], np.cumsum(ctx_lens)]).astype(np.int32)
    ctx_qkv = f16r(rng.standard_normal((ctx_total, (nq + 2 * nkv) * hd)))
    ck, cv = B.alloc_paged_pool(num_blocks, nkv, hd), B.alloc_paged_pool(num_blocks, nkv, hd)
    cosd, sind, td = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda(), torch.from_numpy(tables).cuda()
    scratch = torch.empty(max(ctx_total, 1), nq, hd, dtype=torch.float16, device="cuda")
    B.split_qkv_norm_rope_into_paged_cache_varlen(ctx, dev16(torch, ctx_qkv), dev16(torch, qn), dev16(torch, kn), cosd, sind, scratch,
                                                  ck, cv, torch.from_numpy(ccu).cuda(), torch.zeros(S, dtype=torch.int32, device="cuda"),
                                                  td, S, ctx_total, nq, nkv, hd, 1e-6, 1, bs, max_blocks)
    q_out = torch.empty(m_total, nq, hd, dtype=torch.float16, device="cuda")
    B.split_qkv_norm_rope_into_paged_cache_varlen(ctx, dev16(torch, qkv), dev16(torch, qn), dev16(torch, kn), cosd, sind, q_out, ck, cv,
                                                  torch.from_numpy(cu).cuda(), torch.from_numpy(np.array(pos_offs, np.int32)).cuda(),
                                                  td, S, m_total, nq, nkv, hd, 1e-6, 1, bs, max_blocks)
    out = torch.full((m_total + 1, nq, hd), 5.0, dtype=torch.float16, device="cuda")
    B.paged_varlen_attention(ctx, q_out, ck, cv, out, torch.from_numpy(cu).cuda(), torch.from_numpy(np.array(pos_offs, np.int32)).cuda(),
                             td, S, m_total, max(kv_lens), nq, nkv, hd, 0, bs, max_blocks, max(q_lens))
    ctx.sync()
    got_q, got = host(q_out), host(out)
    assert np.all(got[m_total] == 5.0)
    for s in range(S):
        T = q_lens[s]
        if T == 0:
            continue
        q, k, v = O.split_qkv(qkv[cu[s]:cu[s + 1]], nq * hd, nkv * hd)
        q_ref = O.qk_norm_rope(q.reshape(T, nq, hd), qn, cos, sin, T, nq, hd, pos_offs[s], 1e-6, 1).transpose(1, 0, 2)
        assert nmse(q_ref, got_q[cu[s]:cu[s + 1]]) < NMSE_FP16_TOL, s
        kk, vv = B.paged_kv_read(ctx, ck, cv, td[s], kv_lens[s], nkv, hd)
        ctx.sync()
        ref = _ref_attention(O, got_q[cu[s]:cu[s + 1]], host(kk), host(vv), pos_offs[s], nq, nkv, hd, 0)
        assert nmse(ref, got[cu[s]:cu[s + 1]]) < 1e-5, s


# ── contiguous-KV lane of the core trait (kv_layer.rs:370-513) ────────────────
@pytest.mark.parametrize("nq,nkv,hd,mode,window", [(8, 2, 128, 1, 0), (4, 4, 64, 2, 0), (6, 2, 128, 3, 5), (2, 1, 256, 1, 3)])
def test_contiguous_lane_prefill_then_decode(env, nq, nkv, hd, mode, window):
    """split_qkv → qk_norm_rope (→ head-major) → kv_cache_append_head_major → flash_attention → transpose_head_to_token,
    op by op against the CPU restatement (cpu.rs:1645-1783,1993-2060,2179-2259), for a 9-token prefill followed by a decode
    token at position 9; plus copy_slice / scaled_add_inplace / transpose_token_to_head."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(nq * 7 + hd + mode)
    cap = 32
    cos, sin = _rope(O, hd, cap)
    cosd, sind = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()
    qn, kn = f16r(1 + 0.1 * rng.standard_normal(hd)), f16r(1 + 0.1 * rng.standard_normal(hd))
    q_dim, kv_dim = nq * hd, nkv * hd
    ck = torch.zeros(nkv, cap, hd, dtype=torch.float16, device="cuda")
    cv = torch.zeros_like(ck)
    ck_ref, cv_ref = np.zeros((nkv, cap, hd), np.float32), np.zeros((nkv, cap, hd), np.float32)
    cache_len = 0
    for T in (9, 1):
        qkv = f16r(rng.standard_normal((T, q_dim + 2 * kv_dim)))
        qd, kd, vd = (torch.empty(T, n, dtype=torch.float16, device="cuda") for n in (q_dim, kv_dim, kv_dim))
        B.split_qkv(ctx, dev16(torch, qkv), qd, kd, vd, T, q_dim, kv_dim)
        ctx.sync()
        q, k, v = O.split_qkv(qkv, q_dim, kv_dim)
        assert np.array_equal(host(qd), q) and np.array_equal(host(kd), k) and np.array_equal(host(vd), v)
        qh = torch.empty(nq, T, hd, dtype=torch.float16, device="cuda")
        kh = torch.empty(nkv, T, hd, dtype=torch.float16, device="cuda")
        vh = torch.empty(nkv, T, hd, dtype=torch.float16, device="cuda")
        B.qk_norm_rope(ctx, qd, dev16(torch, qn), cosd, sind, qh, T, nq, hd, cache_len, 1e-6, mode)
        B.qk_norm_rope(ctx, kd, dev16(torch, kn), cosd, sind, kh, T, nkv, hd, cache_len, 1e-6, mode)
        B.qk_norm_rope(ctx, vd, dev16(torch, kn), cosd, sind, vh, T, nkv, hd, cache_len, 1e-6, 0)
        ctx.sync()
        q_ref = O.qk_norm_rope(q.reshape(T, nq, hd), qn, cos, sin, T, nq, hd, cache_len, 1e-6, mode)
        k_ref = O.qk_norm_rope(k.reshape(T, nkv, hd), kn, cos, sin, T, nkv, hd, cache_len, 1e-6, mode)
        v_ref = O.qk_norm_rope(v.reshape(T, nkv, hd), kn, cos, sin, T, nkv, hd, cache_len, 1e-6, 0)
        assert nmse(q_ref, host(qh)) < NMSE_FP16_TOL and nmse(k_ref, host(kh)) < NMSE_FP16_TOL
        assert np.array_equal(host(vh), v_ref)                                   # mode 0 = transpose only
        B.kv_cache_append_head_major(ctx, ck, cv, cache_len, cap, kh, vh, T, nkv, hd)
        ck_ref[:, cache_len:cache_len + T] = host(kh)
        cv_ref[:, cache_len:cache_len + T] = host(vh)
        kv_len = cache_len + T
        out = torch.full((nq, T, hd), 3.0, dtype=torch.float16, device="cuda")
        B.flash_attention(ctx, qh, ck, cv, out, 1, T, kv_len, cache_len, nq, nkv, hd, causal=True, kv_seq_stride=cap,
                          sliding_window=window)
        ctx.sync()
        assert np.array_equal(host(ck), ck_ref) and np.array_equal(host(cv), cv_ref)
        a_ref = O.cpu_attention(host(qh), ck_ref, cv_ref, T, kv_len, True, cache_len, nq, nkv, hd, sliding_window=window,
                                kv_seq_stride=cap)
        assert nmse(a_ref, host(out)) < 1e-5
        tm_ = torch.empty(T, nq, hd, dtype=torch.float16, device="cuda")
        B.transpose_head_to_token(ctx, out, tm_, T, nq, hd)
        back = torch.empty_like(out)
        B.transpose_token_to_head(ctx, tm_, back, T, nq, hd)
        ctx.sync()
        assert np.array_equal(host(tm_), host(out).transpose(1, 0, 2)) and torch.equal(back, out)
        cache_len = kv_len
    a = dev16(torch, rng.standard_normal(1000))
    b = dev16(torch, rng.standard_normal(1000))
    ref = host(a).copy()
    ref[100:400] = f16r(ref[100:400] + np.float32(0.37) * host(b)[5:305])
    B.scaled_add_inplace(ctx, a[100:], b[5:], 0.37, 300)
    c = torch.zeros(64, dtype=torch.float16, device="cuda")
    B.copy_slice(ctx, b, 17, c, 3, 40)
    ctx.sync()
    assert np.array_equal(host(a), ref)
    exp = np.zeros(64, np.float32)
    exp[3:43] = host(b)[17:57]
    assert np.array_equal(host(c), exp)


# ── paged attention ──────────────────────────────────────────────────────────
def _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks):
    """Write per-sequence K/V [len,nkv,hd] into native pools through the product's own writer (mode 0)."""
    pkg, B, ctx, O, torch = env
    ck, cv = B.alloc_paged_pool(num_blocks, nkv, hd), B.alloc_paged_pool(num_blocks, nkv, hd)
    nq = nkv
    for s, n in enumerate(kv_lens):
        qkv = np.concatenate([np.zeros((n, nq * hd), np.float32), K[s].reshape(n, -1), V[s].reshape(n, -1)], axis=1)
        q_out = torch.empty(n, nq, hd, dtype=torch.float16, device="cuda")
        dummy = dev16(torch, np.ones(hd))
        cs = torch.zeros(max(kv_lens) + 1, hd // 2, device="cuda")
        B.split_qkv_norm_rope_into_paged_cache_varlen(
            ctx, dev16(torch, qkv), dummy, dummy, cs, cs, q_out, ck, cv,
            torch.tensor([0, n], dtype=torch.int32, device="cuda"), torch.tensor([0], dtype=torch.int32, device="cuda"),
            torch.from_numpy(tables[s:s + 1].copy()).cuda(), 1, n, nq, nkv, hd, 1e-6, 0, 16, tables.shape[1])
    ctx.sync()
    return ck, cv


def _ref_attention(O, q, K, V, pos_offset, nq, nkv, hd, window=0):
    """q [T,nq,hd] at positions pos_offset.. over K/V [len,nkv,hd] → [T,nq,hd] (cpu.rs:2179-2259)."""
    T, kv_len = q.shape[0], K.shape[0]
    out = O.cpu_attention(q.transpose(1, 0, 2), K.transpose(1, 0, 2), V.transpose(1, 0, 2), T, kv_len, True, pos_offset,
                          nq, nkv, hd, sliding_window=window)
    return out.transpose(1, 0, 2)


def test_paged_decode_uniform_scores_golden(env):
    # ferrum-kv/src/attention.rs:162-195: equal scores → output = mean(V) = 2.0
    pkg, B, ctx, O, torch = env
    nq = nkv = 2
    hd = 64
    K = [np.ones((3, nkv, hd), np.float32)]
    V = [np.stack([np.full((nkv, hd), p + 1, np.float32) for p in range(3)])]
    tables = np.array([[5, 0]], np.int32)
    ck, cv = _fill_pool(env, K, V, tables, [3], nkv, hd, 8)
    out = torch.empty(1, nq, hd, dtype=torch.float16, device="cuda")
    B.paged_batched_decode_attention(ctx, dev16(torch, np.ones((1, nq, hd))), ck, cv, out, torch.from_numpy(tables).cuda(),
                                     torch.tensor([3], dtype=torch.int32, device="cuda"), 1, 3, nq, nkv, hd, 16, 2)
    ctx.sync()
    assert np.all(np.abs(host(out) - 2.0) < 1e-3)


@pytest.mark.parametrize("nq,nkv,hd,kv_lens", [(32, 4, 128, [1, 16, 17, 257, 300, 384, 33, 250]),
                                               (32, 8, 128, [100, 5]), (8, 8, 128, [48]), (16, 1, 128, [700, 31]),
                                               (4, 2, 64, [77]), (8, 2, 256, [40, 130])])
def test_paged_batched_decode_attention(env, nq, nkv, hd, kv_lens):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(nq + nkv + hd + len(kv_lens))
    S = len(kv_lens)
    max_blocks = (max(kv_lens) + 15) // 16 + 1
    num_blocks = sum((n + 15) // 16 for n in kv_lens) + 3
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used = 0
    K, V = [], []
    for s, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    q = f16r(rng.standard_normal((S, nq, hd)))
    out = torch.empty(S, nq, hd, dtype=torch.float16, device="cuda")
    B.paged_batched_decode_attention(ctx, dev16(torch, q), ck, cv, out, torch.from_numpy(tables).cuda(),
                                     torch.from_numpy(np.array(kv_lens, np.int32)).cuda(), S, max(kv_lens), nq, nkv, hd,
                                     16, max_blocks)
    ctx.sync()
    got = host(out)
    for s, n in enumerate(kv_lens):
        ref = _ref_attention(O, q[s:s + 1], K[s], V[s], n - 1, nq, nkv, hd)
        assert nmse(ref, got[s:s + 1]) < 1e-5, (s, n)          # far inside the 5e-3 attention bucket
        # cross-check with the second reference formulation (ferrum-kv attention.rs three-pass softmax)
    assert NMSE_ATTN_TOL > 1e-5


@pytest.mark.parametrize("window,nq,nkv,hd", [(0, 8, 2, 128), (24, 8, 2, 128), (0, 14, 2, 128), (40, 28, 4, 128), (0, 4, 4, 64),
                                              (17, 6, 6, 64), (0, 4, 1, 256), (33, 32, 16, 128), (1, 8, 2, 128)])
def test_paged_varlen_attention_mixed_batch(env, window, nq, nkv, hd, knobs, forms):
    pkg, B, ctx, O, torch = env
    # half of the cases ask for the row-split (prefill) form; it applies from 4 row tiles per sequence (37 tokens × GQA group / 16)
    want_rs = (window + nq) % 2 == 0 and -(-37 * (nq // nkv) // 16) >= 4
    if (window + nq) % 2 == 0:
        knobs.set(ATTN_RS_MIN_WGS=1)
    rng = np.random.default_rng(11 + window + nq + hd)
    q_lens, pos_offs = [37, 1, 16, 3], [0, 90, 20, 250]       # fresh prefill, decode, chunk, late chunk
    S = len(q_lens)
    kv_lens = [p + t for p, t in zip(pos_offs, q_lens)]
    max_blocks = (max(kv_lens) + 15) // 16
    num_blocks = sum((n + 15) // 16 for n in kv_lens) + 1
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used, K, V = 0, [], []
    for s, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    m_total = sum(q_lens)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    q = f16r(rng.standard_normal((m_total, nq, hd)))
    out = torch.zeros(m_total, nq, hd, dtype=torch.float16, device="cuda")
    B.paged_varlen_attention(ctx, dev16(torch, q), ck, cv, out, torch.from_numpy(cu).cuda(),
                             torch.from_numpy(np.array(pos_offs, np.int32)).cuda(), torch.from_numpy(tables).cuda(), S,
                             m_total, max(kv_lens), nq, nkv, hd, window, 16, max_blocks, max(q_lens))
    ctx.sync()
    forms.require("attn_row_split" if want_rs else "attn_kv_narrow", absent=("attn_flash",))
    got = host(out)
    for s in range(S):
        ref = _ref_attention(O, q[cu[s]:cu[s + 1]], K[s], V[s], pos_offs[s], nq, nkv, hd, window)
        assert nmse(ref, got[cu[s]:cu[s + 1]]) < 1e-5, s
    if window == 0:
        # the paged reference (attention.rs:30-114) agrees for the fresh-prefill sequence
        pk = np.zeros((num_blocks, 16, nkv, hd), np.float32)
        pv = np.zeros_like(pk)
        for p in range(kv_lens[0]):
            pk[tables[0, p // 16], p % 16] = K[0][p]
            pv[tables[0, p // 16], p % 16] = V[0][p]
        ref2 = O.paged_attention(q[:q_lens[0]], q_lens[0], nq, nkv, hd, pk, pv, tables[0], 16, kv_lens[0])
        assert nmse(ref2, got[:q_lens[0]]) < 1e-5


@pytest.mark.parametrize("window", [0, 50])
def test_paged_varlen_attention_many_prefill_tiles_row_split(env, window, knobs, forms):
    """24 prompts × 200 tokens (GQA group 2 ⇒ 25 row tiles each): enough workgroups for the row-split prefill form on its own
    heuristic; every sequence against the CPU restatement."""
    pkg, B, ctx, O, torch = env
    knobs.set(ATTN_NO_FLASH=1, ATTN_NO_RESIDENT=1)                 # the flash and resident-K/V forms have their own tests below
    rng = np.random.default_rng(77 + window)
    nq, nkv, hd, S, T = 8, 4, 128, 24, 200
    q_lens, pos_offs = [T] * S, [0] * (S - 2) + [48, 5]            # two of them continue an existing context
    kv_lens = [p + t for p, t in zip(pos_offs, q_lens)]
    max_blocks = (max(kv_lens) + 15) // 16
    num_blocks = sum((n + 15) // 16 for n in kv_lens) + 1
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used, K, V = 0, [], []
    for s, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    m_total = sum(q_lens)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    q = f16r(rng.standard_normal((m_total, nq, hd)))
    out = torch.zeros(m_total, nq, hd, dtype=torch.float16, device="cuda")
    B.paged_varlen_attention(ctx, dev16(torch, q), ck, cv, out, torch.from_numpy(cu).cuda(),
                             torch.from_numpy(np.array(pos_offs, np.int32)).cuda(), torch.from_numpy(tables).cuda(), S,
                             m_total, max(kv_lens), nq, nkv, hd, window, 16, max_blocks, max(q_lens))
    ctx.sync()
    forms.require("attn_row_split", absent=("attn_flash", "attn_kv_narrow"))
    got = host(out)
    for s in range(S):
        ref = _ref_attention(O, q[cu[s]:cu[s + 1]], K[s], V[s], pos_offs[s], nq, nkv, hd, window)
        assert nmse(ref, got[cu[s]:cu[s + 1]]) < 1e-5, s


@pytest.mark.parametrize("window,nq,nkv,hd", [(0, 8, 2, 128), (24, 8, 2, 128), (0, 14, 2, 128), (40, 32, 4, 128), (0, 4, 4, 64),
                                              (17, 6, 6, 64), (0, 4, 1, 256), (33, 32, 16, 128), (1, 8, 2, 128)])
def test_paged_prefill_attention_lds_shared_kv(env, window, nq, nkv, hd, knobs, forms):
    """The flash form (K/V of a block pair staged once per workgroup in LDS, 8 row tiles per workgroup): ragged prefill batch —
    fresh prompts, chunks that continue a context, a sequence shorter than one workgroup unit, odd block counts."""
    pkg, B, ctx, O, torch = env
    knobs.set(ATTN_FLASH_MIN_ROWS=1)
    rng = np.random.default_rng(5 + window + nq + hd)
    q_lens, pos_offs = [70, 33, 64, 17, 49], [0, 90, 20, 5, 300]
    S = len(q_lens)
    kv_lens = [p + t for p, t in zip(pos_offs, q_lens)]
    max_blocks = (max(kv_lens) + 15) // 16
    num_blocks = sum((n + 15) // 16 for n in kv_lens) + 1
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used, K, V = 0, [], []
    for s, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    m_total = sum(q_lens)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    q = f16r(rng.standard_normal((m_total, nq, hd)))
    out = torch.full((m_total + 1, nq, hd), 9.0, dtype=torch.float16, device="cuda")      # guard row
    B.paged_varlen_attention(ctx, dev16(torch, q), ck, cv, out, torch.from_numpy(cu).cuda(),
                             torch.from_numpy(np.array(pos_offs, np.int32)).cuda(), torch.from_numpy(tables).cuda(), S,
                             m_total, max(kv_lens), nq, nkv, hd, window, 16, max_blocks, max(q_lens))
    ctx.sync()
    forms.require("attn_flash", absent=("attn_row_split", "attn_kv_narrow"))
    got = host(out)
    assert np.all(got[m_total] == 9.0)
    for s in range(S):
        ref = _ref_attention(O, q[cu[s]:cu[s + 1]], K[s], V[s], pos_offs[s], nq, nkv, hd, window)
        assert nmse(ref, got[cu[s]:cu[s + 1]]) < 1e-5, s


@pytest.mark.parametrize("window,nq,nkv", [(0, 8, 2), (24, 8, 2), (0, 14, 2), (40, 32, 4), (0, 32, 16), (1, 8, 8)])
def test_paged_prefill_attention_resident_kv(env, window, nq, nkv, knobs, forms):
    """Short prompts whose whole context fits one LDS image (kv ≤ 256, head_dim 128): the resident-K/V form — fresh prompts, chunks
    that continue a context, odd block counts and block counts that are not a multiple of the four-block step, a sequence with
    fewer row tiles than waves, the full 256-key case, GQA groups 1 … 8 (7: rows of a token straddle tiles)."""
    pkg, B, ctx, O, torch = env
    knobs.set(ATTN_RESIDENT_MIN_WGS=1)
    hd = 128
    rng = np.random.default_rng(11 + window + nq)
    q_lens, pos_offs = [200, 33, 64, 256, 49, 100], [0, 90, 20, 0, 200, 70]
    S = len(q_lens)
    kv_lens = [p + t for p, t in zip(pos_offs, q_lens)]
    assert max(kv_lens) <= 256
    max_blocks = (max(kv_lens) + 15) // 16
    num_blocks = sum((n + 15) // 16 for n in kv_lens) + 1
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used, K, V = 0, [], []
    for s_, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s_, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    m_total = sum(q_lens)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    q = f16r(rng.standard_normal((m_total, nq, hd)))
    out = torch.full((m_total + 1, nq, hd), 9.0, dtype=torch.float16, device="cuda")      # guard row
    B.paged_varlen_attention(ctx, dev16(torch, q), ck, cv, out, torch.from_numpy(cu).cuda(),
                             torch.from_numpy(np.array(pos_offs, np.int32)).cuda(), torch.from_numpy(tables).cuda(), S,
                             m_total, max(kv_lens), nq, nkv, hd, window, 16, max_blocks, max(q_lens))
    ctx.sync()
    forms.require("attn_resident", absent=("attn_flash", "attn_row_split", "attn_kv_narrow"))
    got = host(out)
    assert np.all(got[m_total] == 9.0)
    for s_ in range(S):
        ref = _ref_attention(O, q[cu[s_]:cu[s_ + 1]], K[s_], V[s_], pos_offs[s_], nq, nkv, hd, window)
        assert nmse(ref, got[cu[s_]:cu[s_ + 1]]) < 1e-5, s_


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("window,nq,nkv", [(0, 8, 2), (24, 14, 2), (0, 32, 4), (1, 6, 6), (40, 3, 1)])
def test_paged_prefill_attention_in_both_unit_sizes(env, window, nq, nkv, rows, knobs, forms):
    knobs.set(ATTN_FLASH_ROWS=rows)
    test_paged_prefill_attention_lds_shared_kv(env, window, nq, nkv, 128, knobs, forms)


KEYS, WIDE, SHARED, BROAD, OTHER = "attn_keys", "attn_keys_wide", "attn_flash_64", "attn_flash", "attn_kv_narrow"


@pytest.mark.parametrize("q_lens,pos,window,nq,nkv,form", [
    ([250], 0, 0, 64, 8, SHARED), ([300], 0, 0, 64, 8, KEYS), ([300, 260], 0, 0, 64, 8, SHARED), ([700], 0, 0, 64, 8, SHARED), ([740], 0, 0, 64, 8, KEYS), ([500] * 3, 0, 0, 32, 8, SHARED),
    ([513] * 3, 0, 0, 32, 8, KEYS), ([400], 0, 100, 32, 4, SHARED), ([400], 500, 100, 32, 4, KEYS), ([400], 0, 129, 32, 4, KEYS), ([132], 396, 0, 32, 8, OTHER), ([132], 924, 0, 32, 8, WIDE),
    ([264], 800, 0, 16, 2, OTHER), ([500], 800, 0, 16, 2, WIDE), ([1439], 0, 256, 32, 8, KEYS), ([1440], 0, 256, 32, 8, BROAD), ([719], 0, 0, 128, 8, KEYS), ([720], 0, 0, 128, 8, BROAD),
    ([1279], 0, 0, 64, 4, KEYS), ([1280], 0, 0, 64, 4, BROAD)])
def test_form_of_a_prompt_by_its_workgroups_and_keys(env, q_lens, pos, window, nq, nkv, form, forms):
    """Which form a prompt takes on either side of each line; up to 600 tokens its results, too, against float32 (bound: see the test below)."""
    pkg, B, ctx, O, torch = env
    S, total, kv = len(q_lens), sum(q_lens), [pos + t for t in q_lens]
    mb = (max(kv) + 15) // 16
    gen = torch.Generator("cuda").manual_seed(total)
    rand = lambda *n: torch.randn(*n, generator=gen, device="cuda").half()
    K, V, q = [rand(n, nkv, 128) for n in kv], [rand(n, nkv, 128) for n in kv], rand(total, nq, 128)
    tables = torch.randperm(S * mb, generator=gen, device="cuda").to(torch.int32).reshape(S, mb)
    ck, cv = _fill_pool(env, [host(x) for x in K], [host(x) for x in V], tables.cpu().numpy(), kv, nkv, 128, S * mb)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    out = torch.full((total + 1, nq, 128), 9.0, dtype=torch.float16, device="cuda")
    forms.reset()
    B.paged_varlen_attention(ctx, q, ck, cv, out, torch.from_numpy(cu).cuda(), torch.full((S,), pos, dtype=torch.int32, device="cuda"), tables, S, total, max(kv), nq, nkv, 128,
                             window, 16, mb, max(q_lens))
    ctx.sync()
    h = forms.hits()
    assert h.get(form) and not any(h.get(f) for f in (KEYS, WIDE, SHARED, OTHER) if f != form), h
    assert bool((out[total] == 9.0).all()) and bool(torch.isfinite(out).all())
    for s in range(S if total <= 600 else 0):
        ref = _ref_attention(O, host(q[cu[s]:cu[s + 1]]), host(K[s]), host(V[s]), pos, nq, nkv, 128, window)
        assert nmse(ref, host(out[cu[s]:cu[s + 1]])) < 4 * 2.0 ** -22, s


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("q_lens,pos,window,nq,nkv", [
    ([9], [0], 0, 8, 8), ([64], [0], 0, 1, 1), ([65, 31], [0, 97], 0, 2, 2), ([16, 17], [15, 16], 0, 8, 2), ([128, 9], [129, 1000], 0, 14, 2),
    ([300], [0], 33, 4, 2), ([40, 200], [700, 31], 64, 6, 6), ([22, 5, 70], [490, 3, 256], 1, 32, 4), ([258], [511], 0, 16, 8)])
def test_prompt_attention_with_keys_by_wave(env, q_lens, pos, window, nq, nkv, waves, knobs, forms):
    """Keys split over the waves of a workgroup: waves without any, rows and keys that do not fill a tile, a page or a step, groups that do not divide a tile, windows
    that begin inside a step and leave waves nothing.  Against float32: probabilities and results are rounded by at most 2^-11 of themselves, (2 x 2^-11)^2 squared."""
    pkg, B, ctx, O, torch = env
    knobs.set(ATTN_FLASH_ROWS=64, ATTN_FLASH_MIN_ROWS=1, ATTN_KEY_WAVES=waves, ATTN_NO_RESIDENT=1)
    S, total, kv = len(q_lens), sum(q_lens), [p + t for p, t in zip(pos, q_lens)]
    mb = (max(kv) + 15) // 16
    gen = torch.Generator("cuda").manual_seed(total)
    rand = lambda *n: torch.randn(*n, generator=gen, device="cuda").half()
    K, V, q = [rand(n, nkv, 128) for n in kv], [rand(n, nkv, 128) for n in kv], rand(total, nq, 128)
    tables = torch.randperm(S * mb, generator=gen, device="cuda").to(torch.int32).reshape(S, mb)
    ck, cv = _fill_pool(env, [host(x) for x in K], [host(x) for x in V], tables.cpu().numpy(), kv, nkv, 128, S * mb)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    out = torch.full((total + 1, nq, 128), 9.0, dtype=torch.float16, device="cuda")
    B.paged_varlen_attention(ctx, q, ck, cv, out, torch.from_numpy(cu).cuda(), torch.tensor(pos, dtype=torch.int32, device="cuda"), tables, S, total, max(kv), nq, nkv, 128,
                             window, 16, mb, max(q_lens))
    ctx.sync()
    forms.require("attn_keys" if waves == 4 else "attn_keys_wide", absent=("attn_row_split", "attn_kv_narrow"))
    assert bool((out[total] == 9.0).all())
    for s in range(S):
        ref = _ref_attention(O, host(q[cu[s]:cu[s + 1]]), host(K[s]), host(V[s]), pos[s], nq, nkv, 128, window)
        assert nmse(ref, host(out[cu[s]:cu[s + 1]])) < 4 * 2.0 ** -22, s


@pytest.mark.parametrize("nq,nkv,q_lens,pos,flash", [
    (16, 8, [1500, 548], [0, 0], True), (16, 8, [293, 1389, 366], [1133, 0, 0], True), (16, 8, [100] * 6 + [1400], [0] * 7, True),
    (16, 8, [986], [366], True), (16, 8, [767], [0], False), (16, 8, [769], [0], True), (32, 8, [384], [0], True), (32, 8, [383], [1], False),
    (4, 2, [1] * 40 + [2500], [600] * 41, False), (32, 8, [2049], [0], True)])
def test_prompt_attention_takes_the_shared_form_by_size(env, nq, nkv, q_lens, pos, flash, forms, knobs):
    """Ragged batches on either side of the rule, against the forms without shared K/V (fp16 results of two orders of summation)."""
    pkg, B, ctx, O, torch = env
    S, total, kv = len(q_lens), sum(q_lens), max(p + t for p, t in zip(pos, q_lens))
    mb = (kv + 15) // 16
    gen = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *n: torch.randn(*n, device="cuda", generator=gen).half()
    k, v, q = rand(S * mb * nkv * 2048), rand(S * mb * nkv * 2048), rand(total, nq, 128)
    tables = torch.randperm(S * mb, device="cuda", generator=gen).to(torch.int32).reshape(S, mb)
    cu = torch.from_numpy(np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)).cuda()
    po = torch.from_numpy(np.array(pos, np.int32)).cuda()
    outs = []
    for off in (None, 1):
        knobs.set(ATTN_NO_FLASH=off)
        forms.reset()
        out = torch.zeros(total, nq, 128, dtype=torch.float16, device="cuda")
        B.paged_varlen_attention(ctx, q, k, v, out, cu, po, tables, S, total, kv, nq, nkv, 128, 0, 16, mb, max(q_lens))
        ctx.sync()
        assert bool(forms.hits().get("attn_flash")) == (flash and not off)
        outs.append(host(out))
    assert nmse(outs[1], outs[0]) < 1e-5


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("rise", [0.05, 0.12, 0.6, -0.05])
def test_prompt_attention_of_rising_scores(env, rise, rows, forms, knobs):
    """Maxima that move a little or far in every step, or never; four keys of 700 are hidden behind -inf."""
    pkg, B, ctx, O, torch = env
    knobs.set(ATTN_FLASH_ROWS=rows, ATTN_FLASH_MIN_ROWS=1)
    T, nq, nkv = 700, 4, 2
    mb = (T + 15) // 16
    gen = torch.Generator("cuda").manual_seed(5)
    q, k, v = (torch.randn(n, T, 128, generator=gen, device="cuda").half() for n in (nq, nkv, nkv))
    q[:, :, 0], k[:, :, 0] = 16.0, torch.arange(T, device="cuda") * (rise * 128 ** 0.5 / 16)          # a score of rise x position (nepers)
    k[:, 100:104, 0] = -float("inf")
    ck, cv = _fill_pool(env, [host(k.transpose(0, 1))], [host(v.transpose(0, 1))], np.arange(mb, dtype=np.int32)[None], [T], nkv, 128, mb)
    out = torch.empty(T, nq, 128, dtype=torch.float16, device="cuda")
    B.paged_varlen_attention(ctx, q.transpose(0, 1).contiguous(), ck, cv, out, torch.tensor([0, T], dtype=torch.int32, device="cuda"),
                             torch.zeros(1, dtype=torch.int32, device="cuda"), torch.arange(mb, dtype=torch.int32, device="cuda")[None], 1, T, T, nq, nkv, 128, 0, 16, mb, T)
    ctx.sync()
    forms.require("attn_flash")
    for h in range(nq):
        s = q[h].double() @ k[h // 2].double().T * 128 ** -0.5
        p = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -float("inf")).softmax(-1)
        want, size = p @ v[h // 2].double(), p @ v[h // 2].double().abs()
        # 16-bit probabilities in numerator and denominator (2^-11 each), scores of up to 420 in 32 bits (128 roundings of 2^-24 of their terms'
        # size), probabilities below 2^-14 (2^-25 each), the result
        bound = (2.0 ** -10 + 2 ** -24 * 128 * s.abs().nan_to_num(posinf=0).amax() / 4) * size + T * 2.0 ** -25 * 5 + 2.0 ** -11 * want.abs()
        assert ((out[:, h].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("spread", [1.0, 2.0, 4.0])
def test_prompt_attention_errs_as_its_rounded_probabilities(env, spread, rows, forms, knobs):
    """Keys in pairs whose values all but cancel, so that what is left of a result shows the rounding of its probabilities: no more of it than with each probability
    divided by the row's largest so far, which then is exactly 1.  The arithmetic beside that rounding is 32-bit (scores err by about 1e-6 of themselves, against 2.8e-4
    for a rounding), so the two errors agree to a few percent; with a reference 2^8 behind the maximum the first is 1.16 and 1.20 times the second at deviations of 2 and 4."""
    pkg, B, ctx, O, torch = env
    knobs.set(ATTN_FLASH_ROWS=rows, ATTN_FLASH_MIN_ROWS=1)
    T, nq, nkv = 1536, 4, 2
    mb = T // 16
    gen = torch.Generator("cuda").manual_seed(11)
    q, k, v = (torch.randn(n, T, 128, generator=gen, device="cuda") for n in (nq, nkv, nkv))
    q, k = (q * spread ** 0.5).half(), (k * spread ** 0.5).half()
    q[:, :, 0] = 16.0
    k[:, 1::2] = k[:, ::2]
    k[:, ::2, 0], k[:, 1::2, 0] = 0.0, 0.1 + 0.6 * torch.rand(nkv, T // 2, generator=gen, device="cuda").half()
    v[:, 1::2] = -v[:, ::2] * torch.exp(k[:, 1::2, :1].float() * -16 * 128 ** -0.5)
    v = v.half()
    ck, cv = _fill_pool(env, [host(k.transpose(0, 1))], [host(v.transpose(0, 1))], np.arange(mb, dtype=np.int32)[None], [T], nkv, 128, mb)
    out = torch.empty(T, nq, 128, dtype=torch.float16, device="cuda")
    B.paged_varlen_attention(ctx, q.transpose(0, 1).contiguous(), ck, cv, out, torch.tensor([0, T], dtype=torch.int32, device="cuda"),
                             torch.zeros(1, dtype=torch.int32, device="cuda"), torch.arange(mb, dtype=torch.int32, device="cuda")[None], 1, T, T, nq, nkv, 128, 0, 16, mb, T)
    ctx.sync()
    forms.require("attn_flash")
    got = allowed = 0.0
    for h in range(nq):
        s = q[h].double() @ k[h // 2].double().T * 128 ** -0.5
        s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -float("inf"))
        value = v[h // 2].double()
        largest = s.reshape(T, -1, 64).amax(-1).cummax(-1).values.repeat_interleave(64, -1)          # (a step takes 64 keys)
        p = (s - largest).exp().half().double() * (largest - largest[:, -1:]).exp()
        want = s.softmax(-1) @ value
        whole = slice(1, None, 2)                                   # (rows that see both keys of their last pair)
        got += ((out[:, h].double() - want)[whole] ** 2).sum().item()
        allowed += ((p @ value / p.sum(-1, keepdim=True) - want)[whole] ** 2).sum().item()
    assert got <= 1.05 ** 2 * allowed, (got / allowed) ** 0.5


def test_paged_prefill_attention_lds_shared_kv_many_sequences(env, knobs, forms):
    """The flash form over 70 sequences (two passes of its in-kernel sequence lookup), two of them empty."""
    pkg, B, ctx, O, torch = env
    knobs.set(ATTN_FLASH_MIN_ROWS=1)
    rng = np.random.default_rng(404)
    nq, nkv, hd, S = 4, 2, 128, 70
    q_lens = [int(x) for x in rng.integers(15, 26, size=S)]
    q_lens[0], q_lens[64] = 0, 0
    pos_offs = [int(x) for x in rng.integers(0, 40, size=S)]
    kv_lens = [p + t for p, t in zip(pos_offs, q_lens)]
    max_blocks = (max(kv_lens) + 15) // 16
    num_blocks = sum((n + 15) // 16 for n in kv_lens) + 1
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used, K, V = 0, [], []
    for s, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    m_total = sum(q_lens)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    q = f16r(rng.standard_normal((m_total, nq, hd)))
    out = torch.zeros(m_total, nq, hd, dtype=torch.float16, device="cuda")
    B.paged_varlen_attention(ctx, dev16(torch, q), ck, cv, out, torch.from_numpy(cu).cuda(),
                             torch.from_numpy(np.array(pos_offs, np.int32)).cuda(), torch.from_numpy(tables).cuda(), S,
                             m_total, max(kv_lens), nq, nkv, hd, 0, 16, max_blocks, max(q_lens))
    ctx.sync()
    forms.require("attn_flash", absent=("attn_row_split", "attn_kv_narrow"))
    got = host(out)
    for s in range(S):
        if q_lens[s] == 0:
            continue
        ref = _ref_attention(O, q[cu[s]:cu[s + 1]], K[s], V[s], pos_offs[s], nq, nkv, hd, 0)
        assert nmse(ref, got[cu[s]:cu[s + 1]]) < 1e-5, s


def test_paged_decode_long_context_split_kv(env, forms):
    # exercises the grid.z flash-decode split + reduce at a BASELINE-like head config (Qwen3-30B: 32/4 heads)
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(3)
    nq, nkv, hd, kv_lens = 32, 4, 128, [4096, 1500]
    S = 2
    max_blocks = (max(kv_lens) + 15) // 16
    num_blocks = sum((n + 15) // 16 for n in kv_lens)
    tables = np.zeros((S, max_blocks), np.int32)
    perm = rng.permutation(num_blocks)
    used, K, V = 0, [], []
    for s, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    q = f16r(rng.standard_normal((S, nq, hd)))
    q[0, 3] *= 6.0                                          # a peaked row: forces large online-softmax rescales
    out = torch.empty(S, nq, hd, dtype=torch.float16, device="cuda")
    B.paged_batched_decode_attention(ctx, dev16(torch, q), ck, cv, out, torch.from_numpy(tables).cuda(),
                                     torch.from_numpy(np.array(kv_lens, np.int32)).cuda(), S, max(kv_lens), nq, nkv, hd,
                                     16, max_blocks)
    ctx.sync()
    forms.require("attn_kv_wide", "attn_split_reduce")
    got = host(out)
    for s, n in enumerate(kv_lens):
        ref = _ref_attention(O, q[s:s + 1], K[s], V[s], n - 1, nq, nkv, hd)
        assert nmse(ref, got[s:s + 1]) < 1e-5


@pytest.mark.parametrize("nq,nkv,hd,kv_lens,qk_mode,window", [
    (32, 4, 128, [1, 16, 17, 257, 300, 384, 33, 250], 1, 0), (32, 8, 128, [100, 5], 2, 0), (8, 8, 128, [48], 3, 0),
    (16, 2, 128, [700, 31], 0, 0), (4, 2, 64, [77, 64, 65], 1, 0), (8, 2, 256, [40, 130], 1, 0), (32, 4, 128, [4096, 1500], 1, 0),
    (32, 16, 128, [300, 7, 1024, 1025, 40], 1, 64), (8, 2, 128, [90, 33], 2, 17)])
def test_paged_decode_attention_fused_qkv_equals_two_op_chain(env, nq, nkv, hd, kv_lens, qk_mode, window):
    """One-launch decode (QK-norm + RoPE + KV write in the attention prologue) is bit-identical — attention output
    AND both cache pools — to split_qkv_norm_rope_into_paged_cache_varlen + paged_batched_decode_attention."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(nq * 3 + nkv + hd + len(kv_lens) + qk_mode)
    S = len(kv_lens)
    max_blocks = (max(kv_lens) + 15) // 16 + 1
    num_blocks = sum((n + 15) // 16 for n in kv_lens) + 3
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used, K, V = 0, [], []
    for s, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))      # the last slot holds stale values the step overwrites
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    ck2, cv2 = ck.clone(), cv.clone()
    cos, sin = _rope(O, hd, max(kv_lens) + 1)
    cosd, sind = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()
    qkv = dev16(torch, rng.standard_normal((S, (nq + 2 * nkv) * hd)))
    qn, kn = dev16(torch, 1 + 0.1 * rng.standard_normal(hd)), dev16(torch, 1 + 0.1 * rng.standard_normal(hd))
    td = torch.from_numpy(tables).cuda()
    lens = torch.from_numpy(np.array(kv_lens, np.int32)).cuda()
    q_out = torch.empty(S, nq, hd, dtype=torch.float16, device="cuda")
    out1 = torch.empty(S, nq, hd, dtype=torch.float16, device="cuda")
    out2 = torch.zeros_like(out1)
    B.split_qkv_norm_rope_into_paged_cache_varlen(ctx, qkv, qn, kn, cosd, sind, q_out, ck, cv,
                                                  torch.arange(S + 1, dtype=torch.int32, device="cuda"), lens - 1, td, S, S,
                                                  nq, nkv, hd, 1e-6, qk_mode, 16, max_blocks)
    if window:      # sliding window: the varlen op is the two-op reference (decode form: one query token per sequence)
        B.paged_varlen_attention(ctx, q_out, ck, cv, out1, torch.arange(S + 1, dtype=torch.int32, device="cuda"), lens - 1, td, S, S,
                                 max(kv_lens), nq, nkv, hd, window, 16, max_blocks, max_q_len=1)
    else:
        B.paged_batched_decode_attention(ctx, q_out, ck, cv, out1, td, lens, S, max(kv_lens), nq, nkv, hd, 16, max_blocks)
    B.paged_decode_attention_fused_qkv(ctx, qkv, qn, kn, cosd, sind, 1e-6, qk_mode, ck2, cv2, out2, td, lens, S, max(kv_lens),
                                       nq, nkv, hd, 16, max_blocks, sliding_window=window)
    ctx.sync()
    assert torch.equal(ck, ck2) and torch.equal(cv, cv2)
    assert torch.equal(out1, out2)
    assert torch.isfinite(out2.float()).all()


# ── MoE ──────────────────────────────────────────────────────────────────────
@pytest.mark.parametrize("batch,ne,k,norm,seed", [(32, 128, 8, True, 0xDEADBEEF), (1, 128, 8, True, 0x1234),
                                                  (64, 128, 8, True, 0x5678), (8, 64, 4, False, 0xC0FFEE),
                                                  (4, 16, 1, True, 0x42), (3, 256, 8, True, 7)])
def test_route_topk_softmax(env, batch, ne, k, norm, seed):
    # router.rs:203-244 shapes; ids bit-exact, weights within the renorm-divide ulps (1e-6, :219-222)
    pkg, B, ctx, O, torch = env
    logits = O.Lcg(seed).array_f32(batch * ne, -3.0, 3.0).reshape(batch, ne)
    ids = torch.empty(batch, k, dtype=torch.int32, device="cuda")
    w = torch.empty(batch, k, dtype=torch.float32, device="cuda")
    B.route_topk_softmax(ctx, torch.from_numpy(logits).cuda(), ids, w, batch, ne, k, norm)
    ctx.sync()
    rid, rw = O.route_topk(logits, ne, k, norm)
    assert np.array_equal(ids.cpu().numpy().astype(np.uint32), rid)
    assert np.max(np.abs(w.cpu().numpy() - rw)) < 1e-6
    # fp16-logit entry point (moe_router.cu:32 form)
    l16 = f16r(logits)
    B.route_topk_softmax(ctx, dev16(torch, l16), ids, w, batch, ne, k, norm)
    ctx.sync()
    rid, rw = O.route_topk(l16, ne, k, norm)
    assert np.array_equal(ids.cpu().numpy().astype(np.uint32), rid)


def test_route_ties_lowest_index(env):
    pkg, B, ctx, O, torch = env
    logits = np.full((2, 128), 0.5, np.float32)
    ids = torch.empty(2, 8, dtype=torch.int32, device="cuda")
    w = torch.empty(2, 8, dtype=torch.float32, device="cuda")
    B.route_topk_softmax(ctx, torch.from_numpy(logits).cuda(), ids, w, 2, 128, 8, True)
    ctx.sync()
    assert np.array_equal(ids.cpu().numpy(), np.tile(np.arange(8), (2, 1)))
    assert np.all(np.abs(w.cpu().numpy() - 0.125) < 1e-7)


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("ne,k", [(1, 1), (2, 1), (7, 7), (8, 2), (9, 1), (24, 4), (24, 8), (25, 4), (31, 4), (40, 5), (41, 5), (48, 8), (49, 8), (63, 8), (64, 8), (64, 64), (65, 8)])
def test_route_by_place_and_by_maxima(env, ne, k, norm):
    """Up to six experts a choice, counted in eights, are ranked at once, more by one maximum after the other: numbers, ties, -inf and NaN among the logits, against k passes of a maximum in
    which a NaN takes no part, the first expert standing in where none is left."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(ne * 64 + k)
    logits = rng.standard_normal((8, ne)).astype(np.float32)
    logits[1] = 0.25
    logits[2, ::2] = 1.5
    logits[3] = np.round(logits[3])
    logits[4, ne // 2:] = -np.inf
    logits[5, 1:] = -200.0
    logits[6, ne - 1] = np.nan
    logits[7] = -np.inf
    ids, w = torch.empty(8, k, dtype=torch.int32, device="cuda"), torch.empty(8, k, dtype=torch.float32, device="cuda")
    B.route_topk_softmax(ctx, torch.from_numpy(logits).cuda(), ids, w, 8, ne, k, norm)
    ctx.sync()
    with np.errstate(all="ignore"):
        p = np.exp(logits - np.fmax.reduce(logits, axis=1, keepdims=True)).astype(np.float32)
        p /= p.sum(1, keepdims=True)
        for r in range(8):
            v, want, ww = p[r].copy(), [], []
            for _ in range(k):
                ok = np.where(v > -np.inf, v, -np.inf)
                e = int(np.argmax(ok)) if np.any(v > -np.inf) else 0
                want.append(e)
                ww.append(ok[e])
                v[e] = -np.inf
            total = np.float32(sum(ww))
            ww = (np.array(ww) / total if total > 0 else np.full(k, 1.0 / k)) if norm else np.array(ww)
            assert ids[r].tolist() == want, (r, ids[r].tolist(), want)
            got = w[r].cpu().numpy()
            assert np.all((np.abs(got - ww) < 1e-6) | (got == ww)), (r, got, ww)


@pytest.mark.parametrize("tokens,ne,k", [(1, 128, 8), (32, 128, 8), (700, 128, 8), (5, 8, 2), (0, 16, 2)])
def test_moe_align_block_size_bit_exact(env, tokens, ne, k):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens + ne)
    ids = np.stack([rng.choice(ne, size=k, replace=False) for _ in range(tokens)]).astype(np.int32) if tokens else \
        np.zeros((0, k), np.int32)
    n = tokens * k
    sorted_max = n + ne * 16
    sd = torch.full((sorted_max,), -7, dtype=torch.int32, device="cuda")
    bd = torch.full((sorted_max // 16 + 1,), -7, dtype=torch.int32, device="cuda")
    td = torch.zeros(1, dtype=torch.int32, device="cuda")
    B.moe_align_block_size_pair_ids(ctx, torch.from_numpy(ids.reshape(-1).copy()).cuda(), sd, bd, td, n, ne, 16, sorted_max)
    ctx.sync()
    rs, rb, rt = O.moe_align_block_size(ids, ne, 16)
    assert int(td.item()) == rt
    assert np.array_equal(sd.cpu().numpy(), rs)
    assert np.array_equal(bd.cpu().numpy()[:len(rb)], rb)


@pytest.mark.parametrize("tokens,E,K,H,I", [(1, 8, 2, 256, 128), (9, 8, 2, 256, 128), (32, 16, 4, 512, 256), (64, 8, 2, 256, 128),
                                            (32, 128, 8, 2048, 768), (96, 128, 8, 2048, 768),    # Qwen3-30B-A3B expert dims
                                            (1, 128, 8, 2048, 768), (7, 128, 8, 2048, 768)])
def test_moe_grouped_gemm_and_combine(env, tokens, E, K, H, I, forms):
    # whole expert MLP path vs moe_forward_cpu (dispatch.rs:2208-2288), plain and fused-silu stacks
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens * E + H)
    gu = [O.make_synthetic_gptq(H, 2 * I, 128, 100 + e, symmetric=True) for e in range(E)]
    dn = [O.make_synthetic_gptq(I, H, 128, 200 + e, symmetric=True) for e in range(E)]
    gu = [(q, f16r(s / (0.28 * np.sqrt(H))), z) for q, s, z in gu]
    dn = [(q, f16r(s / (0.28 * np.sqrt(I))), z) for q, s, z in dn]
    x = f16r(rng.standard_normal((tokens, H)))
    logits = rng.standard_normal((tokens, E)).astype(np.float32)
    rid, rw = O.route_topk(logits, E, K, True)
    gw = np.stack([O.dequant_gptq(q, s, z, 128, H, 2 * I) for q, s, z in gu])
    dw = np.stack([O.dequant_gptq(q, s, z, 128, I, H) for q, s, z in dn])
    ref = O.moe_forward_cpu(x, H, I, K, rid, rw, gw, dw)
    P = tokens * K
    sorted_max = P + E * 16
    ids_d = torch.from_numpy(rid.astype(np.int32).reshape(-1).copy()).cuda()
    sd = torch.empty(sorted_max, dtype=torch.int32, device="cuda")
    bd = torch.empty(sorted_max // 16 + 1, dtype=torch.int32, device="cuda")
    td = torch.zeros(1, dtype=torch.int32, device="cuda")
    B.moe_align_block_size_pair_ids(ctx, ids_d, sd, bd, td, P, E, 16, sorted_max)
    max_blocks = sorted_max // 16
    xd = dev16(torch, x)
    wd = torch.from_numpy(rw.reshape(-1).copy()).cuda()
    down_stack = B.load_gptq_stacked([q for q, _, _ in dn], [s for _, s, _ in dn], [z for _, _, z in dn], None, 4, 128, I, H)
    for fused in (False, True):
        stack = B.load_gptq_stacked([q for q, _, _ in gu], [s for _, s, _ in gu], [z for _, _, z in gu], None, 4, 128, H,
                                    2 * I, fuse_gate_up=fused)
        act = torch.zeros(P, I, dtype=torch.float16, device="cuda")
        if fused:
            stack.gemm_phase_vllm(ctx, xd, sd, bd, td, act, P, 16, K, max_blocks, fused_silu_mul=True)
        else:
            gup = torch.zeros(P, 2 * I, dtype=torch.float16, device="cuda")
            stack.gemm_phase_vllm(ctx, xd, sd, bd, td, gup, P, 16, K, max_blocks)
            B.fused_silu_mul_split(ctx, gup, act, P, I)
        down = torch.zeros(P, H, dtype=torch.float16, device="cuda")
        down_stack.gemm_phase_vllm(ctx, act, sd, bd, td, down, P, 16, 1, max_blocks)
        out = torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
        B.moe_combine(ctx, down, wd, out, tokens, K, H)
        ctx.sync()
        assert nmse(ref, host(out)) < 3e-6, fused            # three fp16 roundings (act, down, out)
        for blk in ((64, 32) + ((128, 96) if I % 256 == 0 and H % 256 == 0 else ()) if fused and P >= 64 else ()):
            # 64- and 32-row blocks through the prefill tile kernel: same maths, different block shape; 128-row blocks through
            # w4_gemm_big_kernel: the group scale folded into fp16 weights (one more rounding per weight, like the reference's own
            # fp16 dequantisation), so equal within the tolerance, not bit for bit
            sdb = torch.empty(P + E * blk, dtype=torch.int32, device="cuda")
            bdb = torch.empty((P + E * blk) // blk + 1, dtype=torch.int32, device="cuda")
            tdb = torch.zeros(1, dtype=torch.int32, device="cuda")
            B.moe_align_block_size_pair_ids(ctx, ids_d, sdb, bdb, tdb, P, E, blk, P + E * blk)
            mbb = (P + E * blk) // blk
            actb = torch.zeros(P, I, dtype=torch.float16, device="cuda")
            downb = torch.zeros(P, H, dtype=torch.float16, device="cuda")
            stack.gemm_phase_vllm(ctx, xd, sdb, bdb, tdb, actb, P, blk, K, mbb, fused_silu_mul=True)
            down_stack.gemm_phase_vllm(ctx, actb, sdb, bdb, tdb, downb, P, blk, 1, mbb)
            outb = torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
            B.moe_combine(ctx, downb, wd, outb, tokens, K, H)
            ctx.sync()
            if blk < 96: assert torch.equal(actb, act), blk      # per-row sums are independent of the block shape
            else: assert nmse(host(act), host(actb)) < 1e-6, blk
            assert nmse(ref, host(outb)) < 3e-6, blk
        # expert-major grid straight from the raw expert ids (no align arrays): bit-identical outputs; experts with more
        # than 16 pairs (the 64-token / 8-expert case) take further passes, experts without pairs leave early
        # (≤ 16 pairs of a K ≥ 512 stack: the block-major launches above split K over four waves — another fp32 summation order)
        same = (lambda x_, y_: torch.equal(x_, y_)) if P > 16 else (lambda x_, y_: nmse(host(x_), host(y_)) < 1e-6)
        down3 = torch.zeros(P, H, dtype=torch.float16, device="cuda")
        if fused:
            act3 = torch.zeros(P, I, dtype=torch.float16, device="cuda")
            stack.gemm_phase_expert_major(ctx, xd, ids_d, act3, P, E, K, fused_silu_mul=True)
            ctx.sync()
            assert same(act, act3)
        else:
            gup3 = torch.zeros(P, 2 * I, dtype=torch.float16, device="cuda")
            stack.gemm_phase_expert_major(ctx, xd, ids_d, gup3, P, E, K)
            ctx.sync()
            assert same(gup, gup3)
        down_stack.gemm_phase_expert_major(ctx, act3 if fused else act, ids_d, down3, P, E, 1)
        ctx.sync()
        assert same(down, down3)
        if fused and P <= 1024 and I >= 256:
            # gate_up → down as ONE launch (down tiles wait in the launch for their expert's gate_up tiles): the same bits, on
            # poisoned output buffers, three times over (the counters are re-armed per call)
            forms.reset()
            for rep in range(3):
                act4 = torch.full((P, I), float("nan"), dtype=torch.float16, device="cuda")
                down4 = torch.full((P, H), float("nan"), dtype=torch.float16, device="cuda")
                stack.gemm_phase_expert_major_pair(ctx, down_stack, xd, ids_d, act4, down4, P, E, K)
                ctx.sync()
                assert stack.pair_timeouts(ctx) == 0
                assert torch.equal(act3, act4) and torch.equal(down3, down4), rep      # the bits of the two expert-major launches
            forms.require("moe_expert_major_pair")
        if fused and P <= 64:
            # ≤ 64 pairs: gate_up → down as ONE block-major launch (four waves per tile split K, the whole tile in flight; down
            # tiles wait in the launch for their block's gate_up tiles): poisoned outputs, three times over.  ≤ 16 pairs: the bits
            # of the two K-split launches the runner would otherwise take; beyond, those launches do not split K → tolerance
            forms.reset()
            for rep in range(3):
                act5 = torch.full((P, I), float("nan"), dtype=torch.float16, device="cuda")
                down5 = torch.full((P, H), float("nan"), dtype=torch.float16, device="cuda")
                stack.gemm_phase_block_major_pair(ctx, down_stack, xd, ids_d, act5, down5, P, E, K, min(P, E))
                ctx.sync()
                assert stack.pair_timeouts(ctx) == 0
                out5 = torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
                B.moe_combine(ctx, down5, wd, out5, tokens, K, H)
                ctx.sync()
                assert nmse(ref, host(out5)) < 3e-6, rep
                if P <= 16:
                    actk = torch.zeros(P, I, dtype=torch.float16, device="cuda")
                    downk = torch.zeros(P, H, dtype=torch.float16, device="cuda")
                    stack.gemm_phase_inline_align(ctx, xd, ids_d, actk, P, E, K, max_blocks, fused_silu_mul=True)
                    down_stack.gemm_phase_inline_align(ctx, actk, ids_d, downk, P, E, 1, max_blocks)
                    ctx.sync()
                    assert torch.equal(actk, act5) and torch.equal(downk, down5), rep
                else:
                    assert nmse(host(act), host(act5)) < 1e-6 and nmse(host(down), host(down5)) < 1e-6, rep
            forms.require("moe_block_major_pair")
        if fused:
            # align computed inside the GEMM from the raw expert ids: bit-identical outputs
            act2 = torch.zeros(P, I, dtype=torch.float16, device="cuda")
            down2 = torch.zeros(P, H, dtype=torch.float16, device="cuda")
            stack.gemm_phase_inline_align(ctx, xd, ids_d, act2, P, E, K, max_blocks, fused_silu_mul=True)
            down_stack.gemm_phase_inline_align(ctx, act2, ids_d, down2, P, E, 1, max_blocks)
            ctx.sync()
            assert torch.equal(act, act2) and torch.equal(down, down2)


@pytest.mark.parametrize("tokens,E,K,H,I", [(9, 8, 2, 256, 128), (32, 128, 8, 2048, 768), (80, 128, 8, 2048, 768)])
@pytest.mark.parametrize("asym,desc_act", [(True, False), (False, True), (True, True)])
def test_moe_asymmetric_and_act_order_expert_stacks(env, tokens, E, K, H, I, asym, desc_act, forms):
    """Expert stacks with non-8 zero points (the reference's vLLM-Marlin branch, cuda/quant.rs:795-839) and with an act-order
    g_idx shared by the stack (cuda/quant.rs:862 ff., capabilities.rs:180-189) against moe_forward_cpu on weights dequantised
    WITH g_idx (cpu.rs:2283-2315): every phase entry point, at Qwen3-30B-A3B expert dims."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens * E + H + 2 * asym + desc_act)
    gu = [O.make_synthetic_gptq(H, 2 * I, 128, 300 + e, symmetric=not asym) for e in range(E)]
    dn = [O.make_synthetic_gptq(I, H, 128, 500 + e, symmetric=not asym) for e in range(E)]
    gu = [(q, f16r(s / (0.28 * np.sqrt(H))), z) for q, s, z in gu]
    dn = [(q, f16r(s / (0.28 * np.sqrt(I))), z) for q, s, z in dn]
    gi_gu = O.make_desc_act_g_idx(H, 128) if desc_act else None
    gi_dn = O.make_desc_act_g_idx(I, 128) if desc_act else None
    x = f16r(rng.standard_normal((tokens, H)))
    rid, rw = O.route_topk(rng.standard_normal((tokens, E)).astype(np.float32), E, K, True)
    gw = np.stack([O.dequant_gptq(q, s, z, 128, H, 2 * I, g_idx=gi_gu) for q, s, z in gu])
    dw = np.stack([O.dequant_gptq(q, s, z, 128, I, H, g_idx=gi_dn) for q, s, z in dn])
    ref = O.moe_forward_cpu(x, H, I, K, rid, rw, gw, dw)
    P = tokens * K
    ids_d = torch.from_numpy(rid.astype(np.int32).reshape(-1).copy()).cuda()
    xd, x_keep = dev16(torch, x), dev16(torch, x)
    wd = torch.from_numpy(rw.reshape(-1).copy()).cuda()
    stack = B.load_gptq_stacked([q for q, _, _ in gu], [s for _, s, _ in gu], [z for _, _, z in gu], gi_gu, 4, 128, H, 2 * I,
                                fuse_gate_up=True)
    down_stack = B.load_gptq_stacked([q for q, _, _ in dn], [s for _, s, _ in dn], [z for _, _, z in dn], gi_dn, 4, 128, I, H)

    def combine(down):
        out = torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
        B.moe_combine(ctx, down, wd, out, tokens, K, H)
        ctx.sync()
        return host(out)

    base = None
    for blk in (16, 64):
        sd = torch.empty(P + E * blk, dtype=torch.int32, device="cuda")
        bd = torch.empty((P + E * blk) // blk + 1, dtype=torch.int32, device="cuda")
        td = torch.zeros(1, dtype=torch.int32, device="cuda")
        B.moe_align_block_size_pair_ids(ctx, ids_d, sd, bd, td, P, E, blk, P + E * blk)
        mb = (P + E * blk) // blk
        act = torch.full((P, I), float("nan"), dtype=torch.float16, device="cuda")
        down = torch.full((P, H), float("nan"), dtype=torch.float16, device="cuda")
        stack.gemm_phase_vllm(ctx, xd, sd, bd, td, act, P, blk, K, mb, fused_silu_mul=True)
        down_stack.gemm_phase_vllm(ctx, act, sd, bd, td, down, P, blk, 1, mb)
        assert nmse(ref, combine(down)) < 3e-6, blk
        if base is None: base = (act, down)
        else: assert torch.equal(act, base[0]) and torch.equal(down, base[1])      # block shape does not change a row's sum
    act, down = base
    act3 = torch.full((P, I), float("nan"), dtype=torch.float16, device="cuda")
    down3 = torch.full((P, H), float("nan"), dtype=torch.float16, device="cuda")
    stack.gemm_phase_expert_major(ctx, xd, ids_d, act3, P, E, K, fused_silu_mul=True)
    down_stack.gemm_phase_expert_major(ctx, act3, ids_d, down3, P, E, 1)
    ctx.sync()
    assert torch.equal(act, act3) and torch.equal(down, down3)
    act2 = torch.full((P, I), float("nan"), dtype=torch.float16, device="cuda")
    down2 = torch.full((P, H), float("nan"), dtype=torch.float16, device="cuda")
    stack.gemm_phase_inline_align(ctx, xd, ids_d, act2, P, E, K, P // 16 + E, fused_silu_mul=True)
    down_stack.gemm_phase_inline_align(ctx, act2, ids_d, down2, P, E, 1, P // 16 + E)
    ctx.sync()
    assert torch.equal(act, act2) and torch.equal(down, down2)
    if I >= 256:
        act4 = torch.full((P, I), float("nan"), dtype=torch.float16, device="cuda")
        down4 = torch.full((P, H), float("nan"), dtype=torch.float16, device="cuda")
        if desc_act:        # the down stack's input gather cannot sit inside the one launch: refused, callers run two phases
            with pytest.raises(pkg.backend.Unsupported, match="act-order down stack"):
                stack.gemm_phase_expert_major_pair(ctx, down_stack, xd, ids_d, act4, down4, P, E, K)
        else:
            forms.reset()
            stack.gemm_phase_expert_major_pair(ctx, down_stack, xd, ids_d, act4, down4, P, E, K)
            ctx.sync()
            assert stack.pair_timeouts(ctx) == 0
            assert torch.equal(act, act4) and torch.equal(down, down4)
            forms.require("moe_expert_major_pair")
    assert torch.equal(xd, x_keep)                                         # the gather works on a scratch copy


@pytest.mark.parametrize("tokens,H,E,K", [(1, 2048, 128, 8), (32, 2048, 128, 8), (5, 1024, 64, 4), (3, 4096, 16, 2)])
def test_fused_add_rms_norm_route_equals_op_chain(env, tokens, H, E, K):
    # fused.hip B ≡ fused_add_rms_norm → gemm(router) → route_topk_softmax, each as the oracle defines it
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens + H + E)
    r, x = f16r(rng.standard_normal((tokens, H)) * 2), f16r(rng.standard_normal((tokens, H)))
    w = f16r(1 + 0.1 * rng.standard_normal(H))
    rw = f16r(rng.standard_normal((E, H)) * 0.05)
    rd, nd = dev16(torch, r), torch.empty(tokens, H, dtype=torch.float16, device="cuda")
    ids = torch.empty(tokens, K, dtype=torch.int32, device="cuda")
    wt = torch.empty(tokens, K, dtype=torch.float32, device="cuda")
    lg = torch.empty(tokens, E, dtype=torch.float32, device="cuda")
    B.fused_add_rms_norm_route(ctx, rd, dev16(torch, x), dev16(torch, w), 1e-6, nd,
                               B.dense_repack_f16t(ctx, dev16(torch, rw), E, H), E, K, True, ids, wt, lg, tokens, H)
    ctx.sync()
    r_ref, _ = O.fused_add_rms_norm(r, x, w, 1e-6)
    assert nmse(r_ref, host(rd)) < NMSE_FP16_TOL
    n_ref = O.rms_norm(host(rd), w, 1e-6)                                  # norm of the fp16-rounded residual
    assert nmse(n_ref, host(nd)) < NMSE_FP16_TOL
    logits_ref = O.gemm(host(nd), rw, tokens, E, H)                        # router sees the fp16 norm_out
    assert nmse(logits_ref, lg.cpu().numpy()) < 1e-10
    rid, rwt = O.route_topk(lg.cpu().numpy(), E, K, True)                  # routing of the device logits: bit-exact ids
    assert np.array_equal(ids.cpu().numpy().astype(np.uint32), rid)
    assert np.max(np.abs(wt.cpu().numpy() - rwt)) < 1e-6


@pytest.mark.parametrize("tokens,H,E,K,Q,slabs", [(32, 2048, 128, 8, 4, 0), (1, 2048, 128, 8, 4, 3), (9, 1024, 64, 4, 2, 2),
                                                     (5, 512, 16, 2, 1, 0), (16, 2048, 128, 8, 8, 0)])
def test_route_parts_and_merge_equal_single_kernel_route(env, tokens, H, E, K, Q, slabs):
    """Decode path: router split over Q parts + candidate merge in the gate_up GEMM ≡ route_topk_softmax on the
    same logits (ids bit-exact, weights 1e-6), residual/norm as the op chain, align arrays as moe_align_block_size."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens + H + E + Q)
    r = f16r(rng.standard_normal((tokens, H)) * 2)
    w = f16r(1 + 0.1 * rng.standard_normal(H))
    rw = f16r(rng.standard_normal((E, H)) * 0.05)
    if slabs:
        parts = [rng.standard_normal((tokens, H)).astype(np.float32) * 0.5 for _ in range(slabs)]
        xs = torch.from_numpy(np.stack(parts)).cuda()                      # [S, T, H] fp32
        x = f16r(sum(parts[1:], parts[0].copy()))                          # slab-order fp32 sum, rounded like the fp16 o_proj
        xd = None
    else:
        x = f16r(rng.standard_normal((tokens, H)))
        xs, xd = None, dev16(torch, x)
    rd, r2 = dev16(torch, r), torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
    nd = torch.empty(tokens, H, dtype=torch.float16, device="cuda")
    cand = torch.zeros(tokens * Q * 8 * 2, dtype=torch.int32, device="cuda")
    stats = torch.zeros(tokens * Q * 2, dtype=torch.float32, device="cuda")
    lg = torch.empty(tokens, E, dtype=torch.float32, device="cuda")
    B.fused_add_rms_norm_route_parts(ctx, rd, r2, xd, xs, slabs, tokens * H, H, dev16(torch, w), 1e-6, nd,
                                     B.dense_repack_f16t(ctx, dev16(torch, rw), E, H), E, K, Q, cand, stats, lg, tokens, H)
    ctx.sync()
    assert np.array_equal(host(rd), r)                                     # input residual untouched (ping-pong)
    r_ref, _ = O.fused_add_rms_norm(r, x, w, 1e-6)
    assert nmse(r_ref, host(r2)) < NMSE_FP16_TOL
    assert nmse(O.rms_norm(host(r2), w, 1e-6), host(nd)) < NMSE_FP16_TOL
    logits = lg.cpu().numpy()
    assert nmse(O.gemm(host(nd), rw, tokens, E, H), logits) < 1e-10
    # merge inside a grouped GEMM (tiny expert stack; only the routing outputs are checked here)
    Hs, I = 128, 64
    gu = [O.make_synthetic_gptq(Hs, 2 * I, 128, 300 + e, symmetric=True) for e in range(E)]
    stack = B.load_gptq_stacked([q for q, _, _ in gu], [f16r(s) for _, s, _ in gu], [z for _, _, z in gu], None, 4, 128, Hs, 2 * I)
    P = tokens * K
    sorted_max = P + E * 16
    xin = dev16(torch, rng.standard_normal((tokens, Hs)))
    out = torch.zeros(P, 2 * I, dtype=torch.float16, device="cuda")
    ids = torch.full((P,), -1, dtype=torch.int32, device="cuda")
    wts = torch.zeros(P, dtype=torch.float32, device="cuda")
    sd = torch.full((sorted_max,), P, dtype=torch.int32, device="cuda")
    bd = torch.zeros(sorted_max // 16 + 1, dtype=torch.int32, device="cuda")
    td = torch.zeros(1, dtype=torch.int32, device="cuda")
    stack.gemm_phase_merge_route(ctx, xin, cand, stats, out, tokens, Q, K, True, E, sorted_max // 16, ids, wts, sd, bd, td)
    ctx.sync()
    rid, rwt = O.route_topk(logits, E, K, True)
    assert np.array_equal(ids.cpu().numpy().reshape(tokens, K).astype(np.uint32), rid)
    assert np.max(np.abs(wts.cpu().numpy().reshape(tokens, K) - rwt)) < 1e-6
    rs, rb, rt = O.moe_align_block_size(rid.astype(np.int32), E, 16)
    assert int(td.item()) == rt
    assert np.array_equal(sd.cpu().numpy()[:rt], rs[:rt]) and np.array_equal(bd.cpu().numpy()[:len(rb)], rb)
    out2 = torch.zeros_like(out)
    stack.gemm_phase_inline_align(ctx, xin, ids, out2, P, E, K, sorted_max // 16)
    ctx.sync()
    assert torch.equal(out, out2)


@pytest.mark.parametrize("tokens,H,E,K,Q,slabs", [(32, 2048, 128, 8, 4, 8), (64, 2048, 128, 8, 8, 0), (1, 2048, 128, 8, 2, 3),
                                                     (9, 1024, 64, 4, 2, 2), (5, 512, 16, 2, 1, 0), (33, 2048, 128, 8, 4, 0)])
def test_route_split_in_launch_merge_equals_route_topk(env, tokens, H, E, K, Q, slabs):
    """Split router with the merge done by each token's last-arriving part: ids bit-exact and weights 1e-6 against
    route_topk_softmax on the emitted logits; repeated launches reuse cand/stats/arrive (counter re-arm, stale lines)."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(7 * tokens + H + E + Q)
    w = f16r(1 + 0.1 * rng.standard_normal(H))
    rw = f16r(rng.standard_normal((E, H)) * 0.05)
    rwt = B.dense_repack_f16t(ctx, dev16(torch, rw), E, H)
    cand = torch.zeros(tokens * Q * 8 * 2, dtype=torch.int32, device="cuda")
    stats = torch.zeros(tokens * Q * 2, dtype=torch.float32, device="cuda")
    arrive = torch.zeros(tokens, dtype=torch.int32, device="cuda")
    wd = dev16(torch, w)
    for rep in range(4):
        r = f16r(rng.standard_normal((tokens, H)) * 2)
        if slabs:
            parts = [rng.standard_normal((tokens, H)).astype(np.float32) * 0.5 for _ in range(slabs)]
            xs = torch.from_numpy(np.stack(parts)).cuda()
            x = f16r(sum(parts[1:], parts[0].copy()))
            xd = None
        else:
            x = f16r(rng.standard_normal((tokens, H)))
            xs, xd = None, dev16(torch, x)
        rd, r2 = dev16(torch, r), torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
        nd = torch.empty(tokens, H, dtype=torch.float16, device="cuda")
        lg = torch.empty(tokens, E, dtype=torch.float32, device="cuda")
        ids = torch.full((tokens, K), -1, dtype=torch.int32, device="cuda")
        wts = torch.zeros(tokens, K, dtype=torch.float32, device="cuda")
        B.fused_add_rms_norm_route_split(ctx, rd, r2, xd, xs, slabs, tokens * H, H, wd, 1e-6, nd, rwt, E, K, rep % 2, Q, cand,
                                         stats, arrive, ids, wts, lg, tokens, H)
        ctx.sync()
        assert int(arrive.abs().sum().item()) == 0                         # counters re-armed
        r_ref, _ = O.fused_add_rms_norm(r, x, w, 1e-6)
        assert nmse(r_ref, host(r2)) < NMSE_FP16_TOL
        assert nmse(O.rms_norm(host(r2), w, 1e-6), host(nd)) < NMSE_FP16_TOL
        logits = lg.cpu().numpy()
        assert nmse(O.gemm(host(nd), rw, tokens, E, H), logits) < 1e-10
        rid, rwt_ref = O.route_topk(logits, E, K, bool(rep % 2))
        assert np.array_equal(ids.cpu().numpy().astype(np.uint32), rid), f"rep {rep}"
        assert np.max(np.abs(wts.cpu().numpy() - rwt_ref)) < 1e-6


@pytest.mark.parametrize("sign", ["+", "-"])
@pytest.mark.parametrize("bad", ["one", "some", "all"])
@pytest.mark.parametrize("tokens,H,E,K,Q", [(3, 1024, 128, 8, 4), (9, 512, 64, 4, 2), (2, 512, 16, 2, 1), (5, 512, 128, 8, 1)])
def test_router_logits_that_are_nan_come_last(env, tokens, H, E, K, Q, bad, sign):
    """Every place of a choice is an expert's, each expert once: with NaN among the logits, of either sign, those are behind all numbers in the split router, and make
    all probabilities of the single kernel NaN, which then takes the first experts."""
    pkg, B, ctx, O, torch = env
    gen = torch.Generator("cuda").manual_seed(E + K)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda").half()
    r, x, w, rw = rnd(tokens, H), rnd(tokens, H), rnd(H), rnd(E, H) * 0.05
    which = {"one": [E // 2], "some": list(range(0, E, 3)), "all": slice(None)}[bad]
    rw.view(torch.int16)[which] = 0x7e00 if sign == "+" else 0x7e00 - 0x8000
    rwt = B.dense_repack_f16t(ctx, rw, E, H)
    cand, stats = torch.zeros(tokens * Q * 16, dtype=torch.int32, device="cuda"), torch.zeros(tokens * Q * 2, device="cuda")
    nd, lg, arrive = torch.empty_like(x), torch.empty(tokens, E, device="cuda"), torch.zeros(tokens, dtype=torch.int32, device="cuda")
    ids, wts = (torch.full((2, tokens, K), -1, dtype=t, device="cuda") for t in (torch.int32, torch.float32))
    B.fused_add_rms_norm_route_split(ctx, r, torch.empty_like(r), x, None, 0, 0, H, w, 1e-6, nd, rwt, E, K, 1, Q, cand, stats, arrive, ids[0], wts[0], lg, tokens, H)
    B.fused_add_rms_norm_route(ctx, r.clone(), x, w, 1e-6, nd, rwt, E, K, True, ids[1], wts[1], None, tokens, H)
    ctx.sync()
    assert lg.isnan().sum() == rw.isnan().any(1).sum() * tokens
    order = torch.where(lg.isnan(), -float("inf"), lg).sort(dim=1, descending=True, stable=True).indices[:, :K]
    assert torch.equal(ids[0].long(), order)
    assert torch.equal(ids[1].long(), torch.arange(K, device="cuda").expand(tokens, K))
    lists = cand.reshape(tokens, Q, 8, 2)[:, :, :min(K, E // Q), 1].flatten(1)
    assert all(len(set(row)) == len(row) and max(row) < E for row in lists.tolist())


@pytest.mark.parametrize("tokens,H,K,with_norm", [(1, 2048, 8, True), (32, 2048, 8, True), (7, 1024, 2, False)])
def test_moe_combine_add_rms_norm_equals_op_chain(env, tokens, H, K, with_norm):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens * H + K)
    down = f16r(rng.standard_normal((tokens * K, H)))
    wts = rng.random((tokens, K)).astype(np.float32)
    wts /= wts.sum(axis=1, keepdims=True)
    r = f16r(rng.standard_normal((tokens, H)))
    nw = f16r(1 + 0.1 * rng.standard_normal(H))
    rd, nd = dev16(torch, r), torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
    B.moe_combine_add_rms_norm(ctx, dev16(torch, down), torch.from_numpy(wts).cuda(), rd,
                               dev16(torch, nw) if with_norm else None, 1e-6, nd, tokens, K, H)
    ctx.sync()
    comb = np.zeros((tokens, H), np.float32)
    for b in range(tokens):
        for k in range(K):
            comb[b] += wts[b, k] * down[b * K + k]                         # moe_forward_cpu order (dispatch.rs:2277-2283)
    assert nmse(r + comb, host(rd)) < NMSE_FP16_TOL
    if with_norm:
        assert nmse(O.rms_norm(host(rd), nw, 1e-6), host(nd)) < NMSE_FP16_TOL
    else:
        assert not host(nd).any()


# ── sampling ─────────────────────────────────────────────────────────────────
def test_argmax_rows_first_max_and_mask(env):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(9)
    m, n = 5, 151936
    logits = rng.standard_normal((m, n)).astype(np.float32)
    logits[0, 777] = logits[0, 120000] = 9.0               # tie → first index (traits.rs:1547)
    logits[1, n - 1] = 50.0
    logits[2, 0] = 50.0
    ld = torch.from_numpy(logits).cuda()
    assert np.array_equal(B.argmax_rows_f16(ctx, ld, m, n), O.argmax_rows(logits))
    l16 = f16r(logits)
    assert np.array_equal(B.argmax_rows_f16(ctx, dev16(torch, l16), m, n), O.argmax_rows(l16))
    mask = np.ones(n, np.uint8)
    mask[777] = 0
    mask_len = n - 1                                        # ids ≥ mask_len are invalid
    got = B.argmax_rows_f16_masked(ctx, ld, torch.from_numpy(mask).cuda(), mask_len, m, n)
    masked = logits.copy()
    masked[:, 777] = -np.inf
    masked[:, mask_len:] = -np.inf
    assert np.array_equal(got, O.argmax_rows(masked))
    # single-launch entry point (no workspace) and an all -inf row (→ id 0 on both paths)
    logits[3, :] = -np.inf
    ld = torch.from_numpy(logits).cuda()
    out = torch.empty(m, dtype=torch.int32, device="cuda")
    import ctypes
    assert ctx.lib.ferrum_hip_argmax_rows_f32(ctypes.c_void_p(ld.data_ptr()), ctypes.c_void_p(out.data_ptr()), None, 0, m, n,
                                              ctx.stream) == 0
    ctx.sync()
    ref = O.argmax_rows(logits)
    assert ref[3] == 0
    assert np.array_equal(out.cpu().numpy().astype(np.uint32), ref)
    assert np.array_equal(B.argmax_rows_f16(ctx, ld, m, n), ref)


@pytest.mark.parametrize("n", [4096, 5003, 40000, 40004])
def test_argmax_rows_widths_and_mask_tails(env, n):
    """Row widths on both sides of the vector form's conditions (n % 8, ≥ 4096) with a mask shorter than the row."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(n)
    m = 7
    logits = rng.standard_normal((m, n)).astype(np.float32)
    logits[0, n - 1] = 30.0
    logits[1, n - 3] = logits[1, 5] = 30.0
    logits[2, :] = 1.0                                      # all equal → id 0, or the first valid id under the mask
    ld = torch.from_numpy(logits).cuda()
    assert np.array_equal(B.argmax_rows_f16(ctx, ld, m, n), O.argmax_rows(logits))
    l16 = f16r(logits)
    assert np.array_equal(B.argmax_rows_f16(ctx, dev16(torch, l16), m, n), O.argmax_rows(l16))
    mask = (rng.random(n) < 0.7).astype(np.uint8)
    mask[:3] = 0
    mask_len = n - 5
    got = B.argmax_rows_f16_masked(ctx, ld, torch.from_numpy(mask).cuda(), mask_len, m, n)
    masked = logits.copy()
    masked[:, mask == 0] = -np.inf
    masked[:, mask_len:] = -np.inf
    assert np.array_equal(got, O.argmax_rows(masked))


def test_sparse_repetition_penalty_then_argmax(env):
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(10)
    m, n = 3, 4096
    logits = rng.standard_normal((m, n)).astype(np.float32)
    prev = [np.unique(rng.integers(0, n, size=50)).astype(np.uint32) for _ in range(m)]
    for r in range(m):
        logits[r, prev[r][0]] = 20.0                        # the penalised id was the winner
    offs = np.concatenate([[0], np.cumsum([len(p) for p in prev])]).astype(np.int32)
    pens = np.array([1.1, 1.0, 3.0], np.float32)
    ld = torch.from_numpy(logits.copy()).cuda()
    got = B.argmax_rows_f16_sparse_repetition_penalty(
        ctx, ld, None, torch.from_numpy(offs).cuda(), torch.from_numpy(np.concatenate(prev).astype(np.int32)).cuda(),
        torch.from_numpy(pens).cuda(), int(offs[-1]), m, n)
    ref_logits = np.stack([O.repetition_penalty(logits[r], prev[r], float(pens[r])) for r in range(m)])
    assert np.allclose(ld.cpu().numpy(), ref_logits, rtol=1e-6, atol=0)
    assert np.array_equal(got, O.argmax_rows(ref_logits))


# ── trait-surface entry points of the bucketed MoE path and the single-sequence paged attention ─────────────────
@pytest.mark.parametrize("tokens,ne,k,block", [(1, 128, 8, 16), (32, 128, 8, 16), (700, 128, 8, 64), (5, 8, 2, 16), (257, 60, 4, 32)])
def test_moe_build_pairs_by_token_and_packed_row_align_bit_exact(env, tokens, ne, k, block):
    """moe_build_pairs_by_token (capabilities.rs:410) and the packed-row moe_align_block_size (capabilities.rs:429): the
    device plan must equal MoeBucketPlan::rebuild_into (moe/dispatch.rs:1408-1461, restated in the oracle) bit for bit —
    a STABLE counting sort, where the reference's CUDA kernels leave the order inside an expert to atomicAdd."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens * 131 + ne)
    ids = np.stack([rng.choice(ne, size=k, replace=False) for _ in range(tokens)]).astype(np.uint32)
    P = tokens * k
    off_ref, packed_ref, pairs_ref = O.bucket_plan(ids, tokens, ne, k)
    ids_d = torch.from_numpy(ids.astype(np.int32).reshape(-1).copy()).cuda()
    pairs = torch.full((P,), -7, dtype=torch.int32, device="cuda")
    packed = torch.full((P,), -7, dtype=torch.int32, device="cuda")
    offs = torch.full((ne + 1,), -7, dtype=torch.int32, device="cuda")
    B.moe_build_pairs_by_token(ctx, ids_d, pairs, packed, offs, P, ne, k)
    ctx.sync()
    assert np.array_equal(offs.cpu().numpy(), np.asarray(off_ref, np.int32))
    assert np.array_equal(packed.cpu().numpy(), np.asarray(packed_ref, np.int32))
    assert np.array_equal(pairs.cpu().numpy(), np.asarray(pairs_ref, np.int32))
    # packed-row align: expert e's padded region holds expert_offsets[e] + 0, 1, …; padding and the unused tail hold P
    sorted_max = P + ne * block
    sd = torch.full((sorted_max,), -7, dtype=torch.int32, device="cuda")
    bd = torch.full((sorted_max // block + 1,), -7, dtype=torch.int32, device="cuda")
    td = torch.zeros(1, dtype=torch.int32, device="cuda")
    B.moe_align_block_size(ctx, ids_d, sd, bd, td, P, ne, block, sorted_max)
    ctx.sync()
    exp_sorted, exp_blocks = [], []
    for e in range(ne):
        cnt = int(off_ref[e + 1] - off_ref[e])
        pad = -(-cnt // block) * block
        exp_sorted += [int(off_ref[e]) + i for i in range(cnt)] + [P] * (pad - cnt)
        exp_blocks += [e] * (pad // block)
    assert int(td.item()) == len(exp_sorted)
    got = sd.cpu().numpy()
    assert np.array_equal(got[:len(exp_sorted)], np.asarray(exp_sorted, np.int32)) and np.all(got[len(exp_sorted):] == P)
    assert np.array_equal(bd.cpu().numpy()[:len(exp_blocks)], np.asarray(exp_blocks, np.int32))
    # ids outside [0, E) are skipped: pairs_by_token = −1 (kernels/moe_build_pairs.cu:84-87), the rest unchanged in order
    bad = ids.astype(np.int32).reshape(-1).copy()
    bad[::3] = np.where(np.arange(len(bad[::3])) % 2 == 0, -1, ne + 5)
    pairs.fill_(-7)
    B.moe_build_pairs_by_token(ctx, torch.from_numpy(bad).cuda(), pairs, packed, offs, P, ne, k)
    ctx.sync()
    pr, of = pairs.cpu().numpy(), offs.cpu().numpy()
    valid = (bad >= 0) & (bad < ne)
    assert np.all(pr[~valid] == -1) and of[ne] == valid.sum()
    for e in range(ne):
        rows = pr[valid & (bad == e)]
        assert np.array_equal(rows, np.arange(of[e], of[e + 1]))       # ascending pair id inside an expert


@pytest.mark.parametrize("tokens,K,H", [(1, 8, 2048), (32, 8, 2048), (7, 2, 1024)])
def test_moe_combine_by_pairs_and_weighted_sum_batched(env, tokens, K, H):
    """moe_combine with pairs_by_token (capabilities.rs:684-724: out[b] = Σ_k w[b,k]·packed_down[pairs[b,k]], −1 skipped)
    and weighted_sum_batched[_offset] (capabilities.rs:560-600), against the trait's own default loop in f32."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens + K + H)
    P = tokens * K
    down = f16r(rng.standard_normal((P, H)))
    w = rng.random((tokens, K)).astype(np.float32)
    pairs = rng.permutation(P).astype(np.int32).reshape(tokens, K)
    if tokens > 1:
        pairs[1, 0] = -1
    ref = np.zeros((tokens, H), np.float32)
    for b in range(tokens):
        for k in range(K):
            if pairs[b, k] >= 0:
                ref[b] += w[b, k] * down[pairs[b, k]]
    out = torch.full((tokens, H), 3.0, dtype=torch.float16, device="cuda")
    B.moe_combine_pairs(ctx, dev16(torch, down), torch.from_numpy(pairs.reshape(-1).copy()).cuda(), torch.from_numpy(w.reshape(-1).copy()).cuda(),
                        out, tokens, H, K, P)
    ctx.sync()
    assert nmse(ref, host(out)) < NMSE_FP16_TOL
    # weighted_sum_batched: slots [b, k, h]; the offset form reads weights / writes out at element offsets
    ref2 = np.einsum("bk,bkh->bh", w, down.reshape(tokens, K, H)).astype(np.float32)
    out2 = torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
    B.weighted_sum_batched(ctx, dev16(torch, down), torch.from_numpy(w.reshape(-1).copy()).cuda(), out2, tokens, K, H)
    wbig = torch.zeros(16 + P, dtype=torch.float32, device="cuda")
    wbig[16:] = torch.from_numpy(w.reshape(-1).copy()).cuda()
    obig = torch.full((2 * H + tokens * H,), 5.0, dtype=torch.float16, device="cuda")
    B.weighted_sum_batched_offset(ctx, dev16(torch, down), wbig, 16, obig, 2 * H, tokens, K, H)
    ctx.sync()
    assert nmse(ref2, host(out2)) < NMSE_FP16_TOL
    assert torch.equal(obig[2 * H:].reshape(tokens, H), out2) and bool(torch.all(obig[:2 * H] == 5.0))


@pytest.mark.parametrize("tokens,E,K,H,I", [(9, 8, 2, 256, 128), (40, 16, 4, 512, 256), (300, 8, 2, 256, 128)])
def test_gemm_phase_batched_bucketed_dispatch(env, tokens, E, K, H, I):
    """MarlinExpertStack::gemm_phase_batched (marlin_expert_stack.rs:63): per-expert (m × K)·tile[e] over the expert-bucketed
    packed rows of the host plan — the reference's bucketed MoE path (moe/dispatch.rs:1558-2192): gather → gemm1 → silu·mul →
    gemm3 → moe_combine through pairs_by_token — against moe_forward_cpu."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(tokens + E + H)
    gu = [O.make_synthetic_gptq(H, 2 * I, 128, 300 + e, symmetric=True) for e in range(E)]
    dn = [O.make_synthetic_gptq(I, H, 128, 400 + e, symmetric=True) for e in range(E)]
    gu = [(q, f16r(s / (0.28 * np.sqrt(H))), z) for q, s, z in gu]
    dn = [(q, f16r(s / (0.28 * np.sqrt(I))), z) for q, s, z in dn]
    x = f16r(rng.standard_normal((tokens, H)))
    rid, rw = O.route_topk(rng.standard_normal((tokens, E)).astype(np.float32), E, K, True)
    gw = np.stack([O.dequant_gptq(q, s, z, 128, H, 2 * I) for q, s, z in gu])
    dw = np.stack([O.dequant_gptq(q, s, z, 128, I, H) for q, s, z in dn])
    ref = O.moe_forward_cpu(x, H, I, K, rid, rw, gw, dw)
    P = tokens * K
    off, packed_idx, pairs = O.bucket_plan(rid, tokens, E, K)
    xp = dev16(torch, x[np.asarray(packed_idx)])                 # the gather step (embedding_lookup of x into x_packed)
    disp = [(e, int(off[e]), int(off[e]), int(off[e + 1] - off[e])) for e in range(E)]
    g_stack = B.load_gptq_stacked([q for q, _, _ in gu], [s for _, s, _ in gu], [z for _, _, z in gu], None, 4, 128, H, 2 * I,
                                  fuse_gate_up=True)
    d_stack = B.load_gptq_stacked([q for q, _, _ in dn], [s for _, s, _ in dn], [z for _, _, z in dn], None, 4, 128, I, H)
    act = torch.zeros(P, I, dtype=torch.float16, device="cuda")
    g_stack.gemm_phase_batched(ctx, xp, disp, act, H, fused_silu_mul=True)
    # the down phase writes each expert's rows 3 rows further down (out_row_offset ≠ in_row_offset)
    down = torch.zeros(P + 3, H, dtype=torch.float16, device="cuda")
    d_stack.gemm_phase_batched(ctx, act, [(e, i, o + 3, m) for e, i, o, m in disp], down, I)
    out = torch.zeros(tokens, H, dtype=torch.float16, device="cuda")
    B.moe_combine_pairs(ctx, down[3:], torch.from_numpy(np.asarray(pairs, np.int32)).cuda(), torch.from_numpy(rw.reshape(-1).copy()).cuda(),
                        out, tokens, H, K, P)
    ctx.sync()
    assert bool(torch.all(down[:3] == 0))
    assert nmse(ref, host(out)) < 3e-6


@pytest.mark.parametrize("nq,nkv,hd,q_len,ctx_len", [(8, 2, 128, 1, 300), (8, 2, 128, 37, 37), (32, 4, 128, 70, 200), (4, 4, 64, 20, 33)])
def test_paged_decode_attention_trait_form(env, nq, nkv, hd, q_len, ctx_len):
    """BackendPagedKv::paged_decode_attention (traits.rs:1719-1738): q_len == 1 over several sequences (token-major), and the
    single-sequence causal prefill whose q / out are HEAD-major [nq, q_len, hd] with context_lens[0] the final kv length."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(nq + q_len + ctx_len)
    S = 3 if q_len == 1 else 1
    kv_lens = [ctx_len, 17, 130][:S]
    max_blocks = (max(kv_lens) + 15) // 16 + 1
    num_blocks = sum((n + 15) // 16 for n in kv_lens) + 2
    perm = rng.permutation(num_blocks)
    tables = np.zeros((S, max_blocks), np.int32)
    used, K, V = 0, [], []
    for s, n in enumerate(kv_lens):
        nb = (n + 15) // 16
        tables[s, :nb] = perm[used:used + nb]
        used += nb
        K.append(f16r(rng.standard_normal((n, nkv, hd))))
        V.append(f16r(rng.standard_normal((n, nkv, hd))))
    ck, cv = _fill_pool(env, K, V, tables, kv_lens, nkv, hd, num_blocks)
    lens_d = torch.from_numpy(np.array(kv_lens, np.int32)).cuda()
    if q_len == 1:
        q = f16r(rng.standard_normal((S, nq, hd)))
        out = torch.zeros(S, nq, hd, dtype=torch.float16, device="cuda")
        B.paged_decode_attention(ctx, dev16(torch, q), ck, cv, out, torch.from_numpy(tables).cuda(), lens_d, S, nq, nkv, hd, 16, max_blocks, 1)
        ctx.sync()
        got = host(out)
        for s, n in enumerate(kv_lens):
            assert nmse(_ref_attention(O, q[s:s + 1], K[s], V[s], n - 1, nq, nkv, hd), got[s:s + 1]) < 1e-5, s
    else:
        q_tm = f16r(rng.standard_normal((q_len, nq, hd)))        # token-major for the reference …
        q_hm = np.ascontiguousarray(q_tm.transpose(1, 0, 2))     # … head-major for the call
        out = torch.zeros(nq, q_len, hd, dtype=torch.float16, device="cuda")
        B.paged_decode_attention(ctx, dev16(torch, q_hm), ck, cv, out, torch.from_numpy(tables).cuda(), lens_d, 1, nq, nkv, hd, 16, max_blocks, q_len)
        ctx.sync()
        ref = _ref_attention(O, q_tm, K[0], V[0], ctx_len - q_len, nq, nkv, hd)
        assert nmse(ref, host(out).transpose(1, 0, 2)) < 1e-5


def test_backend_graph_capture_and_replay(env):
    """BackendGraph (capabilities.rs:35-70): ops enqueued between begin / end capture are recorded, not run; every replay
    runs them on the current buffer contents."""
    pkg, B, ctx, O, torch = env
    rng = np.random.default_rng(9)
    x = f16r(rng.standard_normal((5, 1024)))
    w = f16r(1 + 0.1 * rng.standard_normal(1024))
    xd, wd = dev16(torch, x), dev16(torch, w)
    out = torch.zeros(5, 1024, dtype=torch.float16, device="cuda")
    ctx.sync()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        c2 = B.new_context()                                       # capture needs a non-default stream
        B.begin_graph_capture(c2)
        B.rms_norm(c2, xd, wd, 1e-6, out, 5, 1024)
        g = B.end_graph_capture(c2)
        c2.sync()
        assert float(out.abs().max()) == 0.0                       # recorded, not executed
        B.replay_graph(c2, g)
        c2.sync()
        assert nmse(O.rms_norm(x, w, 1e-6), host(out)) < NMSE_FP16_TOL
        x2 = f16r(rng.standard_normal((5, 1024)))
        xd.copy_(dev16(torch, x2))
        c2.sync()
        B.replay_graph(c2, g)
        c2.sync()
        assert nmse(O.rms_norm(x2, w, 1e-6), host(out)) < NMSE_FP16_TOL
        B.reset_graph(c2, g)

"""GPU parity: the MFMA flash-attention kernel (tsa_attn_fwd) and its VALU opponent
(tsa_attn_fwd_valu) against the CPU oracle.

Gate: max-abs error < 0.02 on fp16 outputs (the reference's gate, src/attn_sm75.cu:501-502);
a tighter 5e-3 bound guards against regressions that the gate would still let through.
Cases: the float64 fixtures, B=1 H=4 S=256 D=128 non-causal, B=2 H=8 S=512 causal at D=64 and
128, B=1 H=32 S=8192 D=128 causal with outliers (against a seeded sample of oracle rows plus
the full on-device naive kernel), the reference's own inputs
(mt19937(42), N(0, 0.5), src/attn_sm75.cu:398,473-476), ragged S, and size-independent
properties at full size (row 0 of a causal head is V[0] exactly).  The VALU kernel runs the
fixtures, the first two shapes at every D, ragged S and the reference's inputs.
"""
import numpy as np
import pytest

import tsa

pytestmark = pytest.mark.gpu
GATE = 2e-2
TIGHT = 5e-3


def _to_dev(dev, *arrays):
    import torch
    return [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in arrays]


def _run(dev, q, k, v, causal, naive=False, valu=False):
    import torch
    tq, tk, tv = _to_dev(dev, q, k, v)
    o = tsa.attn_fwd(tq, tk, tv, causal=causal, naive=naive, valu=valu)
    torch.cuda.synchronize()
    return o.cpu().numpy()


def _err(a, b):
    return float(np.abs(a.astype(np.float64) - b.astype(np.float64)).max())


def _normal(rng, shape, std=1.0):
    return (std * rng.standard_normal(shape)).astype(np.float16)


@pytest.mark.parametrize("i", range(4))
def test_golden_fixtures(dev, golden, i):
    g = golden("attn_golden.npz")
    B, H, S, D, causal = (int(x) for x in g[f"c{i}_meta"])
    o = _run(dev, g[f"c{i}_q"], g[f"c{i}_k"], g[f"c{i}_v"], bool(causal))
    assert _err(o, g[f"c{i}_o"]) < TIGHT


def test_b1_h4_s256_d128_noncausal(dev, orc):
    rng = np.random.default_rng(101)
    q, k, v = (_normal(rng, (1, 4, 256, 128)) for _ in range(3))
    e = _err(_run(dev, q, k, v, False), orc.attn_naive(q, k, v, False))
    print(f"B=1 H=4 S=256 D=128 non-causal max-abs {e:.5f}")
    assert e < TIGHT


@pytest.mark.parametrize("D", [64, 128])
def test_b2_h8_s512_causal(dev, orc, D):
    rng = np.random.default_rng(102 + D)
    q, k, v = (_normal(rng, (2, 8, 512, D)) for _ in range(3))
    e = _err(_run(dev, q, k, v, True), orc.attn_naive(q, k, v, True))
    print(f"B=2 H=8 S=512 D={D} causal max-abs {e:.5f}")
    assert e < TIGHT


@pytest.mark.parametrize("shape", [(1, 4, 256, 128), (2, 8, 512, 128), (2, 8, 512, 64)])
def test_reference_driver_inputs(dev, orc, shape):
    n = int(np.prod(shape))
    qkv = orc.mt_normal_half(42, 0.0, 0.5, n, 3).view(np.float16).reshape((3,) + shape)
    q, k, v = qkv[0], qkv[1], qkv[2]
    o = _run(dev, q, k, v, True)
    e = _err(o, orc.attn_naive(q, k, v, True))
    print(f"reference inputs {shape} max-abs {e:.5f}")
    assert e < TIGHT
    # the same-binary naive kernel agrees with the oracle too
    assert _err(_run(dev, q, k, v, True, naive=True), orc.attn_naive(q, k, v, True)) < 2e-3


@pytest.mark.parametrize("S", [1, 2, 63, 64, 65, 127, 129, 200, 300])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_ragged_lengths(dev, orc, S, D, causal):
    rng = np.random.default_rng(S * 7 + D + causal)
    q, k, v = (_normal(rng, (1, 3, S, D)) for _ in range(3))
    assert _err(_run(dev, q, k, v, causal), orc.attn_naive(q, k, v, causal)) < TIGHT


def test_b1_h32_s8192_d128_causal_outliers(dev, orc):
    """B=1 H=32 S=8192 D=128 causal, N(0, 0.5) with 1% of entries x8."""
    import torch
    rng = np.random.default_rng(103)
    shape = (1, 32, 8192, 128)

    def gen():
        x = 0.5 * rng.standard_normal(shape, dtype=np.float32)
        x[rng.random(shape) < 0.01] *= 8
        return x.astype(np.float16)

    q, k, v = gen(), gen(), gen()
    tq, tk, tv = _to_dev(dev, q, k, v)
    o = tsa.attn_fwd(tq, tk, tv, causal=True)
    on = tsa.attn_fwd(tq, tk, tv, causal=True, naive=True)
    torch.cuda.synchronize()
    o_np = o.cpu().numpy()
    # full output against the on-device naive kernel (independent fp32 two-pass softmax)
    e_naive = float((o.float() - on.float()).abs().max())
    # seeded sample of rows against the CPU oracle, including first/last rows of heads
    S = shape[2]
    rows = np.concatenate([rng.integers(0, 32 * S, 320), [0, S - 1, 5 * S, 31 * S + S - 1, 17 * S + 4095]])
    rows, _, o16 = orc.attn_rows(q, k, v, np.unique(rows), True)
    e_orc = _err(o_np.reshape(-1, 128)[rows], o16)
    print(f"B=1 H=32 S=8192 D=128 causal max-abs vs naive kernel {e_naive:.5f}, vs oracle rows {e_orc:.5f}")
    assert e_orc < GATE and e_naive < GATE
    assert e_orc < TIGHT
    # size-independent property: a causal row 0 attends only to key 0, so O[0] = V[0]
    assert np.array_equal(o_np[0, :, 0].view(np.uint16), v[0, :, 0].view(np.uint16))


def test_constant_values_full_size(dev):
    import torch
    rng = np.random.default_rng(104)
    q, k = (_normal(rng, (1, 8, 4096, 128)) for _ in range(2))
    row = _normal(rng, (1, 8, 1, 128))
    v = np.broadcast_to(row, (1, 8, 4096, 128)).copy()
    for causal in (False, True):
        o = _run(dev, q, k, v, causal)
        assert _err(o, v) < 2e-3
    torch.cuda.synchronize()


def test_stream_argument(dev, orc):
    import torch
    rng = np.random.default_rng(105)
    q, k, v = (_normal(rng, (1, 2, 130, 64)) for _ in range(3))
    tq, tk, tv = _to_dev(dev, q, k, v)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        o = tsa.attn_fwd(tq, tk, tv, causal=True, stream=s)
    s.synchronize()
    assert _err(o.cpu().numpy(), orc.attn_naive(q, k, v, True)) < TIGHT


# ---- D = 256 and gated grouped-query attention (tsa_attn_gqa_fwd) ----
def _run_gqa(dev, q, k, v, gate, causal, naive=False):
    import torch
    tq, tk, tv = _to_dev(dev, q, k, v)
    tg = _to_dev(dev, gate)[0] if gate is not None else None
    o = tsa.attn_gqa_fwd(tq, tk, tv, tg, causal=causal, naive=naive)
    torch.cuda.synchronize()
    return o.cpu().numpy()


@pytest.mark.parametrize("S", [1, 64, 130, 300])
@pytest.mark.parametrize("causal", [False, True])
def test_d256(dev, orc, S, causal):
    rng = np.random.default_rng(800 + S + causal)
    q, k, v = (_normal(rng, (1, 2, S, 256)) for _ in range(3))
    e = _err(_run(dev, q, k, v, causal), orc.attn_naive(q, k, v, causal))
    print(f"D=256 S={S} causal={causal} max-abs {e:.5f}")
    assert e < TIGHT


@pytest.mark.parametrize("B,Hq,Hkv,S,D,causal", [(1, 24, 4, 200, 256, True), (2, 6, 2, 129, 128, False),
                                                (1, 4, 1, 65, 64, True), (1, 8, 8, 100, 128, True)])
def test_gated_gqa(dev, orc, B, Hq, Hkv, S, D, causal):
    rng = np.random.default_rng(810 + Hq + D + S)
    q = _normal(rng, (B, Hq, S, D))
    k, v = _normal(rng, (B, Hkv, S, D)), _normal(rng, (B, Hkv, S, D))
    gate = _normal(rng, (B, Hq, S, D), 2.0)
    o = _run_gqa(dev, q, k, v, gate, causal)
    rows, ref = orc.attn_gqa_rows(q, k, v, gate, np.arange(B * Hq * S), causal)
    e = _err(o.reshape(-1, D)[rows], ref)
    en = _err(_run_gqa(dev, q, k, v, gate, causal, naive=True).reshape(-1, D)[rows], ref)
    print(f"gated GQA {B}x{Hq}/{Hkv} S={S} D={D} max-abs {e:.5f} (naive kernel {en:.5f})")
    assert e < TIGHT and en < 2e-3


def test_gqa_without_gate_equals_attn_fwd(dev):
    # Hkv = Hq and no gate is tsa_attn_fwd: the same kernel, bit-identical output
    rng = np.random.default_rng(820)
    q, k, v = (_normal(rng, (1, 4, 257, 128)) for _ in range(3))
    o1 = _run(dev, q, k, v, True)
    o2 = _run_gqa(dev, q, k, v, None, True)
    assert np.array_equal(o1.view(np.uint16), o2.view(np.uint16))


def test_gated_gqa_target_layer(dev, orc):
    """The target model's gated attention layer at an 8K prefill: B=1, 24 query / 4 K/V
    heads, D=256, causal, N(0, 0.5) inputs, gate N(0, 1); a seeded sample of rows against
    the oracle and the full output against the on-device naive kernel."""
    import torch
    rng = np.random.default_rng(830)
    B, Hq, Hkv, S, D = 1, 24, 4, 8192, 256
    q = _normal(rng, (B, Hq, S, D), 0.5)
    k, v = _normal(rng, (B, Hkv, S, D), 0.5), _normal(rng, (B, Hkv, S, D), 0.5)
    gate = _normal(rng, (B, Hq, S, D))
    tq, tk, tv, tg = _to_dev(dev, q, k, v, gate)
    o = tsa.attn_gqa_fwd(tq, tk, tv, tg, causal=True)
    on = tsa.attn_gqa_fwd(tq, tk, tv, tg, causal=True, naive=True)
    torch.cuda.synchronize()
    e_naive = float((o.float() - on.float()).abs().max())
    rows = np.unique(np.concatenate([rng.integers(0, Hq * S, 96), [0, S - 1, 7 * S, 23 * S + S - 1]]))
    rows, ref = orc.attn_gqa_rows(q, k, v, gate, rows, True)
    e_orc = _err(o.cpu().numpy().reshape(-1, D)[rows], ref)
    print(f"gated GQA 24/4 D=256 S=8192: max-abs vs naive kernel {e_naive:.5f}, vs oracle rows {e_orc:.5f}")
    assert e_orc < TIGHT and e_naive < GATE


# ---- the VALU opponent (no MFMA): same recurrence, fp32 FMA dots ----
@pytest.mark.parametrize("i", range(4))
def test_valu_golden_fixtures(dev, golden, i):
    g = golden("attn_golden.npz")
    B, H, S, D, causal = (int(x) for x in g[f"c{i}_meta"])
    o = _run(dev, g[f"c{i}_q"], g[f"c{i}_k"], g[f"c{i}_v"], bool(causal), valu=True)
    assert _err(o, g[f"c{i}_o"]) < TIGHT


@pytest.mark.parametrize("shape,causal", [((1, 4, 256, 128), False), ((2, 8, 512, 64), True),
                                          ((2, 8, 512, 128), True), ((1, 2, 300, 256), True),
                                          ((1, 2, 200, 256), False)])
def test_valu_shapes(dev, orc, shape, causal):
    rng = np.random.default_rng(150 + shape[2] + shape[3])
    q, k, v = (_normal(rng, shape) for _ in range(3))
    ref = orc.attn_naive(q, k, v, causal)
    ev = _err(_run(dev, q, k, v, causal, valu=True), ref)
    em = _err(_run(dev, q, k, v, causal), ref)
    print(f"{shape} causal={causal}: valu max-abs {ev:.5f}, mfma {em:.5f}")
    assert ev < TIGHT


@pytest.mark.parametrize("S", [1, 2, 63, 64, 65, 129])
@pytest.mark.parametrize("causal", [False, True])
def test_valu_ragged(dev, orc, S, causal):
    rng = np.random.default_rng(170 + S)
    q, k, v = (_normal(rng, (1, 3, S, 64)) for _ in range(3))
    assert _err(_run(dev, q, k, v, causal, valu=True), orc.attn_naive(q, k, v, causal)) < TIGHT


def test_valu_reference_driver_inputs(dev, orc):
    # the reference's own inputs: mt19937(42), N(0, 0.5) -> fp16 for Q, K, V in that order
    shape = (2, 8, 512, 128)
    n = int(np.prod(shape))
    qkv = orc.mt_normal_half(42, 0.0, 0.5, n, 3).view(np.float16).reshape((3,) + shape)
    q, k, v = qkv[0], qkv[1], qkv[2]
    assert _err(_run(dev, q, k, v, True, valu=True), orc.attn_naive(q, k, v, True)) < TIGHT


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,S,D", [
    # D <= 128: 32-row query tiles around the lines of the split-key forms
    (1, 1, 1, 1, 64), (1, 4, 4, 33, 64), (1, 16, 16, 1024, 64), (1, 16, 16, 1025, 64), (1, 32, 32, 2048, 64),
    (1, 1, 1, 31, 128), (1, 8, 8, 1024, 128), (1, 8, 2, 1025, 128), (1, 16, 16, 3584, 128), (1, 16, 8, 3585, 128),
    # around the one-per-CU and two-per-CU counts of whole tiles
    (1, 16, 16, 3900, 128), (1, 40, 40, 1500, 128),
    # D = 256: 128-row tiles from S = 129, and both sides of the count of 256-row ones
    (1, 6, 1, 128, 256), (1, 6, 1, 129, 256), (1, 24, 4, 2048, 256), (1, 24, 4, 2049, 256), (1, 8, 4, 4097, 256), (1, 40, 8, 2000, 256),
    (1, 40, 8, 2049, 256)])
def test_split_keys_dispatch(dev, B, Hq, Hkv, S, D, causal):
    """Every form of the forward around the sizes where the dispatch changes, with odd lengths,
    grouped heads and the gate, every row against the on-device naive kernel (fp32 dots, exact
    two-pass softmax).  fp16 P and O: 2^-11 relative each against |O| <= ~2 here, 2e-3 absolute."""
    import torch
    g = torch.Generator(device=dev).manual_seed(S * 7 + D)
    mk = lambda h: torch.randn(B, h, S, D, device=dev, generator=g).half()
    q, k, v, gate = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    o = tsa.attn_gqa_fwd(q, k, v, gate, causal=causal).float()
    ref = tsa.attn_gqa_fwd(q, k, v, gate, causal=causal, naive=True).float()
    torch.cuda.synchronize()
    err = float((o - ref).abs().max())
    print(f"B={B} {Hq}/{Hkv} S={S} D={D} causal={causal}: max-abs {err:.2e}")
    assert torch.isfinite(o).all() and err < 2e-3 * max(1.0, float(ref.abs().max()))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,S,D", [
    # D <= 128: lengths at one key tile and around the lengths where the forms change, tiles on
    # both sides of their rounds with and without a mask
    (1, 6, 2, 64, 64), (1, 6, 2, 65, 64), (1, 40, 8, 191, 64), (1, 40, 8, 192, 64), (1, 64, 8, 511, 64), (1, 64, 8, 512, 64),
    (2, 8, 8, 512, 64), (1, 66, 6, 1024, 64), (1, 3, 1, 64, 128), (1, 3, 1, 65, 128), (1, 16, 4, 511, 128), (1, 16, 4, 512, 128),
    (1, 25, 5, 767, 128), (1, 25, 5, 768, 128), (1, 49, 7, 1000, 128),
    # D = 256: short queries over one round of half tiles, ragged and even last tiles
    (1, 96, 16, 300, 256), (1, 80, 8, 448, 256), (1, 80, 8, 449, 256), (1, 64, 8, 768, 256), (1, 64, 8, 769, 256),
    (1, 104, 8, 512, 256), (1, 48, 4, 1100, 256), (1, 70, 7, 700, 256)])
def test_split_keys_lines(dev, B, Hq, Hkv, S, D, causal):
    """Sizes on both sides of the lines by length and mask, checked as test_split_keys_dispatch
    checks its own; a call repeated gives the same values bit for bit."""
    import torch
    test_split_keys_dispatch(dev, B, Hq, Hkv, S, D, causal)
    g = torch.Generator(device=dev).manual_seed(S + D)
    q, k, v = (torch.randn(B, h, S, D, device=dev, generator=g).half() for h in (Hq, Hkv, Hkv))
    o = tsa.attn_gqa_fwd(q, k, v, causal=causal)
    assert all(torch.equal(tsa.attn_gqa_fwd(q, k, v, causal=causal), o) for _ in range(4))

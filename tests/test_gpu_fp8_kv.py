"""GPU parity with KV caches held as fp8 (OCP e4m3, one fp32 scale per tensor), through the C ABI against the
CPU oracle: the appended rows are fp8(k / k_scale), fp8(v / v_scale) and attention sees scale * fp8 for every
key.  The reference has no fp8 cache; the oracle's definition (torch.float8_e4m3fn casts) is the bar.

Tolerances: fp16 outputs rtol = atol = 1e-2, fp32 scores 1e-3.  The appended fp8 codes are compared exactly; a
code may differ by one step where the projection's fp16 rounding (kernel: fp32 accumulation in a different
order) lands on the other side of an fp8 rounding boundary - at most 1 % of the entries."""
import math

import pytest
import torch

import oracle
from gpu_util import projection_parts, scratch_for
from test_gpu_attention import assert_scores
from trinity_amd import ext
from util import assert_close, attn_inputs, proj_std

pytestmark = pytest.mark.gpu
F8 = torch.float8_e4m3fn
K_SCALE, V_SCALE = 0.04, 0.015


def _fp8_inputs(S, N, Hq, Hkv, D, P, dtype=torch.float16):
    t = attn_inputs(S, N, Hq, Hkv, D, P=P, w_std=proj_std(N), with_cache=True)
    t = {k: (v.to(dtype) if v.dtype == torch.float16 else v) for k, v in t.items()}
    kc = (t["k_cache"].float() / K_SCALE).clamp(-448, 448).to(F8)
    vc = (t["v_cache"].float() / V_SCALE).clamp(-448, 448).to(F8)
    kc[:, P:] = torch.zeros_like(kc[:, P:])
    vc[:, P:] = torch.zeros_like(vc[:, P:])
    t["k_cache"], t["v_cache"] = kc, vc
    return t


def _codes_match(got, want, what):
    g, w = got.view(torch.uint8).int(), want.view(torch.uint8).int()
    diff = (g - w).abs()
    frac = (diff != 0).float().mean().item()
    assert frac <= 0.01, "%s: %.3f %% of the fp8 codes differ" % (what, 100 * frac)
    one_step = (diff <= 1) | (((g & 0x7F) + (w & 0x7F)) <= 1)  # neighbours, or +-0 against the smallest value
    assert bool(one_step.all()), what + ": a code differs by more than one step"


def _run(t, dev, variant, *, Hq, Hkv, D, P, causal, qknorm=False, seed=0, tau=1.0, dtype=torch.float16):
    S, N = t["x"].shape
    p = ext.attn_params(Hq, Hkv, D, S, kv_prefix=P, causal=causal, qknorm=qknorm, rms_eps=1e-5, tau=tau,
                        noise_seed=seed, kv_fp8=True, k_scale=K_SCALE, v_scale=V_SCALE)
    d = {k: v.to(dev) for k, v in t.items()}
    out = torch.zeros(S, Hq * D, dtype=dtype, device=dev)
    scratch = scratch_for(p, N, dev)
    res = {}
    if variant == "vanilla":
        ext.qkv_attention(d["x"], None, d["wq"], d["wk"], d["wv"], d["k_cache"], d["v_cache"], scratch, None, out, p)
    elif variant == "roco":
        s1 = torch.zeros(Hq, P + S, dtype=torch.float32, device=dev)
        s2 = torch.zeros(Hq, P + S, dtype=torch.float32, device=dev)
        ext.roco(d["x"], None, d["wq"], d["wk"], d["wv"], d["k_cache"], d["v_cache"], scratch, out, s1, s2, p)
        res["s1"], res["s2"] = s1.cpu(), s2.cpu()
    else:
        score = torch.zeros(Hq, P + S, dtype=torch.float32, device=dev)
        ext.keyformer(d["x"], None, d["wq"], d["wk"], d["wv"], d["k_cache"], d["v_cache"], scratch, None, out, score, p)
        res["score"] = score.cpu()
    torch.cuda.synchronize()
    res["O2"] = out.cpu()
    res["k_cache"], res["v_cache"] = d["k_cache"].cpu(), d["v_cache"].cpu()
    return res


CASES = [
    # S,  N,   Hq, Hkv, D,  P,   causal
    (16, 256, 4, 2, 128, 1024, False),   # the reference's regime: the kernel reads the fp8 rows itself
    (32, 256, 2, 2, 64, 500, True),
    (5, 128, 2, 1, 64, 253, True),       # ragged
    (1, 128, 4, 4, 128, 0, True),        # nothing cached yet
    (100, 256, 4, 2, 128, 60, True),     # more tokens: through the 16-bit copy
    (200, 320, 5, 1, 64, 0, True),
    (16, 128, 4, 2, 128, 4200, True),    # long prefix: the looping key-split kernel converts the fp8 tiles itself
    (20, 128, 6, 1, 64, 3001, False),    # ... 120 stacked rows, ragged last tile
    (33, 128, 4, 4, 128, 2100, True),    # ... chunks: 33 rows of a head, two waves a tile
    (40, 128, 4, 2, 128, 9000, True),    # ... 80 rows, four waves on single tiles: 36 runs of up to four
    (200, 128, 2, 1, 64, 3001, True),    # ... four row blocks, the last one ragged
    (130, 128, 4, 1, 128, 2500, False),
    (33, 128, 2, 1, 64, 2014, True),     # ... one key short of the key-split kernel: through the 16-bit copy
    (64, 64, 32, 8, 128, 7209, True),    # ... chunks in long runs: eight waves on pairs of tiles, two row blocks
    (100, 64, 32, 8, 128, 3650, False),  # ... four row blocks, the last of 16 rows, a ragged last tile
    (100, 64, 32, 8, 64, 3650, True),
]
# models so wide that the projection runs in parts: their merge converts and appends the new rows
PARTS = [
    (16, 4096, 4, 2, 128, 300, True),
    (3, 4544, 6, 1, 64, 70, False),
    (1, 4096, 4, 4, 128, 0, True),
    (16, 4096, 4, 2, 128, 4200, True),   # ... in front of the looping key-split kernel
    (40, 4096, 2, 2, 128, 70, True),     # ... and of the 16-bit copy
    (200, 4544, 5, 1, 64, 33, True),
]


@pytest.mark.parametrize("S,N,Hq,Hkv,D,P,causal", CASES + PARTS)
@pytest.mark.parametrize("qknorm", [False, True])
def test_fp8_cache_vanilla(dev, S, N, Hq, Hkv, D, P, causal, qknorm):
    if N > 320:
        assert projection_parts(N, S, Hq, Hkv, D, P, qknorm=qknorm, kv_fp8=True, k_scale=K_SCALE, v_scale=V_SCALE) > 1
    t = _fp8_inputs(S, N, Hq, Hkv, D, P)
    kw = dict(n_q_heads=Hq, n_kv_heads=Hkv, head_dim=D, scale=1 / math.sqrt(D), causal=causal, kv_prefix=P,
              k_cache=t["k_cache"], v_cache=t["v_cache"], kv_fp8=True, k_scale=K_SCALE, v_scale=V_SCALE)
    want = oracle.qkv_attention(t["x"], t["wq"], t["wk"], t["wv"], qknorm=qknorm, rms_eps=1e-5, **kw)
    got = _run(t, dev, "vanilla", Hq=Hq, Hkv=Hkv, D=D, P=P, causal=causal, qknorm=qknorm)
    _codes_match(got["k_cache"][:, P:P + S], want["k_new"], "appended k")
    _codes_match(got["v_cache"][:, P:P + S], want["v_new"], "appended v")
    assert torch.equal(got["k_cache"][:, :P].view(torch.uint8), t["k_cache"][:, :P].view(torch.uint8))
    assert torch.equal(got["v_cache"][:, :P].view(torch.uint8), t["v_cache"][:, :P].view(torch.uint8))
    assert_close(got["O2"], want["O2"], 1e-2, 1e-2, "O2")


@pytest.mark.parametrize("S,N,Hq,Hkv,D,P,causal", [CASES[0], CASES[2], CASES[4], CASES[6], PARTS[0], PARTS[5]])
def test_fp8_cache_scores(dev, S, N, Hq, Hkv, D, P, causal):
    t = _fp8_inputs(S, N, Hq, Hkv, D, P)
    kw = dict(n_q_heads=Hq, n_kv_heads=Hkv, head_dim=D, scale=1 / math.sqrt(D), causal=causal, kv_prefix=P,
              k_cache=t["k_cache"], v_cache=t["v_cache"], kv_fp8=True, k_scale=K_SCALE, v_scale=V_SCALE)
    # the fp32 score accumulators are held to 1e-3, finer than one flipped fp8 code allows: the appended rows are
    # checked on their own and the attention part against the cache contents the library produced
    got = _run(t, dev, "roco", Hq=Hq, Hkv=Hkv, D=D, P=P, causal=causal)
    rows = (got["k_cache"][:, P:P + S], got["v_cache"][:, P:P + S])
    want = oracle.qkv_attention(t["x"], t["wq"], t["wk"], t["wv"], roco=True, appended_fp8=rows, **kw)
    _codes_match(rows[0], want["k_new"], "appended k")
    _codes_match(rows[1], want["v_new"], "appended v")
    assert_close(got["O2"], want["O2"], 1e-2, 1e-2, "roco O2")
    assert_scores(got["s1"], want["s1"], "s1")
    assert_scores(got["s2"], want["s2"], "s2")
    got = _run(t, dev, "keyformer", Hq=Hq, Hkv=Hkv, D=D, P=P, causal=causal, seed=9)
    rows = (got["k_cache"][:, P:P + S], got["v_cache"][:, P:P + S])
    want = oracle.qkv_attention(t["x"], t["wq"], t["wk"], t["wv"], keyformer=True, noise_seed=9, tau=1.0,
                                appended_fp8=rows, **kw)
    assert_close(got["O2"], want["O2"], 1e-2, 1e-2, "keyformer O2")
    assert_scores(got["score"], want["score"], "score")


@pytest.mark.parametrize("N", [256, 4096])
def test_fp8_cache_bf16_elements(dev, N):
    S, Hq, Hkv, D, P = 16, 4, 2, 128, 300
    t = _fp8_inputs(S, N, Hq, Hkv, D, P, dtype=torch.bfloat16)
    want = oracle.qkv_attention(t["x"], t["wq"], t["wk"], t["wv"], n_q_heads=Hq, n_kv_heads=Hkv, head_dim=D,
                                scale=1 / math.sqrt(D), causal=False, kv_prefix=P, k_cache=t["k_cache"],
                                v_cache=t["v_cache"], kv_fp8=True, k_scale=K_SCALE, v_scale=V_SCALE,
                                elem=torch.bfloat16)
    got = _run(t, dev, "vanilla", Hq=Hq, Hkv=Hkv, D=D, P=P, causal=False, dtype=torch.bfloat16)
    assert_close(got["O2"], want["O2"], 3e-2, 3e-2, "O2 (bf16 elements)")
    _codes_match(got["k_cache"][:, P:P + S], want["k_new"], "appended k")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("group,S,P", [(1, 1, 300), (1, 1, 2100), (2, 16, 4100), (1, 32, 2500), (40, 2, 2300)])
def test_every_code_is_converted_exactly(dev, dtype, D, group, S, P):
    """Zero activations make all weights equal, and every key holds the same codes, all finite ones among its columns: an
    output is its column's value (or the average of P of them and the new rows' zeros), rounded once."""
    Hkv, N = 256 // D, 256  # a column for every code
    Hq = group * Hkv
    codes = torch.arange(Hkv * D, dtype=torch.int32) % 256
    codes[(codes & 0x7F) == 0x7F] = 0  # NaN
    vrow = codes.to(torch.uint8).view(F8).reshape(Hkv, 1, D)
    vc = vrow.view(torch.uint8).repeat(1, P + S, 1).view(F8).contiguous().to(dev)
    kc = torch.zeros(Hkv, P + S, D, dtype=torch.uint8).view(F8).to(dev)
    x = torch.zeros(S, N, dtype=dtype, device=dev)
    w = lambda h: torch.zeros(N, h * D, dtype=dtype, device=dev)
    p = ext.attn_params(Hq, Hkv, D, S, kv_prefix=P, causal=True, rms_eps=1e-5, kv_fp8=True, k_scale=1.0, v_scale=1.0)
    out = torch.zeros(S, Hq * D, dtype=dtype, device=dev)
    ext.qkv_attention(x, None, w(Hq), w(Hkv), w(Hkv), kc, vc, scratch_for(p, N, dev), None, out, p)
    visible = (P + 1 + torch.arange(S, dtype=torch.float64)).reshape(S, 1, 1)
    want = (vrow.float().double().reshape(1, Hkv, 1, D) * (P / visible).reshape(S, 1, 1, 1)).expand(S, Hkv, Hq // Hkv, D).reshape(S, Hq * D)
    # one rounding to the element type, and fp32 sums of at most P + S equal terms: 1e-5 is above both sums' error
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert_close(out.cpu().double(), want, rtol=eps + 1e-5, atol=0.0)


@pytest.mark.parametrize("S,D", [(16, 128), (1, 128), (3, 64)])
@pytest.mark.parametrize("P", [2048, 2200, 2331, 2600, 3100])
def test_odd_and_even_numbers_of_tile_steps(dev, S, D, P):
    """Runs of two to seven tiles, some a tile shorter than others: tiles of even and odd steps travel in registers of their own."""
    Hq, Hkv = 64, 16  # (512 workgroups over 16 KV heads: up to 32 runs of two tiles for one token, of four for more)
    t = _fp8_inputs(S, 256, Hq, Hkv, D, P)
    want = oracle.qkv_attention(t["x"], t["wq"], t["wk"], t["wv"], n_q_heads=Hq, n_kv_heads=Hkv, head_dim=D, scale=1 / math.sqrt(D),
                                causal=True, kv_prefix=P, k_cache=t["k_cache"], v_cache=t["v_cache"], kv_fp8=True,
                                k_scale=K_SCALE, v_scale=V_SCALE)
    got = _run(t, dev, "vanilla", Hq=Hq, Hkv=Hkv, D=D, P=P, causal=True)
    assert_close(got["O2"], want["O2"], 1e-2, 1e-2, "O2")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("group,S,P", [(1, 1, 300), (1, 1, 2100), (40, 2, 2300), (1, 40, 200)])
def test_a_nan_code_stays_nan(dev, dtype, D, group, S, P):
    """Both NaN codes in one row of V: their columns are NaN for every token, all others are the average of ones."""
    Hkv, N = 2, 256
    Hq = group * Hkv
    vc = torch.ones(Hkv, P + S, D).to(F8)
    vc.view(torch.uint8)[0, P // 2, 3], vc.view(torch.uint8)[0, P // 2, D - 1] = 0x7F, 0xFF
    kc = torch.zeros(Hkv, P + S, D).to(F8).to(dev)
    w = lambda h: torch.zeros(N, h * D, dtype=dtype, device=dev)
    p = ext.attn_params(Hq, Hkv, D, S, kv_prefix=P, causal=True, rms_eps=1e-5, kv_fp8=True, k_scale=1.0, v_scale=1.0)
    out = torch.zeros(S, Hq * D, dtype=dtype, device=dev)
    ext.qkv_attention(torch.zeros(S, N, dtype=dtype, device=dev), None, w(Hq), w(Hkv), w(Hkv), kc, vc.to(dev), scratch_for(p, N, dev), None, out, p)
    got = out.cpu().float().view(S, Hkv, group, D)
    bad = torch.zeros(Hkv, D, dtype=torch.bool)
    bad[0, 3] = bad[0, D - 1] = True
    assert torch.equal(got.isnan(), bad.view(1, Hkv, 1, D).expand_as(got))
    want = (P / (P + 1.0 + torch.arange(S))).view(S, 1, 1, 1).expand_as(got)
    ok = ~got.isnan()
    # (one rounding to the element type, and fp32 sums of at most P + S equal terms)
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert ((got - want)[ok].abs() <= (eps + 1e-5) * want[ok]).all()

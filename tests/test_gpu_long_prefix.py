"""Few and middling tokens against a long cached prefix at the sizes where the split of the key axis and the merge of
its parts can go wrong, against the CPU oracle.

Tolerance: both sides hold q, k, v and the output in fp16 and sum in fp32; the kernels also round the probabilities to
fp16.  With values of order one that is a few 2^-11 of the sum of |p v| <= 4 in O2 (2^-7 allowed), and in the
log-sum-exp the rounding of q and k in a dot product of D terms, 2^-11 * sqrt(D) * scale (2e-3 allowed)."""
import math

import pytest

import oracle
from gpu_util import run_qkv
from test_gpu_fp8_kv import K_SCALE, V_SCALE, _fp8_inputs, _run
from util import assert_close, attn_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,Hq,Hkv,D,P", [
    (1, 4, 1, 128, 2047), (1, 4, 1, 128, 2048),   # the last key count with eight parts, and the first with nine
    (3, 2, 2, 64, 8189), (7, 5, 1, 64, 2400),     # 32 parts; a merge whose last workgroup is part empty
    (255, 8, 4, 128, 2100), (256, 8, 4, 128, 2100),  # either side of the row count that one-way merging takes
])
def test_parts_of_the_key_axis(dev, S, Hq, Hkv, D, P):
    t = attn_inputs(S, 64, Hq, Hkv, D, P=P, w_std=0.1)
    scale = 1.0 / math.sqrt(D)
    want = oracle.qkv_attention(t["x"], t["wq"], t["wk"], t["wv"], n_q_heads=Hq, n_kv_heads=Hkv, head_dim=D,
                                scale=scale, causal=True, kv_prefix=P, k_cache=t["k_cache"], v_cache=t["v_cache"],
                                want_lse=True)
    got = run_qkv(t, dev, Hq=Hq, Hkv=Hkv, D=D, P=P, scale=scale, causal=True, want_lse=True)
    assert_close(got["O2"], want["O2"], 2.0 ** -7, 2.0 ** -7, "O2")
    assert_close(got["lse"], want["lse"], 1e-3, 2e-3, "lse")


@pytest.mark.parametrize("S,Hq,Hkv,D,P", [
    (16, 8, 2, 128, 2048), (13, 10, 2, 64, 2111),   # 64 rows per KV head, and 65: half tiles per wave end here
    (4, 4, 1, 128, 2050), (5, 4, 1, 128, 2050),     # runs of two tiles, and of four
    (33, 4, 2, 64, 2100), (70, 4, 4, 128, 2241),    # pairs of tiles: an odd last tile, and none
    (9, 8, 1, 64, 28650), (9, 8, 1, 64, 28740),     # 72 rows, fp8: either side of seven tiles a run, from where pairs
    (17, 4, 1, 128, 28671),                         # ... with a last tile of 48 keys beside a full one
])
@pytest.mark.parametrize("fp8", [False, True])
def test_rows_and_tiles_of_a_run(dev, S, Hq, Hkv, D, P, fp8):
    scale = 1.0 / math.sqrt(D)
    kw = dict(n_q_heads=Hq, n_kv_heads=Hkv, head_dim=D, scale=scale, causal=True, kv_prefix=P)
    if fp8:
        t = _fp8_inputs(S, 64, Hq, Hkv, D, P)
        want = oracle.qkv_attention(t["x"], t["wq"], t["wk"], t["wv"], k_cache=t["k_cache"], v_cache=t["v_cache"],
                                    kv_fp8=True, k_scale=K_SCALE, v_scale=V_SCALE, **kw)
        got = _run(t, dev, "vanilla", Hq=Hq, Hkv=Hkv, D=D, P=P, causal=True)
        # (a new row's fp8 code may land one step, 2^-3 of the value, off: one of more than 2000 keys)
        assert_close(got["O2"], want["O2"], 1e-2, 1e-2, "O2")
    else:
        t = attn_inputs(S, 64, Hq, Hkv, D, P=P, w_std=0.1)
        want = oracle.qkv_attention(t["x"], t["wq"], t["wk"], t["wv"], k_cache=t["k_cache"], v_cache=t["v_cache"], **kw)
        got = run_qkv(t, dev, Hq=Hq, Hkv=Hkv, D=D, P=P, scale=scale, causal=True)
        assert_close(got["O2"], want["O2"], 2.0 ** -7, 2.0 ** -7, "O2")

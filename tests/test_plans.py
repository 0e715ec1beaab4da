"""CPU: what the launchers choose (csrc/launch.h: gemm_plan and the others; no part of the C ABI) - that the plans products are
given are among those measured fastest on the card, and that the GPU tests of a form of a kernel are given that form."""
import ctypes

import pytest

import test_gpu_attention
import test_gpu_fp8_kv
import test_gpu_random_shapes
import test_gpu_ring
from trinity_amd import ext

EIGHT_GROUPS = 3  # (csrc/launch.h: PrefillForm)
NONE, GELU, SWIGLU = 0, 1, 2
LARGE = (256, 256, 1)
# the ring kernels' tiles by number (csrc/ring.h: TRI_RING_TILES)
TILES = [(32, 128), (64, 64), (64, 128), (96, 128), (128, 128), (128, 192), (128, 256), (160, 256), (192, 128), (192, 192),
         (256, 128), (32, 128)]  # (the last for projections only: kRingTileFine)


class Plan(ctypes.Structure):
    _fields_ = [("tile", ctypes.c_int), ("parts", ctypes.c_int), ("us", ctypes.c_float)]


def plan_of(M, K, N, epi=NONE, kcontig=False, workspace=1 << 62):
    """(rows, columns, parts) of the tile that tri_matmul, tri_ffn_gelu or tri_gateup_swiglu run such a product on."""
    plan = Plan()
    takes = ext.lib()._ZN3tri9gemm_planEiiiiblRNS_8RingPlanE
    takes.restype = ctypes.c_bool
    if not takes(M, K, N, epi, ctypes.c_bool(kcontig), ctypes.c_int64(workspace), ctypes.byref(plan)):
        return LARGE
    return TILES[plan.tile] + (plan.parts,)


@pytest.mark.parametrize("M,K,N,epi,fast", [
    (96, 4096, 4096, NONE, [(64, 128, 4), (96, 128, 6)]),
    (128, 4544, 4544, NONE, [(64, 128, 3)]),
    (165, 4096, 4096, NONE, [(96, 128, 4)]),
    (70, 4544, 18176, NONE, [(96, 128, 1), (128, 128, 1), (128, 256, 2)]),
    (420, 4096, 4096, NONE, [(128, 128, 2)]),
    (900, 4096, 14336, SWIGLU, [LARGE]),
    (960, 4096, 14336, SWIGLU, [LARGE]),
    (600, 4544, 18176, GELU, [(128, 192, 1)]),
    (1200, 4544, 4544, NONE, [(192, 128, 1), (128, 192, 1)]),
    (1300, 4096, 4096, NONE, [(192, 128, 1)]),
    (1536, 8192, 4096, NONE, [(192, 128, 1)]),
    (2500, 8192, 2048, NONE, [(192, 128, 1), (160, 256, 2), (128, 192, 1)]),
    (8192, 4096, 1024, NONE, [LARGE]),
    (8192, 14336, 1024, NONE, [LARGE]),
])
def test_plans_are_among_the_fastest_measured(M, K, N, epi, fast):
    """Plans measured within 3 % of the fastest, as (rows, columns, parts) of a ring tile or LARGE for the large tiles; what
    such a product had been given before was 4 to 33 % behind."""
    assert plan_of(M, K, N, epi) in fast


@pytest.mark.parametrize("row", test_gpu_ring.LOADING_WAVES)
def test_loading_waves_are_given(row):
    M, K, N, plan = row
    room = ext.gemm_workspace_bytes(M, K, N)
    for kcontig in (False, True):
        for ws in (0, room) if plan[2] == 1 else (room,):
            assert plan_of(M, K, N, kcontig=kcontig, workspace=ws) == plan


@pytest.mark.parametrize("row", test_gpu_ring.LOADING_WAVES_GATED)
def test_loading_waves_of_gated_products_are_given(row):
    M, K, F, plan = row
    for kcontig in (False, True):
        for ws in (0, ext.gemm_workspace_bytes(M, K, 2 * F)):
            assert plan_of(M, K, F, SWIGLU, kcontig, ws) == plan


@pytest.mark.parametrize("row", test_gpu_ring.GELU_TILES)
def test_gelu_tiles_are_given(row):
    M, K, N, plan = row
    for kcontig in (False, True):
        for ws in (0, ext.ffn_workspace_bytes(M, K, N)):
            assert plan_of(M, K, N, GELU, kcontig, ws) == plan


@pytest.mark.parametrize("row", test_gpu_ring.QKV_TILES)
def test_projection_tiles_are_given(row):
    S, N, Hq, Hkv, D, tiles = row
    takes = ext.lib()._ZN3tri13qkv_ring_planEiiiiblbRNS_8RingPlanE
    takes.restype = ctypes.c_bool
    for qknorm, tile in zip((False, True), tiles):
        for kcontig in (False, True):
            p = ext.attn_params(Hq, Hkv, D, S, kv_prefix=5, qknorm=qknorm, rms_eps=1e-5)
            plan = Plan()
            assert takes(S, N, (Hq + 2 * Hkv) * D, D if qknorm else 0, ctypes.c_bool(kcontig),
                         ctypes.c_int64(ext.qkv_scratch_bytes(p, N)), ctypes.c_bool(False), ctypes.byref(plan))
            assert TILES[plan.tile] + (plan.parts,) == tile


@pytest.mark.parametrize("row", test_gpu_attention.SCORE_CASES)
def test_score_cases_are_given_their_form(row):
    S, _, Hq, _, _, P, causal, form = row
    got = ext.lib()._ZN3tri10score_formEiiib(S, P, Hq, ctypes.c_bool(causal))
    assert ["block", "block pair", "half block", "half block pair"][got] == form


@pytest.mark.parametrize("cfg", test_gpu_random_shapes.EIGHT_GROUP_CASES)
def test_eight_query_groups_are_given(cfg):
    S, _, Hq, _, D, P, causal = cfg
    for kf in (0, 2):  # plain, KeyFormer with seeded noise
        assert ext.lib()._ZN3tri12prefill_formEiiiibi(S, P, Hq, D, ctypes.c_bool(causal), kf) == EIGHT_GROUPS


def test_fp8_chunks_meet_every_form():
    """The key-split attention of more than 32 tokens over fp8 rows: each of its forms at each head width it is tested with."""
    form = ext.lib()._ZN3tri15split_attn_formEiiiib
    seen = {(D, form(S, Hq, Hkv, P + S, ctypes.c_bool(True))) for S, _, Hq, Hkv, D, P, _ in test_gpu_fp8_kv.CASES if S > 32}
    assert seen >= {(128, f) for f in range(3)} | {(64, f) for f in (0, 2)}

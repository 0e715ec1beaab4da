"""The GEMMs of ring.hip / ring_qkv.hip (few and middling rows) at the sizes where their tiles, remainders and parts can
go wrong, against fp32 products on the GPU.

Tolerance: both sides sum in fp32, so a result differs by its one rounding to fp16 (half an ulp, 2^-11 of the value;
two ulps allowed) and by the order of the sums (a few 2^-24 of the summed magnitudes, which are of order one here)."""
import pytest
import torch

from trinity_amd import ext

pytestmark = pytest.mark.gpu
REL, ABS = 2.0 ** -9, 1e-4


@pytest.fixture
def rn():
    g = torch.Generator(device="cuda:0")
    g.manual_seed(5)
    return lambda *s, std=1.0: torch.empty(*s, dtype=torch.float16, device="cuda:0").normal_(0.0, std, generator=g)


def check(got, want, what, rel=REL):
    torch.cuda.synchronize()
    bad = (got.float() - want).abs() > rel * want.abs() + ABS
    assert torch.isfinite(got).all() and not bad.any(), "%s: %d of %d, first at %s" % (
        what, int(bad.sum()), bad.numel(), bad.nonzero()[:1].tolist())


@pytest.mark.parametrize("M,K,N", [
    (1, 64, 8), (1, 96, 136), (32, 4096, 4096), (33, 96, 1000),      # one row; half a k tile at the end; tile edges
    (64, 14336, 4096), (65, 4544, 4544), (97, 4544, 4672),           # parts of K, ragged columns
    (129, 4096, 6144), (160, 4544, 18176), (161, 1056, 5000),        # row blocks with a remainder; K = 16.5 k tiles
    (300, 14336, 4096), (333, 18176, 4544), (700, 4096, 6144),
    (1100, 4096, 4096), (1101, 512, 1024),                           # the largest rows of the family, and one more
    (1101, 2048, 1024), (1500, 14336, 520), (2049, 4544, 1000),      # beyond them: narrow outputs over a deep K
    (8192, 2048, 72), (8193, 2048, 72),
])
@pytest.mark.parametrize("kcontig", [False, True])
@pytest.mark.parametrize("with_ws", [False, True])
def test_plain_and_residual(rn, M, K, N, kcontig, with_ws):
    x, r = rn(M, K), rn(M, N)
    w = rn(N, K, std=K ** -0.5).t() if kcontig else rn(K, N, std=K ** -0.5)
    ws = torch.empty(ext.gemm_workspace_bytes(M, K, N), dtype=torch.uint8, device="cuda:0") if with_ws else None
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda:0")
    ext.matmul(x, w, r, out, workspace=ws)
    check(out, x.float() @ w.float() + r.float(), "x.w + r")


# Tiles whose loads have waves of their own, in one part and in parts (tests/test_plans.py holds the rows against the plans): one k
# tile and two (fewer than the three stages that are requested ahead), K = 16.5, 64.5 and 109.5 k tiles (the last one
# begins half way back), a last row block of one row and full ones, ragged columns
LOADING_WAVES = [  # M, K, N, (rows, columns, parts)
    (193, 64, 16424, (128, 192, 1)), (385, 96, 11264, (128, 192, 1)), (385, 1056, 11264, (128, 192, 1)),
    (131, 64, 16424, (192, 128, 1)), (192, 128, 16584, (192, 128, 1)), (385, 1056, 9000, (192, 128, 1)),
    (257, 128, 24000, (192, 192, 1)), (513, 1056, 14000, (192, 192, 1)), (257, 4128, 24000, (192, 192, 1)),
    (385, 128, 14000, (256, 128, 1)), (512, 1056, 14000, (256, 128, 1)), (700, 1056, 9000, (256, 128, 1)),
    (500, 7008, 6144, (128, 192, 2)), (333, 8192, 4544, (192, 128, 3)), (129, 14336, 3000, (192, 128, 10)),
    (333, 18176, 4544, (192, 192, 5)), (500, 7008, 4544, (256, 128, 3)),
]


@pytest.mark.parametrize("M,K,N,plan", LOADING_WAVES)
@pytest.mark.parametrize("kcontig", [False, True])
@pytest.mark.parametrize("bf16", [False, True])
def test_loading_waves(rn, M, K, N, plan, kcontig, bf16):
    dt, tol = (torch.bfloat16, 2.0 ** -6) if bf16 else (torch.float16, REL)  # (bf16: two ulps of 2^-8)
    x = rn(M, K).to(dt)
    w = (rn(N, K, std=K ** -0.5).to(dt).t() if kcontig else rn(K, N, std=K ** -0.5).to(dt))
    want = x.float() @ w.float()
    for ws in (None, torch.empty(ext.gemm_workspace_bytes(M, K, N), dtype=torch.uint8, device="cuda:0")):
        out = torch.full((M, N), float("nan"), dtype=dt, device="cuda:0")
        ext.matmul(x, w, None, out, workspace=ws)
        check(out, want, "x.w", tol)


LOADING_WAVES_GATED = [
    (385, 96, 5632, (128, 192, 1)), (193, 4128, 8200, (128, 192, 1)), (131, 64, 8200, (192, 128, 1)),
    (150, 1056, 14336, (192, 128, 1)), (257, 128, 11264, (192, 192, 1)), (300, 1056, 11264, (192, 192, 1)),
    (193, 192, 14336, (256, 128, 1)), (700, 1056, 4544, (256, 128, 1)),
]


@pytest.mark.parametrize("M,K,F", [
    (1, 4096, 14336), (16, 96, 72), (48, 4096, 14336), (90, 4096, 14336), (130, 4096, 14336), (300, 4096, 14336),
    (100, 4544, 4544), (256, 4544, 4544), (500, 1024, 4000),
    (190, 4128, 3000), (1000, 96, 3064), (576, 1056, 5632),
] + [row[:3] for row in LOADING_WAVES_GATED])
@pytest.mark.parametrize("kcontig", [False, True])
def test_gated_with_row_scale(rn, M, K, F, kcontig):
    x, rs = rn(M, K), torch.rand(M, device="cuda:0") + 0.5
    wg, wu = ((rn(F, K, std=K ** -0.5).t() if kcontig else rn(K, F, std=K ** -0.5)) for _ in range(2))
    ws = torch.empty(ext.gemm_workspace_bytes(M, K, 2 * F), dtype=torch.uint8, device="cuda:0")
    a, b = (x.float() @ wg.float()) * rs[:, None], (x.float() @ wu.float()) * rs[:, None]
    for workspace in (ws, None):
        out = torch.full((M, F), float("nan"), dtype=torch.float16, device="cuda:0")
        ext.gateup_swiglu(x, wg, wu, rs, out, workspace=workspace)
        check(out, a * torch.sigmoid(a) * b, "gated")


@pytest.mark.parametrize("M,N", [(1, 64), (16, 512), (33, 1024), (64, 4096), (65, 1024), (128, 736)])
def test_few_rows_in_place(rn, M, N):
    """With a workspace a product of few rows may overwrite its input, also where its plan has one part."""
    x, wg, wu = rn(M, N), rn(N, N, std=N ** -0.5), rn(N, N, std=N ** -0.5)
    ws = torch.empty(ext.gemm_workspace_bytes(M, N, 2 * N), dtype=torch.uint8, device="cuda:0")
    a, b = x.float() @ wg.float(), x.float() @ wu.float()
    for call, want in ((lambda t: ext.matmul(t, wg, None, t, workspace=ws), a),
                       (lambda t: ext.gateup_swiglu(t, wg, wu, None, t, workspace=ws), a * torch.sigmoid(a) * b)):
        t = x.clone()
        call(t)
        check(t, want, "in place")
    # two views of one buffer: neighbouring columns, not in place
    buf = torch.cat([x, torch.zeros_like(x)], 1)
    ext.matmul(buf[:, :N], wg, None, buf[:, N:], workspace=ws)
    check(buf, torch.cat([x.float(), a], 1), "side by side")


@pytest.mark.parametrize("stride", [0, 8, 512])
def test_one_row_of_any_stride_in_place(rn, stride):
    """A single row's stride means nothing: zero, or less than the row, as a view may have it."""
    x, w = rn(1, 512), rn(512, 512, std=512 ** -0.5)
    want = x.float() @ w.float()
    ws = torch.empty(ext.gemm_workspace_bytes(1, 512, 512), dtype=torch.uint8, device="cuda:0")
    t = x.as_strided((1, 512), (stride, 1))
    ext.matmul(t, w, None, t, workspace=ws)
    check(t, want, "in place")


# first products with GELU, whose hidden rows go through the epilogue of the same tiles, also beyond 1100 rows
GELU_TILES = [
    (385, 96, 11264, (128, 192, 1)), (257, 1056, 11264, (192, 128, 1)), (513, 96, 14016, (192, 192, 1)),
    (700, 1056, 9024, (256, 128, 1)), (1120, 4544, 18176, (160, 256, 1)), (1500, 4544, 18176, (192, 192, 1)),
]


@pytest.mark.parametrize("M,K,N,plan", GELU_TILES)
@pytest.mark.parametrize("kcontig", [False, True])
def test_gelu_tiles(rn, M, K, N, plan, kcontig):
    x = rn(M, K)
    w = rn(N, K, std=K ** -0.5).t() if kcontig else rn(K, N, std=K ** -0.5)
    w2 = rn(64, N, std=N ** -0.5).t() if kcontig else rn(N, 64, std=N ** -0.5)
    want = torch.nn.functional.gelu(x.float() @ w.float())
    for ws in (None, torch.empty(ext.ffn_workspace_bytes(M, K, N), dtype=torch.uint8, device="cuda:0")):
        hidden = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda:0")
        ext.ffn_gelu(x, w, w2, hidden, torch.empty(M, 64, dtype=torch.float16, device="cuda:0"), workspace=ws)
        check(hidden, want, "gelu(x.w)")


QKV_TILES = [  # S, N, Hq, Hkv, D, (without, with QKNorm)
    (577, 1056, 48, 48, 64, [(128, 192, 1)] * 2), (769, 64, 71, 1, 64, [(192, 128, 1)] * 2),
    (1000, 1056, 71, 1, 64, [(192, 128, 1)] * 2), (900, 1056, 48, 48, 64, [(192, 192, 1)] * 2),
    (700, 1056, 48, 48, 64, [(256, 128, 1)] * 2), (129, 4128, 48, 48, 64, [(192, 128, 3)] * 2),
    (385, 96, 32, 32, 128, [(128, 192, 1), (256, 128, 1)]), (1000, 1056, 32, 8, 128, [(128, 192, 1), (256, 128, 1)]),
    (650, 64, 32, 8, 128, [(192, 128, 1)] * 2), (333, 1056, 64, 64, 128, [(192, 192, 1), (192, 128, 1)]),
    (577, 1056, 64, 8, 128, [(256, 128, 1)] * 2),
    # one round of 32-row tiles: 240 workgroups, last row blocks of one row and full ones, columns that end in half a tile
    (129, 96, 32, 8, 128, [(32, 128, 1)] * 2), (160, 4096, 32, 8, 128, [(32, 128, 1)] * 2),
    (150, 2560, 95, 1, 64, [(32, 128, 1)] * 2), (289, 1056, 16, 4, 128, [(64, 64, 1), (32, 128, 1)]),
]


@pytest.mark.parametrize("S,N,Hq,Hkv,D", [
    (1, 64, 4, 4, 64), (33, 96, 5, 1, 128), (100, 4096, 32, 8, 128), (260, 4096, 32, 8, 128), (200, 4544, 71, 1, 64),
    (700, 128, 32, 8, 128), (1000, 128, 71, 1, 64), (1100, 160, 32, 4, 128),  # a tile across two weight matrices
    (150, 4128, 32, 8, 128),
] + [row[:5] for row in QKV_TILES])
@pytest.mark.parametrize("qknorm", [False, True])
@pytest.mark.parametrize("kcontig", [False, True])
def test_qkv_projection(rn, S, N, Hq, Hkv, D, qknorm, kcontig):
    """The appended K / V rows and the q rows the projection leaves at the start of the scratch buffer."""
    x = rn(S, N)
    wq, wk, wv = ((rn(h * D, N, std=N ** -0.5).t() if kcontig else rn(N, h * D, std=N ** -0.5)) for h in (Hq, Hkv, Hkv))
    P = 5
    kc, vc = rn(Hkv, P + S, D), rn(Hkv, P + S, D)
    kept = kc[:, :P].clone(), vc[:, :P].clone()
    p = ext.attn_params(Hq, Hkv, D, S, kv_prefix=P, qknorm=qknorm, rms_eps=1e-5)
    scratch = torch.empty(ext.qkv_scratch_bytes(p, N), dtype=torch.uint8, device="cuda:0")
    # (a log-sum-exp pass keeps nothing fused away: q is stored by every path)
    s1, s2 = (torch.empty(Hq, P + S, dtype=torch.float32, device="cuda:0") for _ in range(2))
    ext.roco(x, None, wq, wk, wv, kc, vc, scratch, torch.empty(S, Hq * D, dtype=torch.float16, device="cuda:0"), s1, s2, p)

    def proj(w, heads, norm):
        t = (x.float() @ w.float()).view(S, heads, D)
        if norm:
            t = t.half().float()
            t = t * torch.rsqrt((t * t).mean(-1, keepdim=True) + 1e-5)
        return t

    check(scratch[: S * Hq * D * 2].view(torch.float16).view(S, Hq, D), proj(wq, Hq, qknorm), "q")
    check(kc[:, P:], proj(wk, Hkv, qknorm).transpose(0, 1), "k")
    check(vc[:, P:], proj(wv, Hkv, False).transpose(0, 1), "v")
    assert torch.equal(kc[:, :P], kept[0]) and torch.equal(vc[:, :P], kept[1])


@pytest.mark.parametrize("M,N,F", [(1, 64, 64), (16, 4096, 1024), (100, 4544, 512), (1200, 512, 256)])
def test_ffn_block_row_statistic(rn, M, N, F):
    """rsqrt(mean(attn_O2^2)) from the merge of the output projection, and from the kernel of its own."""
    o2, x, wo = rn(M, N), rn(M, N), rn(N, N, std=N ** -0.5)
    wa, wb, w2 = rn(N, F, std=N ** -0.5), rn(N, F, std=N ** -0.5), rn(F, N, std=F ** -0.5)
    attn, rows = torch.empty_like(x), torch.zeros(M, dtype=torch.float32, device="cuda:0")
    ws = torch.empty(max(16, ext.ffn_workspace_bytes(M, N, F)), dtype=torch.uint8, device="cuda:0")
    ext.ffn_block(o2, wo, x, wa, wb, w2, attn, rows, torch.empty(M, F, dtype=torch.float16, device="cuda:0"),
                  torch.empty_like(x), None, workspace=ws)
    check(attn, o2.float() @ wo.float() + x.float(), "attn_O2")
    want = torch.rsqrt((attn.double() ** 2).mean(1)).float()
    assert ((rows - want).abs() <= 1e-5 * want).all()  # fp32 sums of N squares


@pytest.mark.parametrize("M,K,N", [
    (1, 512, 4096), (16, 544, 4096), (7, 608, 1000),        # one 128-deep piece a wave; K ends 32 and 96 into a piece
    (3, 640, 24), (5, 1152, 8), (16, 2016, 520),            # waves with a piece more than others; less than 16 columns
    (16, 4096, 4104), (17, 4096, 4096), (2, 4544, 18176),   # a ragged last strip; one row too many; several a CU
])
def test_strips_over_k_contiguous_weights(rn, M, K, N):
    """Row strides beyond the columns, residual and GELU; what lies between the rows stays as it is."""
    x, r = rn(M, K + 24)[:, 8:K + 8], rn(M, N + 8)[:, :N]
    w = rn(N, K + 8, std=K ** -0.5)[:, :K].t()
    ws = torch.empty(ext.gemm_workspace_bytes(M, K, N), dtype=torch.uint8, device="cuda:0")
    buf = torch.full((M, N + 16), 7.0, dtype=torch.float16, device="cuda:0")
    out = buf[:, 8:N + 8]
    for workspace in (ws, None):
        out.fill_(float("nan"))
        ext.matmul(x, w, r, out, workspace=workspace)
        check(out, x.float() @ w.float() + r.float(), "x.w + r")
        assert (buf[:, :8] == 7).all() and (buf[:, N + 8:] == 7).all()
    w2 = rn(N, 64, std=N ** -0.5) if N % 32 else rn(64, N, std=N ** -0.5).t()  # (K-contiguous: K % 32 == 0)
    y = torch.empty(M, 64, dtype=torch.float16, device="cuda:0")
    ext.ffn_gelu(x, w, w2, out, y, workspace=None)
    want = torch.nn.functional.gelu(x.float() @ w.float())
    check(out, want, "gelu(x.w)")
    check(y, out.float() @ w2.float(), "hidden.w2")


def test_strips_and_a_product_over_its_own_input(rn):
    x, w = rn(4, 1024), rn(1024, 1024, std=1 / 32).t()
    want = x.float() @ w.float()
    ws = torch.empty(ext.gemm_workspace_bytes(4, 1024, 1024), dtype=torch.uint8, device="cuda:0")
    ext.matmul(x, w, None, x, workspace=ws)
    check(x, want, "x = x.w")


@pytest.mark.parametrize("M,K,N", [(1, 4096, 4096), (5, 1152, 8), (16, 544, 4096)])
def test_strips_in_bf16(rn, M, K, N):
    """As above with an element of 8 bits: two of its ulps, 2^-6 of the value, in place of fp16's 2^-9."""
    x, r, w = rn(M, K).bfloat16(), rn(M, N).bfloat16(), rn(N, K, std=K ** -0.5).bfloat16().t()
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    ext.matmul(x, w, r, out, workspace=None)
    want = x.float() @ w.float() + r.float()
    torch.cuda.synchronize()
    assert ((out.float() - want).abs() <= 2.0 ** -6 * want.abs() + ABS).all()


def check_bf16(got, want, what):
    """check() for an element of 8 bits: 2^-6 of the value in place of 2^-9."""
    torch.cuda.synchronize()
    assert ((got.float() - want).abs() <= 2.0 ** -6 * want.abs() + ABS).all(), what


# up to 32 rows on 32 x 128 tiles; which of them run three stages and which four follows from the workgroups of the last round
# (two a CU) and the distance between rows: 133 workgroups, 257, 399 and 195 in three parts, 144 in four, 504 in fourteen
@pytest.mark.parametrize("M,K,N", [(24, 544, 17000), (17, 1056, 32776), (20, 2080, 17000), (24, 4544, 8200), (32, 2080, 4552), (4, 5152, 4552)])
@pytest.mark.parametrize("kcontig", [False, True])
@pytest.mark.parametrize("bf16", [False, True])
def test_stages_of_plain_products(rn, M, K, N, kcontig, bf16):
    el, ok = (torch.bfloat16, check_bf16) if bf16 else (torch.float16, check)
    x, r = rn(M, K).to(el), rn(M, N).to(el)
    w = (rn(N, K, std=K ** -0.5).t() if kcontig else rn(K, N, std=K ** -0.5)).to(el)
    ws = torch.empty(ext.gemm_workspace_bytes(M, K, N), dtype=torch.uint8, device="cuda:0")
    for workspace in (ws, None):
        out = torch.full((M, N), float("nan"), dtype=el, device="cuda:0")
        ext.matmul(x, w, r, out, workspace=workspace)
        ok(out, x.float() @ w.float() + r.float(), "x.w + r")


# 225 workgroups, 257, and 213, 387 and 457 in three parts (of 4 KB of a K-contiguous column)
@pytest.mark.parametrize("M,K,F", [(17, 1056, 14344), (32, 544, 16400), (8, 1056, 4544), (3, 2080, 8200), (3, 6144, 9736)])
@pytest.mark.parametrize("kcontig", [False, True])
@pytest.mark.parametrize("bf16", [False, True])
def test_stages_of_gated_products(rn, M, K, F, kcontig, bf16):
    el, ok = (torch.bfloat16, check_bf16) if bf16 else (torch.float16, check)
    x = rn(M, K).to(el)
    wg, wu = ((rn(F, K, std=K ** -0.5).t() if kcontig else rn(K, F, std=K ** -0.5)).to(el) for _ in range(2))
    ws = torch.empty(ext.gemm_workspace_bytes(M, K, 2 * F), dtype=torch.uint8, device="cuda:0")
    a, b = x.float() @ wg.float(), x.float() @ wu.float()
    for workspace in (ws, None):
        out = torch.full((M, F), float("nan"), dtype=el, device="cuda:0")
        ext.gateup_swiglu(x, wg, wu, None, out, workspace=workspace)
        ok(out, a * torch.sigmoid(a) * b, "gated")


# 134, 208 and 258 workgroups in one part, and 64-wide heads
@pytest.mark.parametrize("S,N,Hq,Hkv,D", [(20, 544, 130, 2, 128), (32, 544, 192, 8, 128), (17, 544, 252, 3, 128), (20, 544, 260, 4, 64)])
@pytest.mark.parametrize("qknorm", [False, True])
@pytest.mark.parametrize("kcontig", [False, True])
def test_stages_of_the_projection(rn, S, N, Hq, Hkv, D, qknorm, kcontig):
    test_qkv_projection(rn, S, N, Hq, Hkv, D, qknorm, kcontig)


# K-contiguous columns 8 KB apart, 64 a workgroup: ragged last tiles, grids that are no multiple of the eight XCDs, plans in one
# part and (24 rows x [4096, 16392]) a plan in parts that this tile replaces; 1025 workgroups
@pytest.mark.parametrize("M,K,N", [(24, 544, 17000), (17, 1056, 32776), (24, 4096, 16392), (1, 1056, 28680), (32, 1088, 17032)])
@pytest.mark.parametrize("bf16", [False, True])
def test_narrow_tiles(rn, M, K, N, bf16):
    el, ok = (torch.bfloat16, check_bf16) if bf16 else (torch.float16, check)
    x, r = rn(M, K).to(el), rn(M, N).to(el)
    w = rn(N, 4096, std=K ** -0.5).to(el)[:, :K].t()
    ws = torch.empty(ext.gemm_workspace_bytes(M, K, N), dtype=torch.uint8, device="cuda:0")
    for workspace in (ws, None):
        buf = torch.full((M, N + 16), 7.0, dtype=el, device="cuda:0")
        out = buf[:, 8:N + 8]
        ext.matmul(x, w, r, out, workspace=workspace)
        ok(out, x.float() @ w.float() + r.float(), "x.w + r")
        assert (buf[:, :8] == 7).all() and (buf[:, N + 8:] == 7).all()
    if N % 32 == 0 or bf16:
        return
    y = torch.empty(M, 64, dtype=el, device="cuda:0")
    ext.ffn_gelu(x, w, rn(N, 64, std=N ** -0.5), out, y, workspace=ws)
    ok(out, torch.nn.functional.gelu(x.float() @ w.float()), "gelu(x.w)")


# 449 workgroups, 276 in place of a plan in parts, and 512, whose gate and up columns lie a multiple of 8 KB apart or 4 KB off that
@pytest.mark.parametrize("M,K,F,shift", [(1, 1056, 14344, 0), (32, 1056, 14344, 0), (17, 4096, 8808, 0), (32, 544, 16384, 0), (32, 544, 16384, 2048)])
@pytest.mark.parametrize("bf16", [False, True])
def test_narrow_gated_tiles(rn, M, K, F, shift, bf16):
    el, ok = (torch.bfloat16, check_bf16) if bf16 else (torch.float16, check)
    x, rs = rn(M, K).to(el), torch.rand(M, device="cuda:0") + 0.5
    both = rn(2 * F * 4096 + shift, std=K ** -0.5).to(el)
    wg, wu = both[:F * 4096].view(F, 4096)[:, :K].t(), both[F * 4096 + shift:].view(F, 4096)[:, :K].t()
    ws = torch.empty(ext.gemm_workspace_bytes(M, K, 2 * F), dtype=torch.uint8, device="cuda:0")
    a, b = (x.float() @ wg.float()) * rs[:, None], (x.float() @ wu.float()) * rs[:, None]
    for workspace in (ws, None):
        out = torch.full((M, F), float("nan"), dtype=el, device="cuda:0")
        ext.gateup_swiglu(x, wg, wu, rs, out, workspace=workspace)
        ok(out, a * torch.sigmoid(a) * b, "gated")

"""GPU parity at the prefill configuration (core prefill at the 3.5b shape: 4 sequences x 4096 tokens, bf16) and of the
tiled MFMA GEMM that serves every product with 33 or more token rows.

All calls go through the C ABI (pkg.hip wrappers).  Reference values: fp32 `F.linear` on the same operands for the
products (the library's GEMMs are row-independent, so a sample of rows is compared at full N), the CPU oracle's
`sdpa` per head for attention, and the oracle's SandwichBlock on a sample of rows of one sequence for the composed block
(attention needs all keys of that sequence, so its K / V rows are all computed by the oracle).
Bars: per kernel max-abs <= 2e-2 (times max(1, |ref|max)) and rel-L2 <= 1e-2; the composed block as in test_gpu_model.py."""

import math

import pytest
import torch
import torch.nn.functional as F

from oracle import raven_oracle as O
from test_gpu_kernels import ULPS_COMPOSED, ULPS_RESIDUAL, ULPS_SWIGLU, check, close, rnd

pytestmark = pytest.mark.gpu

H, NH, HD, INTER = 5280, 55, 96, 17920


def _rows(M, n=48, seed=0):
    """Rows to compare: the first and last tile edges plus a random sample."""
    g = torch.Generator().manual_seed(seed)
    picks = [torch.arange(0, min(M, 8)), torch.arange(max(0, M - 8), M), torch.randint(0, M, (n,), generator=g)]
    for edge in (255, 256, 257, 4095, 4096, 8191, 8192):
        if edge < M:
            picks.append(torch.tensor([edge]))
    return torch.unique(torch.cat(picks))


def _gpu_randn(shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, device="cuda", generator=g) * std).to(torch.bfloat16)


def _ref_rows(x, w, rows):
    """fp32 product of the sampled rows with the whole matrix (a plain PyTorch fp32 reference of nn.Linear)."""
    return F.linear(x[rows].float(), w.float())


# ----------------------------------------------------------------------------- the five products at M = 16384
@pytest.mark.parametrize("name", ["Wqkv", "attn.proj", "mlp.fc", "mlp.proj", "adapter", "lm_head"])
def test_tiled_gemm_nebel_shapes_m16384(pkg, name):
    """RMM:463, 493, 507-509, 776, 711 at 16384 token rows: the tiled kernel with each product's epilogue."""
    dt, M = torch.bfloat16, 16384
    rows = _rows(M).cuda()
    kw = {}
    if name == "Wqkv":
        x, w = _gpu_randn((M, H), 1), _gpu_randn((3 * H, H), 2, 0.02)
        got = pkg.hip.linear(x, w)
        want = _ref_rows(x, w, rows).to(dt)
    elif name == "attn.proj":
        x, w, res = _gpu_randn((M, H), 3), _gpu_randn((H, H), 4, 0.02), _gpu_randn((M, H), 5)
        got = pkg.hip.linear(x, w, residual=res)
        want = (_ref_rows(x, w, rows).to(dt).float() + res[rows].float()).to(dt)
        kw = dict(mag=_ref_rows(x, w, rows), ulps=ULPS_RESIDUAL)
    elif name == "mlp.fc":
        x, w = _gpu_randn((M, H), 6), _gpu_randn((2 * INTER, H), 7, 0.02)
        got = pkg.hip.linear(x, w, swiglu=True)
        z = _ref_rows(x, w, rows).to(dt).float()
        want = (F.silu(z[:, :INTER]).to(dt).float() * z[:, INTER:]).to(dt)
        wrong = (F.silu(z[:, INTER:]).to(dt).float() * z[:, :INTER]).to(dt)
        assert close(got[rows], wrong)[1] > 0.1, "the gate must be the first half of fc's output"
        kw = dict(ulps=ULPS_SWIGLU)
    elif name == "mlp.proj":
        x, w, res = _gpu_randn((M, INTER), 8), _gpu_randn((H, INTER), 9, 0.02), _gpu_randn((M, H), 10)
        got = pkg.hip.linear(x, w, residual=res)
        want = (_ref_rows(x, w, rows).to(dt).float() + res[rows].float()).to(dt)
        kw = dict(mag=_ref_rows(x, w, rows), ulps=ULPS_RESIDUAL)
    elif name == "adapter":
        x0, x1, w = _gpu_randn((M, H), 11), _gpu_randn((M, H), 12), _gpu_randn((H, 2 * H), 13, 0.02)
        got = pkg.hip.linear(x0, w, x1=x1)
        want = _ref_rows(torch.cat([x0[rows], x1[rows]], -1), w, torch.arange(rows.numel()).cuda()).to(dt)
        swapped = _ref_rows(torch.cat([x1[rows], x0[rows]], -1), w, torch.arange(rows.numel()).cuda()).to(dt)
        assert close(got[rows], swapped)[1] > 0.1, "the state is the first operand, the embedded input the second"
    else:  # lm_head: a quarter of the rows is enough for a 65536-wide output (float logits)
        M = 4096
        rows = _rows(M).cuda()
        x, w = _gpu_randn((M, H), 14), _gpu_randn((65536, H), 15, 0.02)
        got = pkg.hip.gemm(x, w, out_f32=True)
        assert got.dtype == torch.float32
        want = _ref_rows(x, w, rows).to(dt).float()
    check(got[rows], want, dt, f"{name} at {M} rows", **kw)
    assert torch.isfinite(got.float()).all()


@pytest.mark.parametrize("M", [33, 64, 65, 96, 128, 129, 160, 161])
def test_products_around_the_switch_between_skinny_passes_and_tiles(pkg, M):
    """33 to 161 token rows with the default dispatch: which kernel takes a product changes with the row count here
    (passes of the 32-row kernels up to 64 rows at K = 5280, 128 at 10560, 160 at 17920; 128 x 128 tiles beyond).  The five
    products of the 3.5b shape, each with its epilogue, on either side of every switch, against fp32 F.linear."""
    dt = torch.bfloat16
    x, e, res = _gpu_randn((M, H), 20 + M), _gpu_randn((M, H), 21 + M), _gpu_randn((M, H), 22 + M)
    g = _gpu_randn((M, INTER), 23 + M)
    rows = torch.arange(M).cuda()
    w = _gpu_randn((3 * H, H), 30, 0.02)
    check(pkg.hip.linear(x, w), _ref_rows(x, w, rows).to(dt), dt, f"Wqkv at {M} rows")
    w = _gpu_randn((H, H), 31, 0.02)
    p = _ref_rows(x, w, rows)
    check(pkg.hip.linear(x, w, residual=res), (p.to(dt).float() + res.float()).to(dt), dt, f"attn.proj at {M} rows", mag=p, ulps=ULPS_RESIDUAL)
    w = _gpu_randn((2 * INTER, H), 32, 0.02)
    z = _ref_rows(x, w, rows).to(dt).float()
    check(pkg.hip.linear(x, w, swiglu=True), (F.silu(z[:, :INTER]).to(dt).float() * z[:, INTER:]).to(dt), dt, f"mlp.fc at {M} rows",
          ulps=ULPS_SWIGLU)
    w = _gpu_randn((H, INTER), 33, 0.02)
    p = _ref_rows(g, w, rows)
    check(pkg.hip.linear(g, w, residual=res), (p.to(dt).float() + res.float()).to(dt), dt, f"mlp.proj at {M} rows", mag=p, ulps=ULPS_RESIDUAL)
    w = _gpu_randn((H, 2 * H), 34, 0.02)
    check(pkg.hip.linear(x, w, x1=e), _ref_rows(torch.cat([x, e], -1), w, rows).to(dt), dt, f"adapter at {M} rows")


@pytest.mark.parametrize("variant", [1, 2, 3])
@pytest.mark.parametrize("M,N,K", [(33, 64, 64), (64, 256, 256), (100, 264, 320), (257, 520, 96), (300, 5280, 5280), (513, 776, 1096), (700, 1032, 136)])
def test_tiled_gemm_edges_against_oracle(pkg, tuned, variant, M, N, K):
    """The three tile kernels (256 x 256 by four waves with an LDS ring, 128 x 128, 256 x 256 by eight waves with staging
    registers) on shapes with partial tiles in M and N, K that is not a multiple of the 64-wide step (down to one and
    two steps, fewer than the ring holds), every epilogue and the two-operand form, against the oracle's linear /
    SwiGLU / residual."""
    dt = torch.bfloat16
    tuned(gemm_tiled_variant=variant)
    x, w, res = rnd((M, K), dt, 500 + M), rnd((N, K), dt, 501 + N, 0.05), rnd((M, N), dt, 502)
    dev = lambda t: t.cuda()
    lin = lambda a, b: F.linear(a.float(), b.float())
    check(pkg.hip.linear(dev(x), dev(w)), lin(x, w).to(dt), dt, "plain")
    check(pkg.hip.linear(dev(x), dev(w), residual=dev(res)), lin(x, w).to(dt) + res, dt, "+ residual", mag=lin(x, w), ulps=ULPS_RESIDUAL)
    yf = pkg.hip.linear(dev(x), dev(w), out_f32=True)
    assert yf.dtype == torch.float32 and torch.equal(yf, pkg.hip.linear(dev(x), dev(w)).float())
    if N % 16 == 0:
        fc = rnd((2 * N, K), dt, 503, 0.05)
        z = lin(x, fc).to(dt)
        check(pkg.hip.linear(dev(x), dev(fc), swiglu=True), F.silu(z[:, :N]) * z[:, N:], dt, "SwiGLU", ulps=ULPS_SWIGLU)
    x1, w2 = rnd((M, K), dt, 504), rnd((N, 2 * K), dt, 505, 0.05)
    check(pkg.hip.linear(dev(x), dev(w2), x1=dev(x1)), lin(torch.cat([x, x1], -1), w2).to(dt), dt, "two operands")
    # against the oracle's own statement of the products (nn.Linear in bf16 on the CPU; small shapes only: it is slow)
    if M * N * K <= 2 * 10 ** 8:
        check(pkg.hip.linear(dev(x), dev(w)), O.linear(x, w), dt, "oracle linear")
    # the same call twice: the same bits; and the tile size does not change a bit either (one accumulation order)
    a = pkg.hip.linear(dev(x), dev(w))
    for other in {1, 2, 3} - {variant}:
        tuned(gemm_tiled_variant=other)
        assert torch.equal(a, pkg.hip.linear(dev(x), dev(w))), (variant, other)


def _assert_unit(pkg, M, N, K, nt, mt, ks, ws):
    """The plain and the SwiGLU product run as units of 2 nt weight tiles or one less, 4 mt - 3 token tiles or more, in ks slices."""
    for swiglu in (False, True):
        n, m, cols, rows, slices, units = pkg.hip.middle_plan(M, N, K, swiglu, ws.numel())
        wtiles = -(-cols * (2 if swiglu else 1) // 16)
        assert (n, m, slices) == (nt, mt, ks) and wtiles in (2 * nt - 1, 2 * nt) and 4 * mt - 3 <= rows // 16 <= 4 * mt and units >= ks, (M, N, K, swiglu)


@pytest.mark.parametrize("ks", [1, 3])
@pytest.mark.parametrize("mt", [1, 2, 3, 4])
@pytest.mark.parametrize("nt", [1, 2, 3, 4, 5, 6])
def test_products_of_a_middling_number_of_rows_in_every_cut(pkg, tuned, nt, mt, ks):
    """gemm_mid.hip: every tile shape, whole and in K slices, at sizes where units, steps and tiles end early: columns that leave the last
    unit and its last tile partly filled, rows past the last tile, fewer K steps than the ring has stages, a K that is no
    multiple of 64, a boundary between two segments inside a step; every epilogue, with rows of x padded or not."""
    dt = torch.bfloat16
    for M, N, K in ((33, 72, 72), (130, 328, 200), (259, 1048, 456), (70, 200, 1096)):
        tuned(gemm_mid_nt=nt, gemm_mid_mt=mt, gemm_mid_ks=ks)
        ws = pkg.hip.linear_workspace(M, 2 * N, "cuda")
        _assert_unit(pkg, M, N, K, nt, mt, min(ks, (K + 63) // 64), ws)
        x, w, res = _gpu_randn((M, K), 700 + M), _gpu_randn((N, K), 701 + N, 0.05), _gpu_randn((M, N), 702)
        z = x.float() @ w.float().T
        what = f"{M} x {N} x {K}"
        check(pkg.hip.linear(x, w, workspace=ws), z.to(dt), dt, what)
        check(pkg.hip.linear(x, w, residual=res, workspace=ws), (z.to(dt).float() + res.float()).to(dt), dt, what + " + residual", mag=z, ulps=ULPS_RESIDUAL)
        check(pkg.hip.linear(x, w, out_f32=True, workspace=ws), z.to(dt).float(), dt, what + ", float")
        fc = _gpu_randn((2 * N, K), 703, 0.05)
        u = (x.float() @ fc.float().T).to(dt).float()
        check(pkg.hip.linear(x, fc, swiglu=True, workspace=ws), (F.silu(u[:, :N]).to(dt).float() * u[:, N:]).to(dt), dt, what + ", SwiGLU", ulps=ULPS_SWIGLU)
        x1, w2 = _gpu_randn((M, K), 704), _gpu_randn((N, 2 * K), 705, 0.05)
        check(pkg.hip.linear(x, w2, x1=x1, workspace=ws), (torch.cat([x, x1], -1).float() @ w2.float().T).to(dt), dt, what + ", two operands")
        bias, resf = torch.randn(N, device="cuda"), torch.randn(M, N, device="cuda")
        got = pkg.hip.linear_epilogue(x, w, bias=bias, residual=resf, scale=0.5, workspace=ws)
        assert close(got, z * 0.5 + bias + resf)[1] < 3e-6, what + ", unrounded"   # fp32 sums of at most 1096 products in another order
        check(pkg.hip.linear_epilogue(x, w, bias=bias, act=pkg.hip.ACT_GELU, out_f32=False, workspace=ws), F.gelu(z + bias).to(dt), dt, what + ", gelu")
        check(pkg.hip.linear_epilogue(x, w, act=pkg.hip.ACT_TANH, out_f32=False, workspace=ws), torch.tanh(z).to(dt), dt, what + ", tanh")
        # the slices' sums do not depend on who adds them, and the same call gives the same bits
        assert torch.equal(pkg.hip.linear(x, w, workspace=ws), pkg.hip.linear(x, w, workspace=ws))


@pytest.mark.parametrize("nt", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("M", [35, 80, 143, 200, 300])
def test_units_with_any_number_of_tiles(pkg, tuned, nt, M):
    """gemm_mid.hip: units of every number of weight tiles and of 3 to 13 token tiles, so that waves get one tile more or less than others, or none;
    weight rows read by one unit (up to 256 rows) and by two; K of 4 steps and of 11, the last one partly filled."""
    dt = torch.bfloat16
    for N in (32 * nt - 24, 32 * nt):
        for K in (232, 680):
            tuned(gemm_mid_nt=nt, gemm_mid_mt=min(4, (M + 63) // 64), gemm_mid_ks=1)
            ws = pkg.hip.linear_workspace(M, 2 * N, "cuda")
            _assert_unit(pkg, M, N, K, nt, min(4, (M + 63) // 64), 1, ws)
            x, w = _gpu_randn((M, K), 760 + M), _gpu_randn((N, K), 761 + N, 0.05)
            check(pkg.hip.linear(x, w, workspace=ws), (x.float() @ w.float().T).to(dt), dt, f"{M} x {N} x {K}")
            half = max(8, N // 2 // 8 * 8)
            fc = _gpu_randn((2 * half, K), 762, 0.05)
            u = (x.float() @ fc.float().T).to(dt).float()
            check(pkg.hip.linear(x, fc, swiglu=True, workspace=ws), (F.silu(u[:, :half]).to(dt).float() * u[:, half:]).to(dt), dt, f"{M} x {half} x {K}, SwiGLU", ulps=ULPS_SWIGLU)


@pytest.mark.parametrize("M", [16, 17, 20, 32, 33])
def test_long_or_large_products_of_few_rows(pkg, M):
    """17 to 32 rows against a matrix with a long K (1032 x 4160) or a large one (20000 x 1024, 2 x 10000 x 1024), and the row counts beside: rounded
    results, SwiGLU, float sums added to a residual."""
    dt = torch.bfloat16
    for N, K in ((1032, 4160), (20000, 1024)):
        ws = pkg.hip.linear_workspace(M, N, "cuda")
        x, w, res = _gpu_randn((M, K), 780 + M), _gpu_randn((N, K), 781, 0.05), _gpu_randn((M, N), 782)
        z = x.float() @ w.float().T
        check(pkg.hip.linear(x, w, residual=res, workspace=ws), (z.to(dt).float() + res.float()).to(dt), dt, f"{M} x {N} x {K} + residual", mag=z, ulps=ULPS_RESIDUAL)
        resf = torch.randn(M, N, device="cuda")
        exact = x.double() @ w.double().T * 0.5 + resf.double()
        got = pkg.hip.linear_epilogue(x, w, residual=resf, scale=0.5, workspace=ws)
        assert ((got.double() - exact).norm() / exact.norm()).item() < 4e-7, f"{M} x {N} x {K}, unrounded"  # 2^-24 sqrt(4160 / 32 / 8) and the residual's own rounding
        assert torch.equal(got, pkg.hip.linear_epilogue(x, w, residual=resf, scale=0.5, workspace=ws))
    fc = _gpu_randn((20000, 1024), 783, 0.05)
    u = (x.float() @ fc.float().T).to(dt).float()
    check(pkg.hip.linear(x, fc, swiglu=True, workspace=ws), (F.silu(u[:, :10000]).to(dt).float() * u[:, 10000:]).to(dt), dt, f"{M} x 10000 x 1024, SwiGLU", ulps=ULPS_SWIGLU)


@pytest.mark.parametrize("M,N,K", [(17, 1024, 4160), (24, 2048, 5440), (32, 2048, 8192), (20, 1280, 17920), (29, 5280, 5312), (32, 10304, 2048)])
def test_float_sums_of_few_rows_are_as_near_as_the_skinny_kernels(pkg, tuned, M, N, K):
    """Sums that leave unrounded, 17 to 32 rows: no further from the exact ones than those of the skinny kernels, which add each up in eight parts; one chain
    is twice as far.  (1.05: the error of M x N sums varies by less than a hundredth.)"""
    x, w = _gpu_randn((M, K), 795 + M), _gpu_randn((N, K), 796, 0.05)
    exact, ws = x.double() @ w.double().T, pkg.hip.linear_workspace(M, N, "cuda")
    far = lambda: ((pkg.hip.linear_epilogue(x, w, workspace=ws).double() - exact).norm() / exact.norm()).item()
    got = far()
    tuned(gemm_mid=0)
    bar = far()
    assert got < 1.05 * bar, f"{M} x {N} x {K}: {got:.3g}, skinny kernels {bar:.3g}"


@pytest.mark.parametrize("M", [17, 32])
@pytest.mark.parametrize("N,K,swiglu,skinny", [(8192, 2560, 0, True), (8208, 2560, 0, False), (3584, 4096, 1, True), (4096, 16384, 0, True), (4096, 16448, 0, False),
                                               (11008, 8192, 0, True), (11008, 8256, 0, False), (2560, 16384, 1, True)])
def test_few_rows_stay_with_the_kernels_that_are_faster(pkg, tuned, M, N, K, swiglu, skinny):
    """17 to 32 rows: matrices of up to 8192 rows and K <= 4096, and slices of whole 4 KB over wide units, are the skinny kernels' (their bits: the order of sums
    differs); their neighbours are not."""
    x, w = _gpu_randn((M, K), 800 + M), _gpu_randn((N * (1 + swiglu), K), 801, 0.02)
    ws = pkg.hip.linear_workspace(M, N * (1 + swiglu), "cuda")
    got = pkg.hip.linear(x, w, swiglu=bool(swiglu), workspace=ws)
    tuned(gemm_mid=0)
    assert torch.equal(got, pkg.hip.linear(x, w, swiglu=bool(swiglu), workspace=ws)) == skinny


@pytest.mark.parametrize("M,N,K,parts", [(33, 1536, 1536, 4), (40, 2048, 2048, 4), (60, 1792, 7168, 8), (80, 2048, 5440, 8), (100, 2304, 2304, 3), (165, 2048, 2048, 4),
                                         (165, 2048, 8192, 8), (230, 2048, 8192, 8), (300, 512, 2048, 3), (450, 1024, 4096, 4), (385, 1280, 5120, 6)])
def test_float_sums_keep_the_parts_they_are_added_up_in(pkg, tuned, M, N, K, parts):
    """Sums that leave unrounded are no further from the exact ones than sums cut into `parts` slices, the fewest these sizes take: a whole chain is
    1.7 to 2.4 times as far.  (1.05: the same sums where the slices are as many; the error of M x N of them varies by less than a hundredth.)"""
    x, w = _gpu_randn((M, K), 790 + M), _gpu_randn((N, K), 791, 0.05)
    exact, ws = x.double() @ w.double().T, pkg.hip.linear_workspace(M, N, "cuda")
    far = lambda: ((pkg.hip.linear_epilogue(x, w, workspace=ws).double() - exact).norm() / exact.norm()).item()
    got = far()
    tuned(gemm_mid_ks=parts)
    bar = far()
    assert got < 1.05 * bar, f"{M} x {N} x {K}: {got:.3g}, in {parts} slices {bar:.3g}"


@pytest.mark.parametrize("ks", [1, 3])
@pytest.mark.parametrize("nt,mt", [(1, 1), (2, 1), (3, 3), (4, 2), (5, 4), (6, 3), (6, 4)])
def test_infinities_stay_in_their_rows_and_columns(pkg, tuned, nt, mt, ks):
    """Rows and columns past the end of a tile are repeats of the last ones, pieces past K are zeros, waves with fewer tiles than their variant multiply
    whatever lies behind them: an infinity or NaN of the last row of x, the last row of w or the last column must reach the outputs it belongs to and no
    other.  (215 x 392: last units with fewer tiles a wave than the variant's less one.)"""
    dt = torch.bfloat16
    for M, N, K in ((33, 72, 72), (130, 328, 200), (70, 200, 1096), (215, 392, 264)):
        tuned(gemm_mid_nt=nt, gemm_mid_mt=mt, gemm_mid_ks=ks)
        ws = pkg.hip.linear_workspace(M, 2 * N, "cuda")
        _assert_unit(pkg, M, N, K, nt, mt, min(ks, (K + 63) // 64), ws)
        x, w = _gpu_randn((M, K), 730 + M), _gpu_randn((2 * N, K), 731 + N, 0.05)
        x[M - 1, K - 1], x[0, 3] = float("inf"), float("nan")
        w[N - 1, 5] = w[2 * N - 1, 5] = float("inf")
        bad = torch.zeros(M, 2 * N, dtype=torch.bool, device="cuda")
        bad[0] = bad[M - 1] = bad[:, N - 1] = bad[:, 2 * N - 1] = True
        got = pkg.hip.linear(x, w[:N].contiguous(), workspace=ws)
        assert torch.equal(~got.isfinite(), bad[:, :N]), f"{M} x {N} x {K}"
        got = pkg.hip.linear(x, w, swiglu=True, workspace=ws)  # (silu of minus infinity is a zero or NaN: that row and column may go either way)
        assert got.isfinite()[~bad[:, :N]].all() and got[0].isnan().all(), f"{M} x {N} x {K}, SwiGLU"


@pytest.mark.parametrize("M,N,K", [(34, 96, 5184), (100, 1280, 1280), (150, 128, 1360), (260, 248, 1168), (400, 1024, 4096)])
def test_products_with_any_room_for_slices(pkg, M, N, K):
    """Shapes that are cut into K slices where the workspace holds them: with none, with room for two slices, with all of it; plain, + residual, float, SwiGLU,
    two operands."""
    dt = torch.bfloat16
    x, w, res = _gpu_randn((M, K), 720), _gpu_randn((N, K), 721, 0.05), _gpu_randn((M, N), 722)
    z = x.float() @ w.float().T
    u = z.to(dt).float()
    for ws in (None, torch.empty(2 * M * N * 4, dtype=torch.uint8, device="cuda"), pkg.hip.linear_workspace(M, N, "cuda")):
        check(pkg.hip.linear(x, w, workspace=ws), u.to(dt), dt, "plain")
        check(pkg.hip.linear(x, w, out_f32=True, workspace=ws), u, dt, "float")
        check(pkg.hip.linear(x, w, residual=res, workspace=ws), (u + res.float()).to(dt), dt, "+ residual", mag=z, ulps=ULPS_RESIDUAL)
        check(pkg.hip.linear(x, w, swiglu=True, workspace=ws), (F.silu(u[:, :N // 2]).to(dt).float() * u[:, N // 2:]).to(dt), dt, "SwiGLU", ulps=ULPS_SWIGLU)
        check(pkg.hip.linear(x[:, :K // 2].contiguous(), w, x1=x[:, K // 2:].contiguous(), workspace=ws), u.to(dt), dt, "two operands")


@pytest.mark.parametrize("M,N,K", [(40, 256, 4096), (100, 1024, 11008)])
def test_a_residual_off_sixteen_bytes(pkg, M, N, K):
    """The middle kernel loads whole 16-byte pieces; rows that the kernels of up to 32 rows can take in passes go there instead."""
    dt = torch.bfloat16
    x, w = _gpu_randn((M, K), 710), _gpu_randn((N, K), 711, 0.05)
    res = _gpu_randn((M * N + 1,), 712)[1:].view(M, N)
    z = x.float() @ w.float().T
    for ws in (None, pkg.hip.linear_workspace(M, N, "cuda")):
        check(pkg.hip.linear(x, w, residual=res, workspace=ws), (z.to(dt).float() + res.float()).to(dt), dt, "residual", mag=z, ulps=ULPS_RESIDUAL)


@pytest.mark.parametrize("M", [40, 100])
def test_slices_of_many_rows_folded_into_the_norm_change_no_bit(pkg, tuned, M):
    """A block over 33 and more rows at widths whose attn.proj and mlp.proj are cut into K slices: the norm launch adds them
    (fuse_sums_norm = 1) or a launch of their own does, with activation rows padded or not; same bits.  A workspace too small for the
    slices is no error: the product then takes another kernel."""
    h, nh, inter, dt = 480, 5, 2816, torch.bfloat16
    g = torch.Generator().manual_seed(3)
    mk = lambda *s: (torch.randn(*s, generator=g) * 0.03).to(dt).cuda()
    norms = [1 + mk(h) for _ in range(4)]
    blk = pkg.hip.make_block_weights(*norms, *(keep := [mk(3 * h, h), mk(2, 1, nh, 96), mk(h, h), mk(2 * inter, h), mk(h, inter)]))
    dims = pkg.hip.make_dims(h, nh, inter, 1e-6, dt)
    freqs = O.rope_table(96, M, 50000).to(dt).float().reshape(M, 48, 2).contiguous().cuda()
    x, ws = _gpu_randn((M, h), 9), pkg.hip.block_workspace(dims, M, "cuda")
    outs = []
    for fuse, pad, ks in ((1, 1, 0), (0, 1, 0), (1, 0, 0), (1, 1, 3), (0, 0, 3)):
        tuned(fuse_sums_norm=fuse, pad_chunk_rows=pad, gemm_mid_ks=ks)
        k, v = (torch.zeros(1, 1, nh, M, 96, dtype=dt, device="cuda") for _ in range(2))
        out = pkg.hip.sandwich_block(dims, blk, x, torch.empty_like(x), freqs, pkg.hip.make_cache(k, v), 0, 1, M, 0, ws)
        outs.append((out.clone(), k, v))
    for o in outs[1:3]:
        assert all(torch.equal(a, b) for a, b in zip(o, outs[0]))
    assert all(torch.equal(a, b) for a, b in zip(outs[3], outs[4]))
    check(outs[3][0], outs[0][0].float(), dt, "three slices against the default", ulps=ULPS_COMPOSED)
    a, w = _gpu_randn((M, inter), 10), keep[4]
    tiny = torch.empty(256, dtype=torch.uint8, device="cuda")
    check(pkg.hip.linear(a, w, workspace=tiny), (a.float() @ w.float().T).to(dt), dt, "without room for slices")


@pytest.mark.parametrize("M", [17, 32])
def test_slices_of_few_rows_folded_into_the_norm_change_no_bit(pkg, tuned, M):
    """17 and 32 rows whose attn.proj and mlp.proj (K > 4096) the middle kernel cuts into K slices: added by the norm launches or by launches of their own, the
    same bits; the skinny kernels' result within rounding."""
    h, nh, inter, dt = 4224, 44, 4352, torch.bfloat16
    mk = lambda seed, *s: _gpu_randn(s, seed, 0.02)
    norms = [1 + mk(810 + i, h) for i in range(4)]
    blk = pkg.hip.make_block_weights(*norms, *(keep := [mk(814, 3 * h, h), mk(815, 2, 1, nh, 96), mk(816, h, h), mk(817, 2 * inter, h), mk(818, h, inter)]))
    dims = pkg.hip.make_dims(h, nh, inter, 1e-6, dt)
    freqs = O.rope_table(96, M, 50000).to(dt).float().reshape(M, 48, 2).contiguous().cuda()
    x, ws = _gpu_randn((M, h), 9), pkg.hip.block_workspace(dims, M, "cuda")
    room = pkg.hip.linear_workspace(M, h, "cuda").numel()
    assert pkg.hip.middle_plan(M, h, h, False, room)[4] > 1 and pkg.hip.middle_plan(M, h, inter, False, room)[4] > 1
    outs = []
    for fuse, mid in ((1, 1), (0, 1), (1, 0)):
        tuned(fuse_sums_norm=fuse, gemm_mid=mid)
        k, v = (torch.zeros(1, 1, nh, M, 96, dtype=dt, device="cuda") for _ in range(2))
        out = pkg.hip.sandwich_block(dims, blk, x, torch.empty_like(x), freqs, pkg.hip.make_cache(k, v), 0, 1, M, 0, ws)
        outs.append((out.clone(), k, v))
    assert all(torch.equal(a, b) for a, b in zip(outs[0], outs[1]))
    check(outs[0][0], outs[2][0].float(), dt, "the middle kernel against the skinny ones", ulps=ULPS_COMPOSED)
    del keep


@pytest.mark.parametrize("h, nh, ks", [(64, 1, 1), (2048, 32, 8), (2080, 26, 5), (8192, 64, 2)])
def test_rows_formed_from_slices_have_the_norm_of_stored_rows(pkg, tuned, h, nh, ks):
    """Rows of fewer than 256 pieces of eight columns, exactly as many, a few more (in padded rows) and the most there may be: the launch that adds the slices of
    attn.proj and mlp.proj and norms the sums gives the bits of the launches that do one after the other."""
    M, inter, dt = 33, 1536, torch.bfloat16
    mk = lambda seed, *s: _gpu_randn(s, seed, 0.02)
    norms = [1 + mk(910 + i, h) for i in range(4)]
    blk = pkg.hip.make_block_weights(*norms, *(keep := [mk(914, 3 * h, h), mk(915, 2, 1, nh, h // nh), mk(916, h, h), mk(917, 2 * inter, h), mk(918, h, inter)]))
    dims = pkg.hip.make_dims(h, nh, inter, 1e-6, dt)
    hd = h // nh
    freqs = O.rope_table(hd, M, 50000).to(dt).float().reshape(M, hd // 2, 2).contiguous().cuda()
    x, ws = _gpu_randn((M, h), 9), pkg.hip.block_workspace(dims, M, "cuda")
    outs = []
    for fuse in (1, 0):
        tuned(fuse_sums_norm=fuse, gemm_mid_ks=ks)
        k, v = (torch.zeros(1, 1, nh, M, hd, dtype=dt, device="cuda") for _ in range(2))
        out = pkg.hip.sandwich_block(dims, blk, x, torch.empty_like(x), freqs, pkg.hip.make_cache(k, v), 0, 1, M, 0, ws)
        outs.append((out.clone(), k, v))
    assert all(torch.equal(a, b) for a, b in zip(*outs)) and outs[0][0].isfinite().all()
    del keep


@pytest.mark.parametrize("M, h, nh", [(33, 4096, 64), (300, 4096, 64), (4096, 5280, 55)])
def test_embedding_half_of_the_adapter_summed_once(pkg, tuned, M, h, nh):
    """Two recurrences over 33 and more rows, whose adapter is split by columns: in K slices that the norm adds, or a launch of their own, and in 256 x 256 tiles with a last
    round of smaller pieces.  The block's output matrices are zero, so that a recurrence is the adapter behind norms."""
    hip, dt, hd, inter = pkg.hip, torch.bfloat16, h // nh, 64
    one, zero = torch.ones(h, dtype=dt, device="cuda"), lambda *s: torch.zeros(*s, dtype=dt, device="cuda")
    keep = [one, _gpu_randn((3 * h, h), 931, 0.02), zero(2, 1, nh, hd), zero(h, h), _gpu_randn((2 * inter, h), 932, 0.02), zero(h, inter)]
    blocks = (hip.BlockWeights * 1)(hip.make_block_weights(one, one, one, one, *keep[1:]))
    dims = hip.make_dims(h, nh, inter, 1e-6, dt)
    ws = hip.block_workspace(dims, M, "cuda")
    freqs = O.rope_table(hd, M, 50000).to(dt).float().reshape(M, hd // 2, 2).contiguous().cuda()
    adapter, state, embeds = _gpu_randn((h, 2 * h), 933, h ** -0.5), _gpu_randn((M, h), 934), _gpu_randn((M, h), 935)

    def norm(x):
        return (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)).to(dt).float()

    want = state.float()
    for _ in range(2):
        z = (want @ adapter[:, :h].float().T + embeds.float() @ adapter[:, h:].float().T).to(dt).float()
        want = norm(norm(z))
    for fuse in (1, 0):
        tuned(fuse_sums_norm=fuse)
        k, v = zero(2, 1, nh, M, hd), zero(2, 1, nh, M, hd)
        got = hip.core_iterations(dims, adapter, blocks, state, embeds, torch.empty_like(state), freqs, hip.make_cache(k, v), [[0], [1]], 1, M, 0, ws)
        check(got, want.to(dt), dt, f"two recurrences, fuse_sums_norm={fuse}", ulps=ULPS_COMPOSED)
    del keep


@pytest.mark.parametrize("rows_of_units", [1, 3])
@pytest.mark.parametrize("mt", [1, 2, 3, 4])
@pytest.mark.parametrize("nt", [1, 2, 3, 4, 5, 6])
def test_rows_of_half_lines_by_parity(pkg, tuned, nt, mt, rows_of_units):
    """Weight rows that start on lines and in their middles by turns, every variant of units, with weights that one unit reads or several: read line by line (gemm_mid_half) they
    give the bits of rows read as they lie, as slices do, which always are; short and long K, a last unit of few columns, SwiGLU, a residual."""
    hip, dt = pkg.hip, torch.bfloat16
    for K, N, swiglu in ((160, 264, False), (672, 1048, False), (672, 520, True), (2080, 136, True)):
        M = 64 * mt - 20 if rows_of_units == 1 else 128 * mt + 5
        x, w = _gpu_randn((M, K), 21), _gpu_randn((N * (1 + swiglu), K), 22, K ** -0.5)
        res = None if swiglu else _gpu_randn((x.shape[0], N), 23)
        for ks in (1, 3):
            ws = hip.linear_workspace(x.shape[0], w.shape[0], "cuda")
            outs = []
            for half in (1, 0):
                tuned(gemm_mid_half=half, gemm_mid_nt=nt, gemm_mid_mt=mt, gemm_mid_ks=ks)
                plan = hip.middle_plan(M, N, K, swiglu, ws.numel())
                assert plan[:2] == (nt, mt) and plan[4] == ks and -(-M // plan[3]) == rows_of_units
                outs.append(hip.linear(x, w, residual=res, swiglu=swiglu, workspace=ws))
            assert torch.equal(*outs), (K, N, swiglu, ks)
            z = x.float() @ w.float().T
            want = F.silu(z[:, :N]) * z[:, N:] if swiglu else z + res.float()
            assert close(outs[0], want, "against float")[1] < 1e-2


def test_few_rows_read_a_copy_where_they_may(pkg, tuned):
    """20 rows against 1032 x 4200, whose rows are not whole lines: with a registered copy the product is the middle kernel's and reads it; with
    pad_decode_rows = 0, or without a copy, it reads the matrix."""
    hip, dt, M, N, K = pkg.hip, torch.bfloat16, 20, 1032, 4200
    x, w = _gpu_randn((M, K), 14), _gpu_randn((N, K), 15, 0.02)
    ws, z = hip.linear_workspace(M, N, "cuda"), x.float() @ w.float().T
    plain = hip.linear(x, w, workspace=ws)
    packed = hip.register_packed_weight(w)
    try:
        w.mul_(2)  # (exact: the copy holds half of it)
        copy = hip.linear(x, w, workspace=ws)
        tuned(pad_decode_rows=0)
        itself = hip.linear(x, w, workspace=ws)
    finally:
        hip.unregister_packed_weight(w)
    check(plain, z.to(dt), dt, "without a copy")
    check(copy, z.to(dt), dt, "the copy")
    assert torch.equal(itself, plain * 2) and torch.equal(itself, hip.linear(x, w, workspace=ws))
    del packed


@pytest.mark.parametrize("N", [16640, 16544])
def test_tiled_gemm_last_round_as_small_tiles_changes_no_bit(pkg, tuned, N):
    """4 x 65 tiles of 256 x 256 (4 x 130 under SwiGLU): the tiles of the last, nearly empty round (the last tile
    columns, whole or partly filled) are multiplied by a second launch over that column range, as units of the middle kernel here.  Same
    bits as one launch, for every epilogue, and right against the fp32 product on sampled columns of both ranges."""
    dt, M, K = torch.bfloat16, 1024, 192
    x, x1 = _gpu_randn((M, K), 600), _gpu_randn((M, K), 601)
    w, w2, res = _gpu_randn((N, K), 602, 0.05), _gpu_randn((N, 2 * K), 603, 0.05), _gpu_randn((M, N), 604)
    fc, bias = _gpu_randn((2 * N, K), 605, 0.05), _gpu_randn((N,), 606).float()
    calls = {"plain": lambda: pkg.hip.linear(x, w), "+ residual": lambda: pkg.hip.linear(x, w, residual=res),
             "float": lambda: pkg.hip.linear(x, w, out_f32=True), "two operands": lambda: pkg.hip.linear(x, w2, x1=x1),
             "SwiGLU": lambda: pkg.hip.linear(x, fc, swiglu=True),
             "gelu": lambda: pkg.hip.linear_epilogue(x, w, bias=bias, act=pkg.hip.ACT_GELU, out_f32=False),
             "tanh": lambda: pkg.hip.linear_epilogue(x, w, bias=bias, act=pkg.hip.ACT_TANH, out_f32=False),
             "unrounded": lambda: pkg.hip.linear_epilogue(x, w, bias=bias, residual=res.float(), scale=0.5)}
    assert all(pkg.hip.middle_plan(M, N - 16384, k, swiglu)[0] for k, swiglu in ((K, False), (2 * K, False), (K, True)))
    for name, call in calls.items():
        tuned(gemm_tiled_split_tail=1)
        split = call()
        tuned(gemm_tiled_split_tail=0)
        whole = call()
        assert torch.equal(split, whole), name
    cols = torch.tensor([0, 255, 256, 8191, 16383, 16384, 16385, 16511, 16512, N - 1]).cuda()
    tuned(gemm_tiled_split_tail=1)
    want = (x.float() @ w[cols].float().T).to(dt).float() + res[:, cols].float()
    check(pkg.hip.linear(x, w, residual=res)[:, cols], want.to(dt), dt, "sampled columns")
    z = (x.float() @ torch.cat([fc[cols], fc[N + cols]]).float().T).to(dt).float()
    want = (F.silu(z[:, :cols.numel()]).to(dt).float() * z[:, cols.numel():]).to(dt)
    check(pkg.hip.linear(x, fc, swiglu=True)[:, cols], want, dt, "sampled columns, SwiGLU")


# ----------------------------------------------------------------------------- attention at 4 x 4096
def test_prefill_attention_config4(pkg):
    """raven_prefill_attention at B=4, S=4096, 55 heads of 96: sampled (sequence, head) pairs against the oracle's sdpa,
    all 4096 query rows of each (the causal case of RMM:484-491)."""
    dt, B, S = torch.bfloat16, 4, 4096
    q = _gpu_randn((B * S, H), 21)
    k = _gpu_randn((1, B, NH, S, HD), 22)
    v = _gpu_randn((1, B, NH, S, HD), 23)
    cache = pkg.hip.make_cache(k, v)
    y = pkg.hip.prefill_attention(q, cache, 0, B, S, 0, NH, HD)
    torch.cuda.synchronize()
    for b, head in ((0, 0), (1, 17), (2, 54), (3, 31), (3, 0)):
        qh = q.view(B, S, NH, HD)[b, :, head].cpu()[None, None]
        want = O.sdpa(qh, k[0, b, head].cpu()[None, None], v[0, b, head].cpu()[None, None])[0, 0]
        check(y.view(B, S, NH, HD)[b, :, head], want, dt, f"sequence {b} head {head}")
    # the chunk kernel and the per-row kernel agree on a sample of rows (two implementations of the same softmax)
    rows = torch.tensor([0, 1, 63, 64, 127, 128, 2047, 2048, 4095])
    for b in (0, 3):
        for r in rows.tolist():
            qr = q.view(B, S, H)[b, r].view(1, NH, 1, HD)
            want = O.sdpa(qr.cpu(), k[0, b, :, :r + 1].cpu()[None], v[0, b, :, :r + 1].cpu()[None]).view(H)
            check(y.view(B, S, H)[b, r], want, dt, f"row {r} of sequence {b}")


def test_prefill_attention_wave_variants_agree(pkg, tuned):
    """head_dim 96 has two workgroup shapes (four waves = 128 query rows, six waves = 192): a row's arithmetic is the same
    in both, so the outputs must be the same bits -- with a chunk length that is no multiple of either, behind cached
    positions, and at the oracle's values on sampled rows."""
    dt, B, S, T0 = torch.bfloat16, 2, 1000, 24
    q = _gpu_randn((B * S, H), 61)
    k = _gpu_randn((1, B, NH, T0 + S, HD), 62)
    v = _gpu_randn((1, B, NH, T0 + S, HD), 63)
    cache = pkg.hip.make_cache(k, v)
    outs = {}
    for waves in (4, 6):
        tuned(prefill_waves=waves)
        outs[waves] = pkg.hip.prefill_attention(q, cache, 0, B, S, T0, NH, HD)
    torch.cuda.synchronize()
    assert torch.equal(outs[4], outs[6])
    for b, r in ((0, 0), (0, 191), (0, 192), (1, 575), (1, 999)):
        qr = q.view(B, S, H)[b, r].view(1, NH, 1, HD)
        want = O.sdpa(qr.cpu(), k[0, b, :, :T0 + r + 1].cpu()[None], v[0, b, :, :T0 + r + 1].cpu()[None]).view(H)
        check(outs[6].view(B, S, H)[b, r], want, dt, f"row {r} of sequence {b}")


# ----------------------------------------------------------------------------- one SandwichBlock at M = 16384
def test_sandwich_block_config4_rows(pkg):
    """raven_sandwich_block on 4 x 4096 rows at the 3.5b dims (tiled products, MFMA chunk attention, fused norms) against
    the oracle's SandwichBlock (RMM:525-536) on sampled rows of one sequence.  The oracle projects K and V for all 4096
    rows of that sequence (attention needs them) and everything else for the sampled rows only."""
    dt, B, S = torch.bfloat16, 4, 4096
    s = O.RavenShape.nebel()
    g = torch.Generator().manual_seed(31)
    prefix = "blk"
    w = {f"{prefix}.norm_{i}.weight": (torch.randn(H, generator=g) * 0.02 + 1).to(dt) for i in (1, 2, 3, 4)}
    w[f"{prefix}.attn.Wqkv.weight"] = (torch.randn(3 * H, H, generator=g) * 0.02).to(dt)
    w[f"{prefix}.attn.qk_bias"] = (torch.randn(2, 1, NH, HD, generator=g) * 0.02).to(dt)
    w[f"{prefix}.attn.proj.weight"] = (torch.randn(H, H, generator=g) * 0.02).to(dt)
    w[f"{prefix}.mlp.fc.weight"] = (torch.randn(2 * INTER, H, generator=g) * 0.02).to(dt)
    w[f"{prefix}.mlp.proj.weight"] = (torch.randn(H, INTER, generator=g) * 0.02).to(dt)
    dev = {k_: v_.cuda() for k_, v_ in w.items()}
    x = _gpu_randn((B * S, H), 32)
    table = O.rope_table(HD, s.block_size, s.rope_base).to(dt)
    freqs = table.float().reshape(s.block_size, HD // 2, 2).contiguous().cuda()
    kd = torch.zeros(1, B, NH, S, HD, dtype=dt, device="cuda")
    vd = torch.zeros_like(kd)
    cache = pkg.hip.make_cache(kd, vd)
    dims = pkg.hip.make_dims(H, NH, INTER, s.norm_eps, dt)
    blk = pkg.hip.make_block_weights(dev[f"{prefix}.norm_1.weight"], dev[f"{prefix}.norm_2.weight"], dev[f"{prefix}.norm_3.weight"],
                                     dev[f"{prefix}.norm_4.weight"], dev[f"{prefix}.attn.Wqkv.weight"], dev[f"{prefix}.attn.qk_bias"],
                                     dev[f"{prefix}.attn.proj.weight"], dev[f"{prefix}.mlp.fc.weight"], dev[f"{prefix}.mlp.proj.weight"])
    ws = pkg.hip.block_workspace(dims, B * S, "cuda")
    out = pkg.hip.sandwich_block(dims, blk, x, torch.empty_like(x), freqs, cache, 0, B, S, 0, ws)
    torch.cuda.synchronize()

    # ---- the oracle, sequence b, fp32-accumulate linears (the same mathematics; the CPU's bf16 GEMM would take minutes)
    b = 2
    rows = torch.tensor([0, 1, 15, 16, 63, 64, 255, 256, 1023, 2048, 3071, 4094, 4095])
    O.set_linear_mode("f32")
    try:
        xb = x.view(B, S, H)[b].cpu()
        n1 = O.rmsnorm(xb, w[f"{prefix}.norm_1.weight"], s.norm_eps)
        wqkv = w[f"{prefix}.attn.Wqkv.weight"]
        kv = O.linear(n1, wqkv[H:])                                     # K and V of every row of the sequence
        k_all, v_all = kv[:, :H].view(1, S, NH, HD), kv[:, H:].view(1, S, NH, HD)
        q_s = O.linear(n1[rows], wqkv[:H]).view(1, -1, NH, HD)          # queries of the sampled rows
        bias = w[f"{prefix}.attn.qk_bias"]
        k_all = (k_all + bias[1:2]).to(dt)
        q_s = (q_s + bias[0:1]).to(dt)
        _, k_rot = O.apply_rope(k_all, k_all, table[:, :S])
        q_rot, _ = O.apply_rope(q_s, q_s, table[:, rows])
        ya = []
        for i, r in enumerate(rows.tolist()):                           # row r attends to positions 0 .. r
            qi = q_rot[:, i:i + 1].transpose(1, 2)
            ya.append(O.sdpa(qi, k_rot[:, :r + 1].transpose(1, 2), v_all[:, :r + 1].transpose(1, 2)).transpose(1, 2).reshape(1, H))
        ya = torch.cat(ya, 0)
        a = O.linear(ya, w[f"{prefix}.attn.proj.weight"])
        x2 = O.rmsnorm(a + xb[rows], w[f"{prefix}.norm_2.weight"], s.norm_eps)
        m = O.gated_mlp(O.rmsnorm(x2, w[f"{prefix}.norm_3.weight"], s.norm_eps), w, prefix)
        want = O.rmsnorm(m + x2, w[f"{prefix}.norm_4.weight"], s.norm_eps)
    finally:
        O.set_linear_mode("native")
    got = out.view(B, S, H)[b][rows.cuda()]
    # the cache rows the block appended: rotated keys and values of every position, one kernel chain deep
    check(kd[0, b].transpose(0, 1), k_rot[0], dt, "appended K of the sequence", ulps=ULPS_COMPOSED)
    check(vd[0, b].transpose(0, 1), v_all[0], dt, "appended V of the sequence")
    err = close(got, want, "block output rows")
    print(f"SandwichBlock at 4 x 4096: sampled rows max-abs {err[0]:.3e} rel-L2 {err[1]:.3e}")
    # a chain of five products and four norms: the composed bar of test_gpu_model.py (per-kernel bars are applied kernel
    # by kernel above and in test_gpu_kernels.py)
    assert err[1] <= 3e-2, f"block output: rel-L2 {err[1]:.3e}"
    scale = max(1.0, want.float().abs().max().item())
    assert err[0] <= 2.5 * 2e-2 * scale, f"block output: max-abs {err[0]:.3e}"
    # rows of other sequences are finite and differ from this one's (no row was skipped or written twice)
    assert torch.isfinite(out.float()).all()
    assert not torch.equal(out.view(B, S, H)[0], out.view(B, S, H)[b])


@pytest.mark.parametrize("nh,hd,B,S,pos0,on_device", [(5, 96, 3, 50, 7, False), (55, 96, 2, 600, 0, True), (22, 128, 4, 512, 3, False),
                                                       (3, 64, 1, 33, 0, False)])
def test_chunk_qkv_epilogue_writes_the_bits_of_the_two_launch_path(pkg, tuned, nh, hd, B, S, pos0, on_device):
    """A chunk's q | k | v product with bias, RoPE and the cache append as its epilogue (fuse_qkv_rope = 1, the default) against
    the stored product followed by raven_qkv_bias_rope_cache_append (RMM:463-481): block output and the K / V rows the block
    appended, bit for bit; likewise with and without padded rows for the activations the tiled GEMM reads (pad_chunk_rows;
    n_embd 480 and 5280 are not multiples of 64).  Shapes: 128 x 128 tiles with rows of three sequences in one tile and heads across tile edges;
    256 x 256 tiles at the 3.5b head layout with the first position on the device; 256 x 256 tiles whose last tile column
    goes to 128 x 128 tiles (2048 rows x 8448 columns: 264 tiles); a single small tile with rows and columns past the end."""
    dt, h, inter = torch.bfloat16, nh * hd, 256
    g = torch.Generator().manual_seed(nh * 1000 + S)
    norms = [(torch.randn(h, generator=g) * 0.02 + 1).to(dt).cuda() for _ in range(4)]
    wqkv = (torch.randn(3 * h, h, generator=g) * 0.02).to(dt).cuda()
    bias = (torch.randn(2, 1, nh, hd, generator=g) * 0.02).to(dt).cuda()
    proj = (torch.randn(h, h, generator=g) * 0.02).to(dt).cuda()
    fc = (torch.randn(2 * inter, h, generator=g) * 0.02).to(dt).cuda()
    mproj = (torch.randn(h, inter, generator=g) * 0.02).to(dt).cuda()
    x = _gpu_randn((B * S, h), 5)
    t_max = pos0 + S + 3
    freqs = O.rope_table(hd, t_max, 50000).to(dt).float().reshape(t_max, hd // 2, 2).contiguous().cuda()
    dims = pkg.hip.make_dims(h, nh, inter, 1e-6, dt)
    blk = pkg.hip.make_block_weights(*norms, wqkv, bias, proj, fc, mproj)
    ws = pkg.hip.block_workspace(dims, B * S, "cuda")
    pos_dev = torch.tensor([pos0], dtype=torch.int32, device="cuda") if on_device else None
    results = []
    for fuse, pad in ((1, 1), (0, 0), (0, 1), (1, 0)):
        tuned(fuse_qkv_rope=fuse, pad_chunk_rows=pad)
        kd = _gpu_randn((2, B, nh, t_max, hd), 6)     # rows outside pos0 .. pos0 + S - 1 must stay as they are
        vd = _gpu_randn((2, B, nh, t_max, hd), 7)
        cache = pkg.hip.make_cache(kd, vd)
        out = pkg.hip.sandwich_block(dims, blk, x, torch.empty_like(x), freqs, cache, 1, B, S, pos0, ws, pos_dev=pos_dev)
        torch.cuda.synchronize()
        results.append((out.clone(), kd, vd))
    (o1, k1, v1), (o0, k0, v0) = results[:2]
    assert torch.equal(k1, k0), "appended K differs between the epilogue and the two-launch path"
    assert torch.equal(v1, v0), "appended V differs"
    assert torch.equal(o1, o0), "block output differs"
    for o, k, v in results[2:]:   # rows of the activations padded to whole cache lines or not, with either q | k | v path
        assert torch.equal(o, o0) and torch.equal(k, k0) and torch.equal(v, v0), "padded activation rows change the result"
    fresh = _gpu_randn((2, B, nh, t_max, hd), 6)
    assert torch.equal(k1[0], fresh[0]) and torch.equal(k1[1, :, :, :pos0], fresh[1, :, :, :pos0]) and torch.equal(k1[1, :, :, pos0 + S:], fresh[1, :, :, pos0 + S:])
    assert not torch.equal(k1[1, :, :, pos0:pos0 + S], fresh[1, :, :, pos0:pos0 + S])


@pytest.mark.parametrize("M,N,K,swiglu", [(300, 5280, 5280, False), (700, 1032, 136, False), (2048, 8448, 2816, False), (1100, 4096, 5280, True),
                                          (40, 64, 72, False), (93, 5280, 5280, False), (195, 5280, 5280, False)])
def test_packed_weight_copies_change_no_bit(pkg, M, N, K, swiglu):
    """raven_register_packed_weight: a product over 33 and more rows reads the line-aligned copy and writes the bits it
    writes from the matrix itself (both tile sizes, the last tile columns as small tiles, SwiGLU's gate / up rows, a
    K with a partial last step, K in slices); a matrix that changes must be registered again; after unregistering the matrix is read."""
    hip = pkg.hip
    x = _gpu_randn((M, K), 11)
    w = _gpu_randn((2 * N if swiglu else N, K), 12, std=0.02)
    res = None if swiglu else _gpu_randn((M, N), 13)
    ws = hip.linear_workspace(M, w.shape[0], "cuda") if M < 200 else None
    run = lambda: hip.linear(x, w, residual=res, swiglu=swiglu, workspace=ws)
    plain = run().clone()
    packed = hip.register_packed_weight(w)
    try:
        ld = (K + 63) // 64 * 64
        assert packed.numel() == w.shape[0] * ld * 2
        view = packed.view(torch.bfloat16).view(w.shape[0], ld)
        assert torch.equal(view[:, :K], w) and not view[:, K:].any()
        assert torch.equal(run(), plain)
        w.mul_(2)                                          # exact in bf16; the copy still holds the old values ...
        assert torch.equal(run(), plain), "the product did not read the registered copy"
        few = hip.linear(x[:8], w, residual=None if res is None else res[:8], swiglu=swiglu).clone()   # ... which 8 rows never read
        packed2 = hip.register_packed_weight(w)            # ... until the matrix is registered again
        again = run().clone()
    finally:
        hip.unregister_packed_weight(w)
    want = run()                                           # the matrix itself
    assert torch.equal(again, want) and not torch.equal(again, plain)
    check(few, want[:8].float(), torch.bfloat16, "8 rows against the first rows of the large product", ulps=ULPS_SWIGLU if swiglu else ULPS_RESIDUAL)
    del packed, packed2


def test_bench_prefill_iteration_runs_through_the_c_abi(pkg):
    """One recurrence over 4 x 512 rows through raven_core_iteration (adapter with two K segments, four blocks, chunk
    attention over a cache that already holds 512 positions): determinism, and the call equals adapter + four
    raven_sandwich_block calls bit for bit (one composition of the block behind the C ABI)."""
    dt, B, S, T = torch.bfloat16, 4, 512, 512
    s = O.RavenShape.nebel()
    w = O.make_weights(s, seed=0, dtype=dt, only_core=True)
    dev = {k_: v_.cuda() for k_, v_ in w.items()}
    from test_gpu_model import _block_weights
    blocks = (pkg.hip.BlockWeights * 4)(*[_block_weights(pkg, dev, f"transformer.core_block.{j}") for j in range(4)])
    dims = pkg.hip.make_dims(H, NH, INTER, s.norm_eps, dt)
    table = O.rope_table(HD, s.block_size, s.rope_base).to(dt)
    freqs = table.float().reshape(s.block_size, HD // 2, 2).contiguous().cuda()
    state, embeds = _gpu_randn((B * S, H), 41, 0.632), _gpu_randn((B * S, H), 42)
    k0, v0 = _gpu_randn((4, B, NH, T + S, HD), 43), _gpu_randn((4, B, NH, T + S, HD), 44)
    ws = pkg.hip.block_workspace(dims, B * S, "cuda")
    outs = []
    for _ in range(2):
        kd, vd = k0.clone(), v0.clone()
        out = torch.empty_like(state)
        pkg.hip.core_iteration(dims, dev["transformer.adapter.weight"], blocks, state, embeds, out, freqs, pkg.hip.make_cache(kd, vd), 0, B, S,
                               T, ws)
        outs.append((out, kd, vd))
    assert all(torch.equal(a, b) for a, b in zip(outs[0], outs[1]))
    kd, vd = k0.clone(), v0.clone()
    cache = pkg.hip.make_cache(kd, vd)
    cur = pkg.hip.linear(state, dev["transformer.adapter.weight"], x1=embeds)
    for j in range(4):
        nxt = torch.empty_like(cur)
        pkg.hip.sandwich_block(dims, blocks[j], cur, nxt, freqs, cache, j, B, S, T, ws)
        cur = nxt
    assert torch.equal(cur, outs[0][0]) and torch.equal(kd, outs[0][1]) and torch.equal(vd, outs[0][2])
    assert torch.isfinite(cur.float()).all()


@pytest.mark.parametrize("hd", [64, 96, 128])
def test_prefill_attention_reference_follows_every_lane(pkg, hd):
    """Scores far apart inside a tile, the largest at each of its places in turn: the running reference must see all of them."""
    S, nh, dt = 128, 2, torch.bfloat16
    g = torch.Generator().manual_seed(hd)
    k, v, q = (torch.randn(1, nh, S, hd, generator=g) for _ in range(3))
    for i in range(64, S):
        q[0, :, i] = 40 * k[0, :, i - 64]  # its score is about 40 sqrt(hd), the others' a small part of that
    q, k, v = q.to(dt), k.to(dt), v.to(dt)
    kc, vc = k[None].cuda(), v[None].cuda()
    cache = pkg.hip.make_cache(kc, vc)
    rows = q.transpose(1, 2).reshape(S, nh * hd).contiguous().cuda()
    got = pkg.hip.prefill_attention(rows, cache, 0, 1, S, 0, nh, hd).float().cpu().view(S, nh, hd)
    want = torch.nn.functional.scaled_dot_product_attention(q.double(), k.double(), v.double(), is_causal=True)[0].transpose(0, 1)
    assert torch.isfinite(got).all()
    assert (got - want).abs().max() < 5e-2

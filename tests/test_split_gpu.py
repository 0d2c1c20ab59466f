"""GPU checks of the fp32 tiles that multiply on the bf16 matrix cores
(gemm_split.hpp): each tile by name at sizes around its edges, K tails and
every transpose against the oracle accumulating in double; an error no larger
than fp32 sums in order leave; and the operands the split cannot hold
(infinities, NaN, values past bf16's largest, values below 2^-110 that a
result rests on), for which the kernel computes the tile again with fp32 MFMAs."""
import numpy as np
import pytest

import oracle
from gemm_cases import TOL, c_window, make_inputs, normwise, run_oracle, run_sbx

pytestmark = pytest.mark.gpu

SEED = 20261240

# plan, m, n, k: one tile short, one past, ragged; K from a part of a k tile on
TILES = [
    ("mfma_f32_256x128x16_w4x1", 255, 129, 96), ("mfma_f32_256x128x16_w4x1", 513, 260, 1031),
    ("mfma_f32_256x128x16_w4x1", 300, 140, 31), ("mfma_f32_256x128x16_w4x1+splitk3", 130, 127, 333),
    ("mfma_f32_128x128x16_w2x2", 127, 129, 33), ("mfma_f32_128x128x16_w2x2", 257, 130, 1030),
    ("mfma_f32_128x128x16_w2x2+splitk2", 100, 131, 64), ("mfma_f32_128x128x16_w2x2_o3", 129, 255, 65),
    ("mfma_f32_128x128x16_w2x2_o3", 1, 2, 700), ("mfma_f32_128x128x16_w2x2_o3+splitk5", 260, 3, 403),
    ("mfma_f32_256x64x32_w8x1", 257, 63, 127), ("mfma_f32_256x64x32_w8x1+splitk2", 300, 5, 1025),
    ("mfma_f32_256x48x32_w8x1", 511, 47, 129), ("mfma_f32_64x256x32_w1x8", 61, 257, 98),
    ("mfma_f32_48x256x32_w1x8+splitk2", 40, 257, 1026), ("mfma_f32_256x256x32_w4x2", 257, 255, 163),
]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_split_tiles_match_the_oracle(cuda, ta, tb):
    for i, (plan, m, n, k) in enumerate(TILES):
        off = ((0, 0, 0), (1, 2, 3))[i % 2]
        A, lda, B, ldb, C, ldc = make_inputs(np.float32, 0, ta, tb, m, n, k, SEED + i, pad=(3, 5, 2))
        C0 = C.copy()
        print(f"split case {m}x{n}x{k} t{ta}{tb} -> {plan}", flush=True)
        got = run_sbx(cuda, np.float32, 0, ta, tb, m, n, k, 1.25, A, lda, B, ldb, -0.5, C, ldc,
                      offsets=off, plan=plan)
        want = run_oracle(0, ta, tb, m, n, k, 1.25, A, lda, B, ldb, -0.5, C0, ldc)
        assert normwise(0, got, want, m, n, ldc) <= TOL[np.float32], plan
        pad = np.ones(C.size, bool)
        for r in range(m):
            pad[r * ldc:r * ldc + n] = False
        np.testing.assert_array_equal(got[pad], C0[pad])


@pytest.mark.parametrize("dist", ["uniform", "normal", "positive"])
def test_split_error_is_below_fp32_sums(cuda, dist):
    """Against double sums, the tile is no further off than the fp32 kernel
    that sums in order (the generic one), 64 to 4096 terms."""
    for i, k in enumerate((64, 257, 1000, 4096)):
        m, n = 256, 128
        A, lda, B, ldb, C, ldc = make_inputs(np.float32, 0, 0, 0, m, n, k, SEED + 40 + i,
                                             dist="normal" if dist == "normal" else "uniform")
        if dist == "positive":
            A, B = np.abs(A), np.abs(B)
        want = A.reshape(m, lda)[:, :k].astype(np.float64) @ B.reshape(k, ldb)[:, :n].astype(np.float64)
        errs = []
        for kw in ({"plan": "mfma_f32_256x128x16_w4x1"}, {"algo": 1}):
            got = run_sbx(cuda, np.float32, 0, 0, 0, m, n, k, 1.0, A, lda, B, ldb, 0.0, C, ldc, **kw)
            d = got.reshape(m, ldc)[:, :n].astype(np.float64) - want
            errs.append(float(np.linalg.norm(d) / np.linalg.norm(want)))
        print(f"{dist} k={k}: split {errs[0]:.2e}, fp32 in order {errs[1]:.2e}", flush=True)
        assert errs[0] <= errs[1]


PLANS = ["mfma_f32_256x128x16_w4x1", "mfma_f32_128x128x16_w2x2", "mfma_f32_128x128x16_w2x2_o3+splitk2",
         "mfma_f32_256x64x32_w8x1", "mfma_f32_64x256x32_w1x8"]


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
@pytest.mark.parametrize("plan", PLANS)
def test_operands_the_split_cannot_hold(cuda, plan, ta, tb):
    m, n, k = 270, 150, 200
    A, lda, B, ldb, C, ldc = make_inputs(np.float32, 0, ta, tb, m, n, k, SEED + 60)
    opa = A.reshape(k, lda).T if ta else A.reshape(m, lda)   # views: writes go to A, B
    opb = B.reshape(n, ldb).T if tb else B.reshape(k, ldb)
    opa[3, 17] = np.inf
    opa[5, 199] = np.nan
    opb[100, 70] = -np.inf
    opa[9, :] = np.float32(3.4e38)       # rounds to an infinite bf16
    opb[:, 7] *= np.float32(1e-6)
    opa[20, :] *= np.float32(1e-36)      # a row below 2^-100: pieces would lose bits
    opa[21, :] = 0.0
    opb[:, 9] *= np.float32(1e-34)
    # one tiny value in an ordinary row (the bound below is the row's: results that rest on
    # such a value are test_values_below_bf16_beside_ordinary_ones')
    opa[30, 40] = np.float32(1e-36)
    got = run_sbx(cuda, np.float32, 0, ta, tb, m, n, k, 1.0, A, lda, B, ldb, 0.0, C, ldc, plan=plan)
    got = c_window(0, got, m, n, ldc).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        want = opa.astype(np.float64) @ opb.astype(np.float64)
    # every sum past fp32's largest is far past it or far below it here,
    # except row 9's: k values of 3.4e38 times [-1, 1)
    free = np.zeros((m, n), bool)
    free[9, :] = True
    free[9, 7] = free[9, 9] = False      # ... which these two columns scale back into range
    nan = np.isnan(want)
    inf = np.isinf(want)
    np.testing.assert_array_equal(np.isnan(got) & ~free, nan & ~free)
    np.testing.assert_array_equal(got[inf & ~free], want[inf & ~free])
    fin = np.isfinite(want) & ~free
    assert np.isfinite(got[fin]).all()
    for r in range(m):  # row by row, so that the tiny row counts by itself
        for cols in ([9], [c for c in range(n) if c != 9]):
            f = [c for c in cols if fin[r, c]]
            if not f:
                continue
            scale = np.abs(opa[r].astype(np.float64)) @ np.abs(opb[:, f].astype(np.float64))
            with np.errstate(invalid="ignore"):
                e = np.abs(got[r, f] - want[r, f])
            # |error| <= 1e-6 of the sum of magnitudes (200 terms); results below
            # 2^-126 are rounded to multiples of 2^-149
            assert (e <= 1e-6 * scale + 2.0 ** -149 * k).all(), (r, float((e / (scale + 1e-300)).max()))


ALL_TILES = ["mfma_f32_256x128x16_w4x1", "mfma_f32_128x128x16_w2x2", "mfma_f32_128x128x16_w2x2+splitk3",
             "mfma_f32_128x128x16_w2x2_o3", "mfma_f32_256x256x32_w4x2", "mfma_f32_256x64x32_w8x1",
             "mfma_f32_256x48x32_w8x1", "mfma_f32_64x256x32_w1x8", "mfma_f32_48x256x32_w1x8"]


def _below_bf16(rng, m, n, k, kind):
    """Operands whose results rest on values that three bf16 values do not hold."""
    A = rng.uniform(0.5, 1.0, (m, k))
    B = rng.uniform(-1.0, 1.0, (k, n))
    if kind == "graded":        # A D^-1 times D B
        d = 2.0 ** np.round(np.linspace(0, 124, k))
        A, B = A / d, B * d[:, None]
    elif kind == "one":         # one such value a row, against large ones; 1.0 against a zero
        A[:] = 0.0
        A[:, 3], A[:, k - 2] = 1.0, 1e-41
        B[3] = 0.0
        B[k - 2] *= 1e30
    elif kind == "single":      # one result of the tile rests on such a value
        A[:, k - 2], B[:, 9] = 0.0, 0.0
        A[5, k - 2], B[k - 2, 9] = 1e-41, 1e30
    elif kind == "identity":    # B's values come through alone, beside an ordinary one a column
        A[:] = 0.0
        A[np.arange(min(m, k)), np.arange(min(m, k))] = 1.0
        B *= 1e-36
        B[0] = 1.0
    else:                       # half of each row 2^-e, its ordinary half against zeros
        A[:, k // 2:] *= 2.0 ** -kind
        B[:k // 2] = 0.0
    return A.astype(np.float32), B.astype(np.float32)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("kind", [112, 120, 126, 135, "graded", "one", "single", "identity"])
def test_values_below_bf16_beside_ordinary_ones(cuda, kind, ta, tb):
    for i, plan in enumerate(ALL_TILES):
        m, n, k = {"256x48": (300, 47), "48x256": (40, 300)}.get(plan[9:15], (259, 141)) + (230,)
        A, B = _below_bf16(np.random.default_rng(SEED + 80 + i), m, n, k, kind)
        sA, sB = np.ascontiguousarray(A.T if ta else A), np.ascontiguousarray(B.T if tb else B)
        print(f"{kind} t{ta}{tb} {plan}", flush=True)
        got = run_sbx(cuda, np.float32, 0, ta, tb, m, n, k, 1.0, sA.ravel(), sA.shape[1], sB.ravel(),
                      sB.shape[1], 0.0, np.zeros(m * n, np.float32), n, plan=plan)
        got = got.reshape(m, n).astype(np.float64)
        A, B = A.astype(np.float64), B.astype(np.float64)
        # |error| <= 1e-6 of each result's sum of magnitudes (230 terms in fp32), and half of
        # 2^-149 for each addition of a subnormal result
        err = np.abs(got - A @ B)
        assert (err <= 1e-6 * (np.abs(A) @ np.abs(B)) + 2.0 ** -150 * 2 * k).all(), (plan, float(err.max()))


@pytest.mark.parametrize("e", [126, 132, 140])
def test_subnormal_products_of_ordinary_operands(cuda, e):
    """Products below fp32's normal range: each is rounded to a multiple of 2^-149 and so
    is each addition, in the six partial products of a term too."""
    rng = np.random.default_rng(SEED + 95)
    m, n, k = 257, 130, 256
    A = (rng.uniform(-1, 1, (m, k)) * 2.0 ** -(e // 2)).astype(np.float32)
    B = (rng.uniform(-1, 1, (k, n)) * 2.0 ** -(e - e // 2)).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    scale = np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64))
    for plan in ALL_TILES[:5]:
        got = run_sbx(cuda, np.float32, 0, 0, 0, m, n, k, 1.0, A.ravel(), k, B.ravel(), n, 0.0,
                      np.zeros(m * n, np.float32), n, plan=plan).reshape(m, n)
        assert (np.abs(got - want) <= 1e-6 * scale + 2.0 ** -150 * 6 * k).all(), plan


@pytest.mark.parametrize("upper", [0, 1])
@pytest.mark.parametrize("trans", [0, 1])
def test_syrk_operands_the_split_cannot_hold(cuda, upper, trans):
    import sushiblas_amd as sbx
    import torch
    n, k = 400, 300
    rng = np.random.default_rng(SEED + 97)
    A = rng.uniform(-1, 1, (n, k)).astype(np.float32)
    A[150, 7] = np.inf
    A[260, 200] = np.nan
    A[33] *= np.float32(1e-36)
    A[40, 250:] *= np.float32(1e-37)
    A[40, :250] = 0.0
    A[41, 250:] *= np.float32(1e20)
    for plan in ("mfma_f32_128x128x16_w2x2", "mfma_f32_128x128x16_w2x2_o3+splitk2",
                 "mfma_f32_256x256x32_w4x2"):
        dA = torch.from_numpy(np.ascontiguousarray(A.T if trans else A)).to(cuda)
        dC = torch.full((n, n), 5.0, device=cuda)
        sbx.syrk_ex_plan(sbx.F32, 0, upper, trans, n, k, 1.0, dA, dA.shape[1], 0, 0.0, dC, n, 0, 1, plan)
        got = dC.cpu().numpy().astype(np.float64)
        a = A.astype(np.float64)
        with np.errstate(invalid="ignore"):
            want = a @ a.T
            scale = np.abs(a) @ np.abs(a).T
        want[41, 41] = np.inf  # row 41 times itself, 1.6e41, past fp32's largest
        i, j = np.indices((n, n))
        tri = j >= i if upper else j <= i
        assert (got[~tri] == 5.0).all()
        fin = tri & np.isfinite(want)
        np.testing.assert_array_equal(np.isnan(got) & tri, np.isnan(want) & tri)
        inf = tri & np.isinf(want)
        np.testing.assert_array_equal(got[inf], want[inf])
        e = np.abs(got[fin] - want[fin])
        # fp32 sums in order, the diagonal's of one sign: k roundings of at most 2^-24 of the sum
        # of magnitudes
        assert (e <= k * 2.0 ** -24 * scale[fin] + 2.0 ** -150 * 2 * k).all(), plan


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("fill", [np.nan, np.inf, 1e-40])
def test_memory_beside_the_operands_changes_nothing(cuda, fill, ta, tb):
    """Vector loads of an edge tile bring in the leading dimension's padding:
    whatever lies there, the result's bits are those of a zero padding."""
    for i, plan in enumerate(ALL_TILES):
        m, n, k = {"256x48": (301, 47), "48x256": (41, 301)}.get(plan[9:15], (257, 141)) + (165,)
        A, lda, B, ldb, C, ldc = make_inputs(np.float32, 0, ta, tb, m, n, k, SEED + 110 + i, pad=(3, 5, 2))
        got = []
        for v in (0.0, fill):
            for X, ld, width in ((A, lda, m if ta else k), (B, ldb, k if tb else n)):
                X[np.arange(X.size) % ld >= width] = v
            print(f"{fill} t{ta}{tb} {plan}", flush=True)
            got.append(run_sbx(cuda, np.float32, 0, ta, tb, m, n, k, 1.0, A, lda, B, ldb, 0.0, C, ldc, plan=plan))
        np.testing.assert_array_equal(got[0], got[1], plan)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_fp32_pass(cuda, ta, tb):
    """The tiles' fp32 products: short K, around the 16 and 32 k that its steps
    take, and longer K with an infinity in each corner of the tiles, whose
    finite results are fp32 sums in order."""
    for i, (k, inf) in enumerate([(1, 0), (3, 0), (15, 0), (16, 0), (17, 0), (31, 0), (33, 1), (100, 1), (271, 1)]):
        for plan in ALL_TILES:
            if "splitk" in plan and k < 96:
                continue
            m, n = {"256x48": (513, 48), "48x256": (48, 513)}.get(plan[9:15], (257, 259))
            A, lda, B, ldb, C, ldc = make_inputs(np.float32, 0, ta, tb, m, n, k, SEED + 130 + i, pad=(1, 2, 3))
            if inf:
                # (flat offsets of op(A)[0, 0] and op(A)[m - 1, k - 1])
                A[0] = np.inf
                A[(k - 1) * lda + m - 1 if ta else (m - 1) * lda + k - 1] = -np.inf
            print(f"fp32 pass {m}x{n}x{k} t{ta}{tb} {plan}", flush=True)
            got = run_sbx(cuda, np.float32, 0, ta, tb, m, n, k, 1.5, A, lda, B, ldb, 0.5, C, ldc, plan=plan)
            got = c_window(0, got, m, n, ldc)
            if inf:
                assert not np.isfinite(got[0]).any() and not np.isfinite(got[m - 1]).any(), plan
                A[0] = A[(k - 1) * lda + m - 1 if ta else (m - 1) * lda + k - 1] = 0
            want = c_window(0, run_oracle(0, ta, tb, m, n, k, 1.5, A, lda, B, ldb, 0.5, C, ldc), m, n, ldc)
            rows = slice(1, m - 1) if inf else slice(None)
            err = np.linalg.norm(got[rows].astype(np.float64) - want[rows]) / np.linalg.norm(want[rows])
            assert err <= TOL[np.float32], (plan, k, err)


@pytest.mark.parametrize("plan", ["mfma_f32_256x128x16_w4x1", "mfma_f32_128x128x16_w2x2_o3",
                                  "mfma_f32_128x128x16_w2x2+splitk2"])
@pytest.mark.parametrize("ld", [(1 << 24) + 3, (1 << 25) - 2])
def test_rows_more_than_2gib_apart_in_a_k_tile(cuda, plan, ld):
    """Operands whose 32 k rows span 2 to 4 GiB (unsigned buffer offsets): the
    bits are those of the same values stored densely."""
    import sushiblas_amd as sbx
    import torch
    m, n, k = 259, 131, 71
    if ld * 16 * 4 + 4 * 256 >= 0x7ffffff0 - 64:
        ld = (0x7ffffff0 - 64 - 4 * 256) // 64 - 1  # the largest that a 16-k step's offsets allow
    gen = torch.Generator(device=cuda).manual_seed(SEED)
    a = torch.empty(k, m, device=cuda).uniform_(-1, 1, generator=gen)
    b = torch.empty(k, n, device=cuda).uniform_(-1, 1, generator=gen)
    big = [torch.empty((k - 1) * ld + w, device=cuda) for w in (m, n)]
    for x, src in zip(big, (a, b)):
        for r in range(k):
            x[r * ld:r * ld + src.shape[1]] = src[r]
    out = []
    for A, lda, B, ldb in ((a, m, b, n), (big[0], ld, big[1], ld), (a, m, big[1], ld), (big[0], ld, b, n)):
        C = torch.zeros(m, n, device=cuda)
        print(f"{plan} lda {lda} ldb {ldb}", flush=True)
        sbx.gemm_ex_plan(sbx.F32, 0, 1, 0, m, n, k, 1.0, A, lda, 0, B, ldb, 0, 0.0, C, n, 0, 1, plan)
        out.append(C.cpu().numpy())
    for o in out[1:]:
        np.testing.assert_array_equal(o, out[0])
    want = (a.double().T @ b.double()).cpu().numpy()
    assert np.linalg.norm(out[0] - want) <= TOL[np.float32] * np.linalg.norm(want)


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
@pytest.mark.parametrize("batch,m,n", [(1, 513, 385), (3, 260, 300), (2, 255, 128)])
def test_pairs_in_batches_and_with_relu(cuda, batch, m, n, ta, tb):
    """Unsplit 256x128 plans with K >= 1024 whose few tiles would leave half the CUs
    idle run singly, in whole or fuller rounds in pairs: both through the batched
    and the fused entry points, on grids past one round, with ragged edges."""
    import sushiblas_amd as sbx
    import torch
    k = 1056
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = -(-m // 256) * -(-n // 128) * batch
    # copies of the batch until the last round holds fewer tiles than CUs, or more
    for want_more in (False, True):
        reps = next(r for r in range(1, 4 * cus) if (lambda left: left > cus if want_more else 0 < left <= cus)(
            tiles * r % (2 * cus)))
        nb = batch * reps
        gen = torch.Generator(device=cuda).manual_seed(SEED + nb)
        A = torch.empty((batch, k, m) if ta else (batch, m, k), device=cuda).uniform_(-1, 1, generator=gen)
        B = torch.empty((batch, n, k) if tb else (batch, k, n), device=cuda).uniform_(-1, 1, generator=gen)
        A, B = A.repeat(reps, 1, 1), B.repeat(reps, 1, 1)
        C0 = torch.empty(nb, m, n, device=cuda).uniform_(-1, 1, generator=gen)
        want = (A[:batch].mT if ta else A[:batch]).double().contiguous() @ (
            (B[:batch].mT if tb else B[:batch]).double().contiguous())
        args = (sbx.F32, 0, ta, tb, m, n, k, 1.5, A, A.shape[2], A[0].numel(), B, B.shape[2], B[0].numel(),
                0.5)
        C, R = C0.clone(), C0.clone()
        print(f"{nb} x {m}x{n}x{k} t{ta}{tb}: {tiles * reps} tiles", flush=True)
        sbx.gemm_ex_plan(*args, C, n, m * n, nb, "mfma_f32_256x128x16_w4x1")
        sbx.gemm_fused(*args, R, n, m * n, nb)
        for z in range(0, nb, max(1, nb // 7)):
            w = 1.5 * want[z % batch] + 0.5 * C0[z].double()
            for got, ref in ((C[z], w), (R[z], w.clamp_min(0))):
                assert (got - ref).norm() <= TOL[np.float32] * ref.norm(), (nb, z)

"""GPU parity (through the C ABI): the device stream, the FP64 factor and the
fused fp32 path kernels against the CPU oracle.

Bar: bit-exact for the normals, per-path crash counts S, per-path losses,
the exceedance count, the near-threshold count and the S histogram (the fp32
kernels mirror the oracle's fixed fma order); FP64 factor within 1e-10
relative of LAPACK."""
from __future__ import annotations

import ctypes
import json
import math
import os

import numpy as np
import pytest

from helpers import factor_like, random_spd

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")


def device_model(mcr, orc, mu, sigma, x, w=None):
    m = mcr.prepare(mu, sigma, x, w)
    return orc.F32Model(m["L32"], m["mu32"], m["v32"], m["mp32"], m["thr32"]), m


# ------------------------------------------------------------------ stream ---
@pytest.mark.parametrize("seed,path0,n", [(0, 0, 13), (67, 2**32 - 5, 8), (2**64 - 1, 2**63, 5),
                                          (0x123456789ABCDEF0, 12345, 64), (1, 7, 1)])
def test_device_stream_equals_oracle(mcr, orc, seed, path0, n):
    z = mcr.normals(seed, path0, 8192, n)
    ref = orc.normals_f32(seed, path0, 8192, n)
    assert np.array_equal(z.view(np.uint32), ref.view(np.uint32))


def test_device_stream_golden(mcr):
    g = json.load(open(os.path.join(GOLD, "normals_golden.json")))
    for c in g["cases"]:
        z = mcr.normals(int(c["seed"], 16), int(c["path"], 16), 1, c["n"])[0]
        assert [f"0x{int(b):08x}" for b in z.view(np.uint32)] == c["bits"]


def test_device_stream_one_million_paths(mcr, orc):
    z = mcr.normals(42, 1000, 1 << 20, 4)
    ref = orc.normals_f32(42, 1000, 1 << 20, 4)
    assert np.array_equal(z.view(np.uint32), ref.view(np.uint32))


# ------------------------------------------------------------------ factor ---
@pytest.mark.parametrize("n,cond", [(1, 1.0), (2, 10.0), (7, 1e2), (50, 1e4), (200, 1e6),
                                    (600, 1e4)])
def test_factor_matches_lapack(mcr, n, cond):
    A = random_spd(n, seed=100 + n, cond=cond)
    L, att, jit, cl = mcr.factor(A)
    assert att == 1 and jit == 0.0 and cl == 0
    ref = np.linalg.cholesky(A)
    assert np.all(np.triu(L, 1) == 0)
    assert np.max(np.abs(L - ref)) <= 1e-10 * np.max(np.abs(ref)) * max(1.0, cond**0.5)
    assert np.linalg.norm(L @ L.T - A) <= 64 * n * np.finfo(float).eps * np.linalg.norm(A)


def test_factor_jitter_policy_matches_oracle(mcr, orc):
    rng = np.random.default_rng(4)
    B = rng.uniform(0.2, 0.8, (20, 3)) * 0.01
    A = B @ B.T
    L, att, jit, cl = mcr.factor(A)
    oatt, oL, ojit, ocl = orc.factor(A)
    assert (att, cl) == (oatt, ocl) and att > 1
    # same policy step; the diagonal mean is summed in another order
    assert jit == pytest.approx(ojit, rel=1e-13)
    assert np.allclose(L, oL, rtol=1e-8, atol=1e-12)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 96, 97, 127, 128, 129, 160,
                               161, 288, 289, 767, 1024])
def test_factor_at_block_edges(mcr, n):
    """L L^T = A at the edges of the factor's 16-column panels, 32-column
    launches, 128-row workgroups and 64 x 64 update tiles.  Each entry's sum of
    at most n products and the factor's own rounding stay within (n + 10) eps
    of sqrt(A_ii A_jj) (the standard bound for Cholesky)."""
    A = random_spd(n, 100 + n, cond=50.0)
    L, att, jit, cl = mcr.factor(A)
    assert (att, jit, cl) == (1, 0.0, 0)
    assert np.all(np.triu(L, 1) == 0) and np.all(np.diag(L) > 0)
    d = np.sqrt(np.diag(A))
    assert np.max(np.abs(L @ L.T - A) / np.outer(d, d)) <= 2 * (n + 10) * np.finfo(float).eps


@pytest.mark.parametrize("col", [0, 1, 15, 16, 31, 32, 33, 63, 64, 95, 96, 100])
def test_factor_retries_from_any_column(mcr, orc, col):
    """A pivot that fails in any column of any launch sends the factor through
    the jitter policy, with the oracle's decisions; a non-finite entry in either
    triangle is refused."""
    # positive semidefinite: asset col's factor row is a mixture of the earlier
    # ones, so its pivot is rounding noise (exactly 0 for col = 0) and the first
    # jitter step makes it positive
    A = random_spd(101, 7, cond=10.0)
    F = np.linalg.cholesky(A)
    F[col] = np.random.default_rng(col).dirichlet(np.ones(col)) @ F[:col] if col else 0.0
    B = F @ F.T
    L, att, jit, cl = mcr.factor(B)
    oatt, oL, ojit, ocl = orc.factor(B)
    assert (att, cl) == (oatt, ocl) and att == 2
    assert jit == pytest.approx(ojit, rel=1e-13)
    for i, j in ((col, 100), (100, col)):
        C = A.copy()
        C[i, j] = np.nan
        with pytest.raises(mcr.McrError) as e:
            mcr.factor(C)
        assert e.value.code == mcr.MCR_E_FACTOR


@pytest.mark.parametrize("exp", [-760, -702, -698, 0, 988, 992, 1010])
@pytest.mark.parametrize("n", [7, 16, 70])
def test_factor_scales_with_the_covariance(mcr, n, exp):
    """A covariance times 4^k has the factor times 2^k, bit for bit, on either
    side of the diagonal sizes that the short root and reciprocal take."""
    A = random_spd(n, 300 + n, cond=50.0)
    A /= np.max(np.diag(A))
    L0 = mcr.factor(A)[0]
    L, att, jit, cl = mcr.factor(np.ldexp(A, exp))
    assert (att, jit, cl) == (1, 0.0, 0)
    assert np.array_equal(L, np.ldexp(L0, exp // 2))


@pytest.mark.parametrize("below", [1.0, 2.0, 4.0])
@pytest.mark.parametrize("exp", [-300, -2, 0, 8, 400])
def test_factor_root_and_reciprocal_are_correctly_rounded(mcr, below, exp):
    """L_jj = sqrt(d_j) and, beside a power of two c, L_nj = c (1 / sqrt(d_j)), bit
    for bit, for the last doubles below powers of two and four (a root whose
    significand is all ones has the one reciprocal that a fused correction rounds
    the wrong way), in both 16-column halves of two launches."""
    d, x = [], below
    for _ in range(40):
        x = np.nextafter(x, 0.0)
        d.append(np.ldexp(x, exp))
    d = np.array(d)
    c = np.ldexp(1.0, exp - 8)
    A = np.diag(np.append(d, np.ldexp(1.0, exp)))
    A[-1, :-1] = A[:-1, -1] = c
    L, att, jit, cl = mcr.factor(A)
    assert (att, jit, cl) == (1, 0.0, 0)
    assert np.array_equal(np.diag(L)[:-1], np.sqrt(d))
    assert np.array_equal(L[-1, :-1], c * (1.0 / np.sqrt(d)))


def _factor_replay(A):
    """The factor by panels of 16 columns, operation by operation: inside a panel
    one fused multiply-add per column, to the columns behind it a chain of 16 from
    zero, then one subtraction."""
    fma = ctypes.CDLL("libm.so.6").fma
    fma.restype, fma.argtypes = ctypes.c_double, [ctypes.c_double] * 3
    n = len(A)
    L = np.tril(A).tolist()
    for k0 in range(0, n, 16):
        k1 = min(k0 + 16, n)
        for c in range(k0, k1):
            root = math.sqrt(L[c][c])
            rl = 1.0 / root
            L[c][c] = root
            for r in range(c + 1, n):
                L[r][c] *= rl
            for r in range(c + 1, n):
                for c2 in range(c + 1, min(r + 1, k1)):
                    L[r][c2] = fma(-L[r][c], L[c2][c], L[r][c2])
        for i in range(k1, n):
            for j in range(k1, i + 1):
                acc = 0.0
                for p in range(k0, k1):
                    acc = fma(L[i][p], L[j][p], acc)
                L[i][j] -= acc
    return np.array(L)


@pytest.mark.parametrize("n", [17, 33, 70, 101])
def test_factor_bits_are_its_chains_of_fused_multiply_adds(mcr, n):
    """Every entry of the first attempt, whose updates run on the FP64 matrix
    instruction over several launches, bit for bit as a host replay computes it."""
    A = random_spd(n, 500 + n, cond=50.0)
    L, att, _, _ = mcr.factor(A)
    assert att == 1
    assert np.array_equal(L, _factor_replay(A))


def test_factor_clamp_fallback(mcr, orc):
    A = np.diag([1.0, 1.0, -0.5, 1.0]) * 1e-4
    L, att, jit, cl = mcr.factor(A)
    oatt, oL, ojit, ocl = orc.factor(A)
    assert att == oatt == 10 and cl == ocl == 1
    assert jit == pytest.approx(ojit, rel=1e-13)
    assert np.allclose(L, oL)


def test_factor_rejects_nonfinite(mcr):
    A = np.eye(4)
    A[2, 1] = np.inf
    with pytest.raises(mcr.McrError) as e:
        mcr.factor(A)
    assert e.value.code == mcr.MCR_E_FACTOR


def test_device_model_is_rounded_factor(mcr, orc):
    mu, sigma = factor_like(30, 3, 12)
    w = np.random.default_rng(1).dirichlet(np.ones(30))
    model, m = device_model(mcr, orc, mu, sigma, 0.02, w)
    L64 = m["L64"]
    assert np.array_equal(m["L32"], np.tril(L64).astype(np.float32))
    assert np.array_equal(m["mu32"], mu.astype(np.float32))
    v = L64.T @ w
    assert np.all(np.abs(m["v32"].astype(np.float64) - v) <= 1.5 * np.spacing(np.abs(v).astype(np.float32)))
    assert m["thr32"] == np.float32(-0.02)
    assert m["loss_sd"] == pytest.approx(np.sqrt(w @ sigma @ w), rel=1e-9)


# ------------------------------------------------------------ exact paths ---
def _exact_case(mcr, orc, n, M, k, kernel, seed=2024, path_offset=0, x=0.02, K=3, msd=31):
    mu, sigma = factor_like(n, min(K, n), msd + n)
    model, _ = device_model(mcr, orc, mu, sigma, x)
    r = mcr.run(mu, sigma, x, k, M, seed, kernel=kernel, want_S=True, want_loss=True, near=True,
                want_hist=True, path_offset=path_offset)
    ref = orc.simulate_f32(model, seed, path_offset, M, k, want_S=True, want_loss=True,
                           want_hist=True, nthreads=8)
    bad = np.nonzero(r.S != ref["S"])[0]
    assert bad.size == 0, f"{bad.size} paths differ, first {bad[:5]}"
    assert np.array_equal(r.loss.view(np.uint32), ref["loss"].view(np.uint32))
    assert r.count == ref["count"]
    assert r.near_threshold == ref["near"]
    assert np.array_equal(r.s_hist, ref["hist"])
    return r


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 13, 20, 31, 32, 33, 50, 63, 64])
def test_register_kernel_exact(mcr, orc, n):
    r = _exact_case(mcr, orc, n, 20000, max(1, n // 5), mcr.KERNEL_VALU_REG)
    assert r.kernel == "valu_reg"


@pytest.mark.parametrize("n", [1, 5, 8, 9, 50, 64, 65, 100, 129, 257, 600, 608])
def test_tile_kernel_exact(mcr, orc, n):
    M = 20000 if n <= 129 else 4000
    r = _exact_case(mcr, orc, n, M, max(1, n // 5), mcr.KERNEL_VALU_TILE)
    assert r.kernel == "valu_tile"


@pytest.mark.parametrize("n", [31, 32, 62, 63, 64, 90, 95, 96, 97, 126, 127])
def test_wave_kernel_exact(mcr, orc, n):
    """The fp32 wave kernel at the edges of its 32-row tiles, 8-column octets
    and half blocks, over paths whose ids cross 2^32 inside a 64-path group."""
    r = _exact_case(mcr, orc, n, 5000, max(1, n // 5), mcr.KERNEL_VALU_TILE,
                    path_offset=2**32 - 2469)
    assert r.kernel == "valu_tile"


@pytest.mark.parametrize("kernel", [2, 5])
@pytest.mark.parametrize("n", [128, 148, 149, 160, 308, 309, 320, 511, 512, 513, 608])
def test_lds_kernel_exact_at_shape_edges(mcr, orc, n, kernel):
    """The fp32 LDS kernel at the edges of its workgroup shapes (n = 148 / 149,
    308 / 309), row tiles and column chunk, with and without a spare row for
    the loss, over paths whose ids cross 2^32 inside a 64-path group."""
    _exact_case(mcr, orc, n, 1500, max(1, n // 5), kernel, path_offset=2**32 - 741)


@pytest.mark.parametrize("n", [152, 153, 304, 305])
def test_lds_kernel_exact_where_workgroups_fit(mcr, orc, n):
    """The same at the last n where four workgroups (of four waves) and two (of
    eight) share a compute unit's LDS, and the first where they do not."""
    _exact_case(mcr, orc, n, 1500, max(1, n // 5), 2, path_offset=2**32 - 741)


@pytest.mark.parametrize("n", [609, 640, 1024])
def test_column_chunks_of_a_group_across_32_bits(mcr, orc, n):
    """The same past 608 assets, where a group whose path ids cross 2^32 goes
    through its column chunks twice."""
    _exact_case(mcr, orc, n, 1500, n // 5, 5, path_offset=2**32 - 741, K=12)


@pytest.mark.parametrize("scale,x", [(1e-38, 1e-40), (1e-40, 1e-42), (3e39, 1e38), (1e41, 1e38)])
@pytest.mark.parametrize("n,kernel", [(50, 1), (50, 2), (95, 2), (127, 2), (128, 5), (143, 2), (305, 2),
                                      (608, 2), (640, 5)])
def test_fp32_kernels_exact_at_the_ends_of_the_range(mcr, orc, n, kernel, scale, x):
    """Subnormal factors and sums, overflowing sums, infinite factor entries (their
    NaNs included) and means: S, the losses (any NaN equal to any other), the counts
    and the histogram are the oracle's, so the matrix instruction neither flushes
    nor reorders."""
    mu, sigma = factor_like(n, 3, 31 + n, T=max(1500, 2 * n))
    mu, sigma = mu * scale, sigma * scale * scale
    if scale > 1e40:
        mu[::3] *= -1e5  # past fp32, most to +-infinity
        mu[1::3] = 1.0
    model, m = device_model(mcr, orc, mu, sigma, x)
    low = np.abs(m["L32"][np.tril_indices(n)])
    assert np.all(low < 2.0**-126) if scale < 1 else np.any(np.isinf(low)) == (scale > 1e40)
    k = max(1, n // 5)
    r = mcr.run(mu, sigma, x, k, 1500, 2024, kernel=kernel, want_S=True, want_loss=True, near=True,
                want_hist=True)
    ref = orc.simulate_f32(model, 2024, 0, 1500, k, want_S=True, want_loss=True, want_hist=True,
                           nthreads=8)
    assert np.array_equal(r.S, ref["S"])
    assert np.array_equal(np.isnan(r.loss), np.isnan(ref["loss"]))
    ok = ~np.isnan(r.loss)
    assert np.array_equal(r.loss[ok].view(np.uint32), ref["loss"][ok].view(np.uint32))
    assert (r.count, r.near_threshold) == (ref["count"], ref["near"])
    assert np.array_equal(r.s_hist, ref["hist"])


@pytest.mark.parametrize("n", [1, 5, 9, 50, 129, 257, 600, 608, 609, 700, 1000, 1024])
def test_chunk_kernel_exact(mcr, orc, n):
    """The column-chunk kernel (any n <= 1024; fp32 past 608): per-path
    S and loss bits, count, near-threshold count and S histogram equal the
    oracle's.  n = 609-1024 covers one and two 512-column chunks, a last
    chunk of one 4-column block (n = 1024 - 3 .. 1024 ends on block 255) and
    n not a multiple of 4 or 8."""
    M = 20000 if n <= 129 else (4000 if n <= 608 else 1500)
    T = max(4000, 2 * n)
    mu, sigma = factor_like(n, min(12, n), 31 + n, T=T)
    model, _ = device_model(mcr, orc, mu, sigma, 0.02)
    k = max(1, n // 5)
    r = mcr.run(mu, sigma, 0.02, k, M, 2024, kernel=mcr.KERNEL_VALU_CHUNK, want_S=True,
                want_loss=True, near=True, want_hist=True)
    ref = orc.simulate_f32(model, 2024, 0, M, k, want_S=True, want_loss=True, want_hist=True,
                           nthreads=8)
    assert r.kernel == "valu_chunk"
    bad = np.nonzero(r.S != ref["S"])[0]
    assert bad.size == 0, f"{bad.size} paths differ, first {bad[:5]}"
    assert np.array_equal(r.loss.view(np.uint32), ref["loss"].view(np.uint32))
    assert r.count == ref["count"] and r.near_threshold == ref["near"]
    assert np.array_equal(r.s_hist, ref["hist"])


def test_chunk_and_tile_kernels_agree_at_scale(mcr):
    """Size-independent property at the n = 600 workload's shape (1e6
    paths): the column-chunk and tile kernels compute identical per-path
    results, so their counts, tails and quantiles are identical."""
    mu, sigma = factor_like(600, 20, 6000, T=4000)
    a = mcr.run(mu, sigma, 0.02, 597, 1_000_000, 5, kernel=mcr.KERNEL_VALU_TILE, alphas=(0.99,))
    b = mcr.run(mu, sigma, 0.02, 597, 1_000_000, 5, kernel=mcr.KERNEL_VALU_CHUNK, alphas=(0.99,))
    assert a.count == b.count and a.var == b.var and a.tail_sum_fixed == b.tail_sum_fixed


def test_past_767_assets_every_precision_runs_the_chunk_kernel(mcr):
    """Above 767 assets (the LDS MFMA kernel's 24 row tiles) every precision
    (and the automatic choice) runs the column-chunk kernel and gives the same
    result; naming the tile or an MFMA kernel there is refused, as is
    n = 1025."""
    mu, sigma = factor_like(800, 10, 8000, T=2000)
    rs = [mcr.run(mu, sigma, 0.02, 80, 5000, 3, precision=p, alphas=(0.99,))
          for p in (mcr.PREC_FP32, mcr.PREC_BF16X3, mcr.PREC_AUTO)]
    assert all(r.kernel == "valu_chunk" for r in rs)
    assert len({(r.count, r.var[0]) for r in rs}) == 1
    for kernel in (mcr.KERNEL_VALU_TILE, mcr.KERNEL_MFMA_LDS, mcr.KERNEL_MFMA):
        with pytest.raises(mcr.McrError) as e:
            mcr.run(mu, sigma, 0.02, 80, 100, 3, kernel=kernel)
        assert e.value.code == mcr.MCR_E_UNSUPPORTED
    with pytest.raises(mcr.McrError) as e:
        mcr.run(np.zeros(1025), np.eye(1025) * 1e-4, 0.02, 1, 10, 1)
    assert e.value.code == mcr.MCR_E_UNSUPPORTED


# MCR_PARITY_RANDOM_CASES raises the number of randomized cases for a longer run
@pytest.mark.parametrize("case", range(int(os.environ.get("MCR_PARITY_RANDOM_CASES", "4"))))
def test_randomized_fp32_queries_match_oracle(mcr, orc, case):
    """Random single queries on the fp32 kernels (every kernel valid for the
    drawn n in 1-1024: register, tile, column chunk), path counts, path
    offsets, seeds, thresholds, k and weights: per-path S and loss bits,
    count, near-threshold count and S histogram equal the oracle's."""
    rng = np.random.default_rng(4242 + case)
    n = int(rng.choice([int(rng.integers(1, 65)), int(rng.integers(65, 609)),
                        int(rng.integers(609, 1025))]))
    kernels = ([mcr.KERNEL_VALU_REG] if n <= 64 else []) + \
        ([mcr.KERNEL_VALU_TILE] if n <= 608 else []) + [mcr.KERNEL_VALU_CHUNK]
    kernel = int(rng.choice(kernels))
    M = int(np.exp(rng.uniform(0.0, np.log(4e6 / max(n, 40)))))
    seed = int(rng.integers(0, 2**63)) * 2 + int(rng.integers(0, 2))
    path0 = int(rng.choice([0, int(rng.integers(0, 2**40)), 2**32 - M // 2]))
    x = float(rng.uniform(-0.005, 0.04))
    k = int(rng.integers(0, n + 2))
    mu, sigma = factor_like(n, int(rng.integers(1, min(20, n) + 1)), 900 + case, T=max(1500, 2 * n))
    w = None if rng.uniform() < 0.5 else rng.dirichlet(np.ones(n))
    model, _ = device_model(mcr, orc, mu, sigma, x, w)
    r = mcr.run(mu, sigma, x, k, M, seed, weights=w, kernel=kernel, want_S=True, want_loss=True,
                near=True, want_hist=True, path_offset=path0)
    ref = orc.simulate_f32(model, seed, path0, M, k, want_S=True, want_loss=True, want_hist=True,
                           nthreads=8)
    tag = (n, kernel, M, path0, k)
    assert np.array_equal(r.S, ref["S"]), tag
    assert np.array_equal(r.loss.view(np.uint32), ref["loss"].view(np.uint32)), tag
    assert (r.count, r.near_threshold) == (ref["count"], ref["near"]), tag
    assert np.array_equal(r.s_hist, ref["hist"]), tag


@pytest.mark.parametrize("M", [1, 63, 64, 65, 257, 1000])
@pytest.mark.parametrize("kernel", [1, 2, 5])
def test_ragged_path_counts(mcr, orc, M, kernel):
    _exact_case(mcr, orc, 20, M, 5, kernel)


@pytest.mark.parametrize("kernel", [1, 2, 5])
def test_path_ids_cross_32_bits_and_large_seed(mcr, orc, kernel):
    _exact_case(mcr, orc, 11, 5000, 3, kernel, seed=2**64 - 1, path_offset=2**32 - 2500)


@pytest.mark.parametrize("k", [0, 1, 20, 21])
def test_k_edges(mcr, orc, k):
    r = _exact_case(mcr, orc, 20, 3000, k, mcr.KERNEL_VALU_REG)
    if k == 0:
        assert r.count == 3000
    if k == 21:
        assert r.count == 0


def test_threshold_edges(mcr, orc):
    # x huge: nobody crashes; x negative enough: everybody crashes on every asset
    mu, sigma = factor_like(10, 2, 3)
    r = mcr.run(mu, sigma, 10.0, 1, 1000, 1)
    assert r.count == 0
    r = mcr.run(mu, sigma, -10.0, 10, 1000, 1)
    assert r.count == 1000
    _exact_case(mcr, orc, 10, 5000, 2, mcr.KERNEL_VALU_REG, x=0.0)


def test_register_and_tile_agree_at_scale(mcr):
    """Size-independent property at the fused-kernel workload's size (n = 50,
    1e8 paths): the two fp32 kernels compute identical per-path results, so
    their counts, tails and quantiles are identical."""
    mu, sigma = factor_like(50, 5, 1002)
    a = mcr.run(mu, sigma, 0.02, 10, 100_000_000, 7, kernel=mcr.KERNEL_VALU_REG, alphas=(0.99,))
    b = mcr.run(mu, sigma, 0.02, 10, 100_000_000, 7, kernel=mcr.KERNEL_VALU_TILE, alphas=(0.99,))
    assert a.count == b.count
    assert a.var == b.var and a.tail_sum_fixed == b.tail_sum_fixed


def test_subrange_of_large_run_matches_oracle(mcr, orc):
    """Path ids address the stream directly: a 20000-path window at offset
    99,980,000 of the n = 50 workload equals the oracle's same window."""
    _exact_case(mcr, orc, 50, 20000, 10, mcr.KERNEL_VALU_REG, seed=7, path_offset=99_980_000, K=5,
                msd=952)


@pytest.mark.parametrize("paths", [262143, 262144, 262145, 524288, 786433])
def test_per_path_outputs_across_staging_pieces(mcr, paths):
    """S and loss of paths on both sides of the 1 MiB staging pieces' edges: the
    parts of a run split elsewhere, the crash count and the S histogram."""
    mu, sigma = factor_like(7, 2, 91, T=1500)
    r = mcr.run(mu, sigma, 0.02, 2, paths, 5, want_S=True, want_loss=True, want_hist=True)
    cut = 100_003
    a = mcr.run(mu, sigma, 0.02, 2, cut, 5, want_S=True, want_loss=True)
    b = mcr.run(mu, sigma, 0.02, 2, paths - cut, 5, want_S=True, want_loss=True, path_offset=cut)
    assert np.array_equal(r.S, np.concatenate([a.S, b.S]))
    assert np.array_equal(r.loss, np.concatenate([a.loss, b.loss]))
    assert np.array_equal(r.s_hist, np.bincount(r.S, minlength=8))
    assert r.count == int((r.S >= 2).sum())

"""Neighbor-list build on the GPU (build_neighbors, src/neighbors.rs:180-281):
identical CSR lists to the exact f32 brute-force restatement."""

import numpy as np
import pytest

from dynamics_amd import api, systems
from oracle import reference_path as rp

pytestmark = pytest.mark.gpu


def _check(ctx, outer, inner, static, ext, symmetric, thr):
    rp_g, col_g = ctx.build_neighbors(outer, inner, static, ext, symmetric, thr)
    rp_o, col_o = rp.build_neighbors(outer, inner, static, ext, symmetric, thr)
    assert np.array_equal(rp_g, rp_o)
    assert np.array_equal(col_g, col_o)
    return rp_g, col_g


@pytest.mark.parametrize("seed", [2, 5])
def test_build_all_neighbors_matches_bruteforce(gpu, seed):
    s = systems.solvated_chain(27.0, 600, 30, 40, seed=seed, lattice_n=10)
    ctx = api.ForcesPositsGpu(s.n_dyn, s.n_water, 10.0, 0.3123)
    ext = s.box.astype(np.float32)
    thr = np.float32(14.0 * 14.0)
    wpos = rp.wrap_ref(s.pos_o, np.zeros(3, np.float32), ext)
    static = np.zeros(s.n_dyn, np.uint8)
    static[::7] = 1
    _check(ctx, s.pos_dyn, s.pos_dyn, static, ext, True, thr)
    _check(ctx, s.pos_dyn, s.pos_dyn, None, ext, True, thr)
    _check(ctx, s.pos_dyn, wpos, None, ext, False, thr)
    _check(ctx, wpos, wpos, None, ext, True, thr)


def test_unwrapped_solute_and_threshold_ties(gpu):
    """Solute coordinates outside the box and points placed exactly on the
    threshold distance and on half-box separations."""
    rng = np.random.default_rng(7)
    ext = np.array([30.0, 30.0, 30.0], np.float32)
    p = (rng.uniform(-45, 75, (400, 3))).astype(np.float32)
    p[1] = p[0] + np.array([12.0, 0, 0], np.float32)   # |d| = 12 exactly: strict '<' excludes
    p[3] = p[2] + np.array([15.0, 0, 0], np.float32)   # half box
    p[5] = p[4] + np.array([-15.0, 0, 0], np.float32)
    ctx = api.ForcesPositsGpu(400, 0, 10.0, 0.3)
    _check(ctx, p, p, None, ext, True, np.float32(144.0))


def test_config0_water_water(gpu):
    s = systems.config0()
    ext = s.box.astype(np.float32)
    wpos = rp.wrap_ref(s.pos_o, np.zeros(3, np.float32), ext)
    ctx = api.ForcesPositsGpu(0, s.n_water, 10.0, 0.3123)
    rp_g, col_g = _check(ctx, wpos, wpos, None, ext, True, np.float32(196.0))
    # symmetric: j ∈ row i ⇔ i ∈ row j
    n = len(rp_g) - 1
    rows = np.repeat(np.arange(n), np.diff(rp_g.astype(np.int64)))
    a = set(zip(rows.tolist(), col_g.tolist()))
    assert all((j, i) in a for (i, j) in list(a)[:20000])


def test_neighbor_errors_and_empty(gpu):
    ctx = api.ForcesPositsGpu(4, 0, 10.0, 0.3)
    p = np.zeros((4, 3), np.float32)
    ext = np.full(3, 20.0, np.float32)
    with pytest.raises(api.DynError):
        ctx.build_neighbors(p, p, np.zeros(4, np.uint8), ext, False, 100.0)
    with pytest.raises(api.DynError):
        ctx.build_neighbors(p, p[:3], None, ext, True, 100.0)
    rp_g, col_g = ctx.build_neighbors(p, np.zeros((0, 3), np.float32), None, ext, False, 100.0)
    assert not rp_g.any() and col_g.size == 0


@pytest.mark.parametrize("n_outer,n_inner,ext,radius,spread", [
    (1, 1, 20.0, 6.0, 1.0), (70, 2047, 25.0, 6.0, 1.0), (70, 2048, 25.0, 9.0, 3.0),
    (300, 2049, 18.0, 6.0, 25.0),          # up to 12 boxes out: beyond the approximate test
    (500, 3000, 300.0, 12.0, 1.0),         # 15,625 cells
    (40, 140_000, 120.0, 8.0, 1.0),        # two ranges of indices
    (64, 4000, 11.0, 6.0, 2.0),            # one cell per axis, rows across the whole box
])
def test_neighbor_rows_sizes(gpu, n_outer, n_inner, ext, radius, spread):
    """Rows equal the brute-force lists at the edges of the bitmap's words
    and ranges, of the cell counts and of the approximate test, with points
    exactly at the threshold distance."""
    rng = np.random.default_rng(n_inner)
    mid, half = 0.5 * ext, 0.5 * ext * spread
    po = rng.uniform(mid - half, mid + half, (n_outer, 3)).astype(np.float32)
    pi = rng.uniform(mid - half, mid + half, (n_inner, 3)).astype(np.float32)
    k = min(n_outer, n_inner)
    pi[:k:3] = po[:k:3] + np.array([0, radius, 0], np.float32)
    e = np.full(3, ext, np.float32)
    print(f"neighbors: {n_outer} x {n_inner}, box {ext}, radius {radius}", flush=True)
    ctx = api.ForcesPositsGpu(n_outer, 0, 10.0, 0.3)
    _check(ctx, po, pi, None, e, False, np.float32(radius * radius))
    _check(ctx, po, po, (np.arange(n_outer) % 3 == 0).astype(np.uint8), e, True, np.float32(radius * radius))


@pytest.mark.parametrize("n_outer,n_inner,ext,radius", [
    (70, 32_768, 60.0, 6.0), (70, 32_769, 60.0, 6.0),  # bitmap and sort
    (40, 33_000, 30.0, 9.0),      # rows of nearly 4,096
    (200, 40_000, 1500.0, 10.0),  # rows of none to a few
    (64, 65_537, 120.0, 7.0),
])
def test_neighbor_rows_sorted(gpu, n_outer, n_inner, ext, radius):
    """Rows of many inner points, put in order by a sort, equal the
    brute-force lists; those of the bitmap's largest set too."""
    rng = np.random.default_rng(n_inner)
    po = rng.uniform(0, ext, (n_outer, 3)).astype(np.float32)
    pi = rng.uniform(0, ext, (n_inner, 3)).astype(np.float32)
    pi[:n_outer:3] = po[::3] + np.array([0, radius, 0], np.float32)
    e = np.full(3, ext, np.float32)
    print(f"neighbors: {n_outer} x {n_inner}, box {ext}, radius {radius}", flush=True)
    ctx = api.ForcesPositsGpu(n_outer, 0, 10.0, 0.3)
    _check(ctx, po, pi, None, e, False, np.float32(radius * radius))


def test_neighbor_total_beyond_32_bits(gpu):
    """More neighbours than row_ptr can count (1.25 million rows of about
    3,600) are refused."""
    n = 1_250_000
    rng = np.random.default_rng(3)
    p = (rng.random((n, 3), np.float32) * np.float32(60.0)).astype(np.float32)
    print("neighbors: total beyond 32 bits", flush=True)
    ctx = api.ForcesPositsGpu(16, 0, 10.0, 0.3)
    with pytest.raises(api.DynError):
        ctx.build_neighbors(p, p, None, np.full(3, 60.0, np.float32), True, 5.3 ** 2)
    row_ptr, col = ctx.build_neighbors(p[:100], p, None, np.full(3, 60.0, np.float32), False, 5.3 ** 2)
    assert row_ptr[-1] == col.size > 100 * 3000


def test_neighbor_many_inner_points(gpu):
    """Inner points beyond 2¹⁸ workgroups of 256 are sorted into cells too
    (68 million points, the last few around the outer ones)."""
    n, n_outer = 68_000_000, 64
    rng = np.random.default_rng(5)
    ext = np.full(3, 4000.0, np.float32)
    pi = rng.random((n, 3), np.float32)
    pi *= np.float32(4000.0)
    po = (2000.0 + 20.0 * rng.random((n_outer, 3))).astype(np.float32)
    pi[-200:] = (po[rng.integers(0, n_outer, 200)] + rng.normal(0, 1.0, (200, 3))).astype(np.float32)
    print("neighbors: 68 million inner points", flush=True)
    ctx = api.ForcesPositsGpu(n_outer, 0, 10.0, 0.3)
    row_ptr, col = ctx.build_neighbors(po, pi, None, ext, False, 16.0)
    near = np.flatnonzero((np.abs(pi - 2010.0) < 20.0).all(1))  # (far from the box faces)
    rp_o, col_o = rp.build_neighbors(po, np.ascontiguousarray(pi[near]), None, ext, False, np.float32(16.0))
    assert np.array_equal(row_ptr, rp_o) and np.array_equal(col, near[col_o])
    assert (col >= n - 200).any()

"""The panel kernels (lion-codes_amd/csrc/lup_panel.hpp) where they can go
wrong: sizes at the edges of their panels, row slots and matrices per wave,
columns whose criteria tie in the upper word or exactly, criteria outside the
corrected quotient's range, zero pivots and non-finite entries in the middle
of a panel.  Every compiled launch shape of each size equals the oracle's
mirror bit for bit (mantissa, exponent, pivots, status); a NaN mantissa need
only be NaN on both sides, and a zero determinant has no sign."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = (17, 20, 21, 24, 25, 28, 29, 31, 32, 33, 36, 37, 48, 49, 52, 53, 61, 63, 64)


def same(g, o):
    o = np.where(o == 0, 0.0 + 0.0j, o)  # a zero determinant is written as +0 + 0i
    g = np.ascontiguousarray(g).view(np.float64)
    o = np.ascontiguousarray(o).view(np.float64)
    return bool(((g.view(np.uint64) == o.view(np.uint64)) | (np.isnan(g) & np.isnan(o))).all())


def check(lc, orc, dev, A):
    n = A.shape[1]
    d = torch.from_numpy(np.ascontiguousarray(A)).to(dev)
    for policy in ("crout_ref", "abs"):
        o = orc.mirror(A, policy, "fused")
        keep = lc.get_shape(policy, "fused", n)
        try:
            for shape in range(lc.shape_count(n)):
                assert lc.set_shape(policy, "fused", n, shape | lc.SHAPE_PINNED)
                r = lc.det_batched(d, policy=policy, pivots=True)
                torch.cuda.synchronize()
                what = (n, policy, shape)
                assert np.array_equal(r.info.cpu().numpy(), o["info"]), what
                assert same(r.mant.cpu().numpy(), o["mant"]), what
                assert np.array_equal(r.exp.cpu().numpy(), o["exp"]), what
                ok = o["info"] >= 0
                assert np.array_equal(r.piv.cpu().numpy()[ok].astype(np.int32), o["piv"][ok]), what
        finally:
            lc.set_shape(policy, "fused", n, keep)


@pytest.mark.parametrize("n", SIZES)
def test_batches_that_do_not_fill_a_wave(lc, orc, wl, dev, n):
    for count in (1, 2, 3, 67):
        check(lc, orc, dev, wl.gaussian_np(count, n, seed=10 * n + count))


@pytest.mark.parametrize("n", SIZES)
def test_ties_and_zero_pivots(lc, orc, wl, dev, n):
    rng = np.random.default_rng(n)
    ints = rng.integers(-2, 3, (9, n, n)) + 1j * rng.integers(-2, 3, (9, n, n))
    ints[:, :, 0].real[:, ::2] = 2  # equal criteria in the first column
    perm = np.zeros((4, n, n), np.complex128)
    for m in range(4):
        perm[m, np.arange(n), rng.permutation(n)] = rng.choice([1, -1, 2, 1 + 1j], n)
    rank = ints[:3].copy()
    rank[0, :, n // 2] = rank[0, :, n // 2 - 1]  # zero pivots inside and at the ends of panels
    rank[1, n - 1] = rank[1, 0]
    rank[2, :, 5] = 0
    # upper words of the criteria equal, lower words deciding
    close = np.tile(wl.gaussian_np(3, 1, seed=n), (1, n, n)) * (1 + 1e-9 * rng.standard_normal((3, n, n)))
    check(lc, orc, dev, np.concatenate([ints, perm, rank, close]).astype(np.complex128))


@pytest.mark.parametrize("n", [17, 28, 32, 33, 48, 52, 64])
def test_criteria_outside_the_corrected_range(lc, orc, wl, dev, n):
    """Columns scaled so far down (with a large entry kept in each row) that
    their criteria need the division, rows above the reciprocal's range, and
    non-finite entries met inside a panel."""
    base = wl.gaussian_np(8, n, seed=4000 + n)
    A = base.copy()
    A[0][:, : n // 2] *= 2.0 ** -900
    A[1][:, 1::3] *= 2.0 ** -1000
    A[2] *= 2.0 ** 1000
    A[3][::2] *= 2.0 ** 970
    A[4][:, 6] *= 2.0 ** -1040
    A[5][n // 3, n - 2] = np.inf
    A[6][n // 2, 9] = complex(np.nan, 1.0)
    A[7][:, 3] = 0.0
    A[7][n - 1, 3] = 2.0 ** -950
    check(lc, orc, dev, A)


@pytest.mark.parametrize("n,limit", [(17, 1024), (20, 1024), (24, 1024), (25, 1024), (32, 1024),
                                     (49, 256), (53, 256), (57, 256), (60, 256), (64, 256)])
def test_small_batches(lc, orc, wl, dev, n, limit):
    """The low-latency kernels of batches that leave SIMDs idle, on both sides
    of the line where they end (256 compute units), in a padded layout."""
    base = wl.gaussian_np(64, n, seed=900 + n)
    base[0] = np.round(base[0])
    base[1] = np.round(base[1].real)
    base[2, :, 3] = 0
    base[3] *= 2.0 ** 980
    for policy in ("crout_ref", "abs"):
        o = orc.mirror(base, policy, "fused")
        keep = lc.get_shape(policy, "fused", n)
        for count in (1, 2, 64, limit, limit + 1):
            want = lc.SHAPE_SMALL_BATCH if count <= limit else keep
            assert lc.uniform_shape(policy, "fused", n, count) == want
            idx = np.arange(count) % 64
            A = torch.zeros(count, n, n + 3, dtype=torch.complex128, device=dev)
            A[:, :, :n] = torch.from_numpy(base[idx]).to(dev)
            r = lc.det_batched(A[:, :, :n], policy=policy, pivots=True)
            torch.cuda.synchronize()
            what = (n, policy, count)
            assert np.array_equal(r.info.cpu().numpy(), o["info"][idx]), what
            assert same(r.mant.cpu().numpy(), o["mant"][idx]), what
            assert np.array_equal(r.exp.cpu().numpy(), o["exp"][idx]), what
            ok = o["info"][idx] >= 0
            assert np.array_equal(r.piv.cpu().numpy()[ok].astype(np.int32), o["piv"][idx][ok]), what


@pytest.mark.parametrize("n", [17, 24, 32, 49, 57, 64])
def test_small_batches_built_on_the_device(lc, wl, dev, n):
    """The same kernels building their matrices from permuted positions (one
    permutation entry out of range) equal the pinned shape's."""
    rng = np.random.default_rng(n)
    z = torch.from_numpy(wl.fqhe_positions(n, rng)[None, :]).to(dev)
    perm = np.argsort(rng.random((9, n)), axis=1).astype(np.uint8)
    perm[4, n - 1] = n
    p = torch.from_numpy(perm).to(dev)
    assert lc.uniform_shape("crout_ref", "fused", n, 9) == lc.SHAPE_SMALL_BATCH
    small = lc.fqhe_det(z, row_perm=p, count=9, pivots=True)
    sh = lc.get_shape("crout_ref", "fused", n)
    try:
        assert lc.set_shape("crout_ref", "fused", n, sh | lc.SHAPE_PINNED)
        assert lc.uniform_shape("crout_ref", "fused", n, 9) == sh
        big = lc.fqhe_det(z, row_perm=p, count=9, pivots=True)
    finally:
        lc.set_shape("crout_ref", "fused", n, sh)
    torch.cuda.synchronize()
    assert small.info.cpu().tolist() == big.info.cpu().tolist()
    assert small.info[4].item() == -1000
    assert torch.equal(small.piv, big.piv) and torch.equal(small.exp, big.exp)
    assert same(small.mant.cpu().numpy(), big.mant.cpu().numpy())


def test_tuning_leaves_the_small_batch_kernels_on(lc, dev):
    """The tuner pins each shape while it times it, small counts included, and
    leaves its choice as the default."""
    from importlib import import_module
    tune = import_module("lion-codes_amd.autotune").tune
    try:
        table = tune(ns=[20, 32, 64], reps=1, count=96, log=lambda m: None)
        for e in table["entries"]:
            assert lc.get_shape(e["policy"], "fused", e["n"]) == e["shape"]
            assert lc.uniform_shape(e["policy"], "fused", e["n"], 48) == lc.SHAPE_SMALL_BATCH
    finally:
        lc.apply_shape_table()

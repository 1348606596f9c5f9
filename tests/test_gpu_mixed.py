"""GPU parity of mixed-size batches (one flat buffer, n = 1..64 per matrix).

Every mode -- one hipGraph replayed (own and class kernels), forked streams,
plain per-size launches, class kernels for every size -- must give the
oracle's determinants bit for bit at each matrix's own index. The graphs are
replayed several times with eager work and synchronisation in between; every
replay is checked.
"""
import numpy as np
import pytest
import torch

from conftest import bits

pytestmark = pytest.mark.gpu


def mixed_input(wl, count, seed, lo=1, hi=64):
    flat, ns, offs, sing = wl.mixed_batch(count, seed, n_lo=lo, n_hi=hi, near_singular=0.05)
    return flat, ns, offs


def check(orc, flat_np, ns, offs, res, policy):
    o = orc.mirror_mixed(flat_np, ns, offs, policy, "fused")
    assert np.array_equal(res.info.cpu().numpy(), o["info"])
    assert np.array_equal(bits(res.mant.cpu().numpy()), bits(o["mant"]))
    assert np.array_equal(res.exp.cpu().numpy(), o["exp"])


@pytest.mark.parametrize("policy", ["crout_ref", "abs"])
def test_mixed_modes_bit_exact(lc, orc, wl, dev, policy):
    flat, ns, offs = mixed_input(wl, 1500, seed=71)
    flat_np = flat.numpy()
    d = flat.to(dev)
    plan = lc.MixedPlan(ns, offs, policy=policy, nstreams=4)
    assert sorted(b[0] for b in plan.buckets()) == sorted(set(ns.tolist()))
    side = torch.cuda.Stream()
    for mode in ("plain", "streams", "graph", "persistent"):
        res = lc.alloc_result(len(ns), 64, dev)
        with torch.cuda.stream(side):
            plan.execute(d, res, mode=mode, stream=side)
        side.synchronize()
        check(orc, flat_np, ns, offs, res, policy)
    plan.close()


@pytest.mark.parametrize("mode", ["graph", "persistent"])
def test_graph_replays_with_eager_work_between(lc, orc, wl, dev, mode):
    flat, ns, offs = mixed_input(wl, 900, seed=5, lo=8, hi=64)
    flat_np = flat.numpy()
    d = flat.to(dev)
    plan = lc.MixedPlan(ns, offs, nstreams=3)
    res = lc.alloc_result(len(ns), 64, dev)
    side = torch.cuda.Stream()
    o = orc.mirror_mixed(flat_np, ns, offs, "crout_ref", "fused")
    for rep in range(4):
        res.mant.zero_()
        res.exp.fill_(-7)
        with torch.cuda.stream(side):
            plan.execute(d, res, mode=mode, stream=side)
        side.synchronize()
        # eager work of the program between replays
        x = torch.randn(1 << 16, device=dev).sum()
        torch.cuda.synchronize()
        assert np.array_equal(bits(res.mant.cpu().numpy()), bits(o["mant"])), rep
        assert np.array_equal(res.exp.cpu().numpy(), o["exp"]), rep
        del x
    plan.close()


def test_persistent_new_pointers_and_single_class(lc, orc, wl, dev):
    """Changing the output buffers or the mode captures the graph again, and
    switching back works; a batch whose sizes fall in two classes (n = 3..9)
    has two class launches in persistent mode, one with n = 1..64 five."""
    side = torch.cuda.Stream()
    for lo, hi, count in ((3, 9, 700), (1, 64, 1200)):
        flat, ns, offs = mixed_input(wl, count, seed=lo + hi, lo=lo, hi=hi)
        flat_np = flat.numpy()
        d = flat.to(dev)
        o = orc.mirror_mixed(flat_np, ns, offs, "crout_ref", "fused")
        plan = lc.MixedPlan(ns, offs, nstreams=2)
        launches, at = plan.launches("persistent")
        assert launches == (2 if hi == 9 else 5) and not any(own for _, own in at.values())
        r1 = lc.alloc_result(len(ns), 64, dev)
        r2 = lc.alloc_result(len(ns), 64, dev)
        for res, mode in ((r1, "persistent"), (r2, "persistent"), (r1, "graph"),
                          (r1, "persistent"), (r2, "streams"), (r2, "persistent")):
            res.mant.zero_()
            with torch.cuda.stream(side):
                plan.execute(d, res, mode=mode, stream=side)
            side.synchronize()
            assert np.array_equal(bits(res.mant.cpu().numpy()), bits(o["mant"])), (lo, mode)
            assert np.array_equal(res.exp.cpu().numpy(), o["exp"]), (lo, mode)
        plan.close()


def fill_line(lc, policy, n):
    """The fewest matrices of one size that fill the device's wave slots with
    the selected shape (8 waves per compute unit, 64 / lanes matrices each)."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    per_wave = 64 // lc.shape_info(n, lc.get_shape(policy, "fused", n))[0]
    return (8 * cus - 1) * per_wave + 1


def random_batch(sizes, counts, seed, dev):
    """Packed N(0,1) matrices, the sizes shuffled: (flat on the device, ns, offs)."""
    ns = np.repeat(np.array(sizes, np.int32), counts)
    np.random.default_rng(seed).shuffle(ns)
    offs = np.zeros(len(ns), np.int64)
    offs[1:] = np.cumsum(ns.astype(np.int64) ** 2)[:-1]
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    flat = torch.randn(int(offs[-1]) + int(ns[-1]) ** 2, 2, generator=g, dtype=torch.float64,
                       device=dev)
    return torch.view_as_complex(flat), ns, offs


def sample_check(orc, flat, ns, offs, res, policy, per_size=6):
    idx = np.sort(np.concatenate([np.nonzero(ns == n)[0][:per_size] for n in np.unique(ns)]))
    so = np.zeros(len(idx), np.int64)
    so[1:] = np.cumsum(ns[idx].astype(np.int64) ** 2)[:-1]
    sub = np.concatenate([flat[offs[i]:offs[i] + ns[i] ** 2].cpu().numpy() for i in idx])
    o = orc.mirror_mixed(sub, ns[idx], so, policy, "fused")
    assert np.array_equal(bits(res.mant.cpu().numpy()[idx]), bits(o["mant"]))
    assert np.array_equal(res.exp.cpu().numpy()[idx], o["exp"])


def assert_same_results(a, b, what):
    for f in ("mant", "exp", "logabs", "phase", "info"):
        x, y = getattr(a, f), getattr(b, f)
        if x.is_complex():
            x, y = torch.view_as_real(x), torch.view_as_real(y)
        if x.is_floating_point():
            x, y = x.view(torch.int64), y.view(torch.int64)
        assert torch.equal(x, y), (what, f)


@pytest.mark.parametrize("policy", ["crout_ref", "abs"])
def test_own_and_class_launches_of_one_plan(lc, orc, dev, policy):
    """Per class one size just below the fill line and one with a few matrices
    (a class launch), and one at the line (its own launch): every matrix has
    the bits of the per-size kernels."""
    below, line, few = (5, 11, 20, 38, 60), (6, 12, 21, 39, 61), (7, 13, 23, 40, 62)
    counts = [fill_line(lc, policy, n) - 1 for n in below]
    counts += [fill_line(lc, policy, n) for n in line] + [40] * 5
    flat, ns, offs = random_batch(below + line + few, counts, 17, dev)
    plan = lc.MixedPlan(ns, offs, policy=policy, nstreams=4)
    count, at = plan.launches("graph")
    assert count == 10 and len({a for a, _ in at.values()}) == 10
    for b, l, f in zip(below, line, few):
        assert at[b] == at[f] and not at[b][1] and at[l][1], (b, l, f)
    assert plan.launches("streams") == (count, at)
    plain_count, plain_at = plan.launches("plain")
    assert plain_count == 15 and all(own for _, own in plain_at.values())
    assert [plain_at[n][0] for n in sorted(plain_at, reverse=True)] == list(range(15))
    side = torch.cuda.Stream()
    want = lc.alloc_result(len(ns), 64, dev)
    with torch.cuda.stream(side):
        plan.execute(flat, want, mode="plain", stream=side)
    side.synchronize()
    sample_check(orc, flat, ns, offs, want, policy)
    shared, class_at = plan.launches("persistent")
    assert shared == 5 and not any(own for _, own in class_at.values())
    for mode in ("streams", "graph", "persistent"):
        res = lc.alloc_result(len(ns), 64, dev)
        res.mant.zero_()
        with torch.cuda.stream(side):
            plan.execute(flat, res, mode=mode, stream=side)
        side.synchronize()
        assert_same_results(res, want, mode)
    plan.close()


@pytest.mark.parametrize("policy", ["crout_ref", "abs"])
def test_a_size_alone_in_its_class_runs_its_own_kernel(lc, orc, dev, policy):
    """Small buckets that share a launch with nothing: one size of each class
    (and a single-size plan), beside a size that fills the device."""
    side = torch.cuda.Stream()
    for sizes, counts, launches in (((24,), (1000,), 1),
                                    ((8, 16, 24, 48, 64), (90, 70, 50, 30, 9), 5),
                                    ((30, 31), (50, fill_line(lc, policy, 31)), 2),
                                    ((57, 64, 20), (3, 5, 7), 2)):
        flat, ns, offs = random_batch(sizes, counts, sum(sizes), dev)
        plan = lc.MixedPlan(ns, offs, policy=policy, nstreams=3)
        count, at = plan.launches()
        assert count == launches
        assert all(own == (sizes != (57, 64, 20) or n == 20) for n, (_, own) in at.items())
        streams = {n: s for n, _, s in plan.buckets()}
        if 57 in streams:  # buckets of one launch are on its stream
            assert streams[57] == streams[64]
        want = lc.alloc_result(len(ns), 64, dev)
        res = lc.alloc_result(len(ns), 64, dev)
        with torch.cuda.stream(side):
            plan.execute(flat, want, mode="plain", stream=side)
            for _ in range(3):
                plan.execute(flat, res, mode="graph", stream=side)
        side.synchronize()
        assert_same_results(res, want, sizes)
        sample_check(orc, flat, ns, offs, res, policy)
        plan.close()


def test_mixed_graph_rejects_default_stream(lc, wl, dev):
    flat, ns, offs = mixed_input(wl, 10, seed=1, lo=4, hi=8)
    plan = lc.MixedPlan(ns, offs)
    res = lc.alloc_result(len(ns), 8, dev)
    with pytest.raises(lc.LufqheError):
        plan.execute(flat.to(dev), res, mode="graph", stream=torch.cuda.default_stream())
    plan.close()


def test_config4_full_size(lc, orc, wl, dev):
    """The mixed-size batch at full size: 200000 matrices, n ~ U{8..64}, 5% near-singular.
    Statuses clean, a sample bit-exact against the mirror, the rest against
    the long-double truth by matrix class."""
    flat, ns, offs, sing = wl.mixed_batch(200000, seed=2024, device=dev)
    plan = lc.MixedPlan(ns, offs, nstreams=4)
    res = lc.alloc_result(len(ns), 64, dev)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        plan.execute(flat, res, mode="graph", stream=side)
    side.synchronize()
    assert int((res.info != 0).sum()) == 0
    rng = np.random.default_rng(0)
    idx = np.sort(rng.choice(len(ns), 600, replace=False))
    sub_ns = ns[idx]
    sub_offs = np.zeros(len(idx), np.int64)
    sub_offs[1:] = np.cumsum(sub_ns.astype(np.int64) ** 2)[:-1]
    flat_cpu = flat.cpu().numpy()
    sub = np.concatenate([flat_cpu[offs[i]:offs[i] + ns[i] ** 2] for i in idx])
    o = orc.mirror_mixed(sub, sub_ns, sub_offs, "crout_ref", "fused")
    assert np.array_equal(bits(res.mant.cpu().numpy()[idx]), bits(o["mant"]))
    # the sizes' own kernels and the class kernels give the same bits for every matrix
    assert all(own for _, own in plan.launches("plain")[1].values())
    assert not any(own for _, own in plan.launches("persistent")[1].values())
    for mode in ("plain", "persistent"):
        rp = lc.alloc_result(len(ns), 64, dev)
        with torch.cuda.stream(side):
            plan.execute(flat, rp, mode=mode, stream=side)
        side.synchronize()
        assert_same_results(rp, res, mode)
    t = orc.truth_mixed(sub, sub_ns, sub_offs)
    la = res.logabs.cpu().numpy()[idx]
    ph = res.phase.cpu().numpy()[idx]
    err = np.abs(np.expm1((la - t["logabs"]) + 1j * np.angle(np.exp(1j * (ph - t["phase"])))))
    well = ~sing[idx]
    assert np.median(err[well]) < 1e-13 and np.quantile(err[well], 0.99) < 1e-10
    assert np.median(err[~well]) < 1e-6  # cond ~ 1e8: error ~ cond * eps
    plan.close()

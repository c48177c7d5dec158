"""Adjoint of the batched evaluation (tree and lists fixed) on the GPU.

1. Central finite differences (h = 1e-5, FP64 forward through the same lists
   with moments recomputed for the moved body) on 64 sampled coordinates and
   masses agree with the FP32 adjoint.
2. At N = 8192 the tree adjoint approximates the oracle's FP64 direct-sum
   gradient to the tree's own accuracy.
3. The torch.autograd.Function returns the same gradients, from CPU tensors
   through host arrays and from GPU tensors through the device entry points.
4. Two calls give bit-identical gradients (no atomics).
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _loss(plan, w4, variant="f64"):
    plan.evaluate(variant)
    return float((plan.result(variant) * w4).sum())


@pytest.mark.parametrize("mode", [1, 5])
def test_adjoint_matches_finite_differences(gpu_lib, mode):
    """mode 5: bisection groups, whose sinks the adjoint kernels read and write
    through the slot table."""
    from pgrav import batch, ics
    pos, mass = ics.clustered(6000, seed=31, nhalo=8)
    rng = np.random.default_rng(5)
    w4 = rng.normal(size=(pos.shape[0], 4))
    plan = batch.Plan(pos, mass, theta=0.6, order=4, eps=1e-3, soft="plummer", merge_groups=mode,
                      rcb_cell=1024)
    grad = plan.adjoint(w4)
    h = 1e-5
    picks = rng.choice(pos.shape[0], 16, replace=False)
    fd, ad = [], []
    for k in picks:
        for q in range(4):
            p1, p2 = pos.copy(), pos.copy()
            m1, m2 = mass.copy(), mass.copy()
            if q < 3:
                p1[k, q] += h
                p2[k, q] -= h
                step = h
            else:
                m1[k] *= 1 + h
                m2[k] *= 1 - h
                step = mass[k] * h
            plan.update(p1, m1)
            lp = _loss(plan, w4)
            plan.update(p2, m2)
            lm = _loss(plan, w4)
            fd.append((lp - lm) / (2 * step))
            ad.append(grad[k, q])
    plan.update(pos, mass)
    fd, ad = np.array(fd).reshape(-1, 4), np.array(ad).reshape(-1, 4)
    for q, name in ((slice(0, 3), "position"), (slice(3, 4), "mass")):
        scale = np.sqrt((fd[:, q] ** 2).mean())
        err = np.abs(ad[:, q] - fd[:, q]).max() / scale
        assert err < 2e-3, (name, err)
    plan.close()


def test_adjoint_approximates_direct_sum_gradient(gpu_lib):
    from pgrav import batch, ics
    pos, mass = ics.clustered(8192, seed=32, nhalo=8)
    rng = np.random.default_rng(6)
    w4 = rng.normal(size=(pos.shape[0], 4))
    eps = 2e-3
    plan = batch.Plan(pos, mass, theta=0.4, order=4, eps=eps, soft="plummer")
    grad = plan.adjoint(w4)
    ref = oracle.direct_grad(pos, mass, w4, soft_type=1, eps=eps)
    dx = np.linalg.norm(grad[:, :3] - ref[:, :3], axis=1) / np.linalg.norm(ref[:, :3], axis=1)
    dm = np.abs(grad[:, 3] - ref[:, 3]) / np.abs(ref[:, 3])
    assert np.median(dx) < 1e-3, np.median(dx)
    assert np.median(dm) < 1e-3, np.median(dm)
    plan.close()


def test_autograd_function(gpu_lib):
    import torch
    from pgrav import batch, ics
    from pgrav.autograd import gravity
    pos, mass = ics.clustered(4000, seed=33, nhalo=4)
    plan = batch.Plan(pos, mass, theta=0.6, order=4, eps=1e-3)
    w4 = np.random.default_rng(7).normal(size=(pos.shape[0], 4))
    tp = torch.tensor(pos, dtype=torch.float64, requires_grad=True)
    tm = torch.tensor(mass, dtype=torch.float64, requires_grad=True)
    acc = gravity(tp, tm, plan)
    loss = (acc.double() * torch.tensor(w4)).sum()
    loss.backward()
    ref = plan.adjoint(w4)
    # the same weights, the same fixed-order sums
    np.testing.assert_array_equal(tp.grad.numpy(), ref[:, :3])
    np.testing.assert_array_equal(tm.grad.numpy(), ref[:, 3])
    plan.close()


def test_adjoint_is_deterministic(gpu_lib):
    """Fixed-order sums, no atomics: two adjoint calls give identical gradients,
    also for K1 and unsoftened bodies and bisection groups."""
    from pgrav import batch, ics
    pos, mass = ics.clustered(12000, seed=34, nhalo=6)
    w4 = np.random.default_rng(8).normal(size=(pos.shape[0], 4))
    for soft, eps, mode in (("plummer", 1e-3, 1), ("k1", 2e-3, 5), ("none", 0.0, 5)):
        print("adjoint determinism soft=%s mode=%d" % (soft, mode), flush=True)
        plan = batch.Plan(pos, mass, theta=0.6, order=4, eps=eps, soft=soft, merge_groups=mode,
                          rcb_cell=2048)
        g1 = plan.adjoint(w4)
        g2 = plan.adjoint(w4)
        np.testing.assert_array_equal(g1, g2)
        assert np.isfinite(g1).all()
        plan.close()


def test_autograd_device_path_and_stale_plan(gpu_lib):
    """GPU tensors through the device entry points (no host copies) give the
    host path's gradients; a backward after a second forward on the same plan
    (other positions) still differentiates at its own forward's bodies."""
    import torch
    from pgrav import batch, ics
    from pgrav.autograd import gravity
    pos, mass = ics.clustered(5000, seed=35, nhalo=4)
    plan = batch.Plan(pos, mass, theta=0.6, order=4, eps=1e-3)
    rng = np.random.default_rng(9)
    w4 = rng.normal(size=(pos.shape[0], 4))
    pos2 = pos + rng.normal(size=pos.shape) * 1e-4
    ref1 = plan.adjoint(w4)  # the plan holds pos
    plan.update(pos2, mass)
    ref2 = plan.adjoint(w4)
    plan.evaluate("rel32c")
    acc2_ref = plan.result("rel32c")
    dev = torch.device("cuda")
    tw = torch.tensor(w4, dtype=torch.float32, device=dev)
    tp1 = torch.tensor(pos, dtype=torch.float64, device=dev, requires_grad=True)
    tm1 = torch.tensor(mass, dtype=torch.float64, device=dev, requires_grad=True)
    tp2 = torch.tensor(pos2, dtype=torch.float64, device=dev, requires_grad=True)
    tm2 = torch.tensor(mass, dtype=torch.float64, device=dev, requires_grad=True)
    acc1 = gravity(tp1, tm1, plan)
    acc2 = gravity(tp2, tm2, plan)  # the plan now holds pos2
    np.testing.assert_array_equal(acc2.detach().cpu().numpy(), acc2_ref.astype(np.float32))
    (acc1 * tw).sum().backward()  # must move the plan back to pos
    (acc2 * tw).sum().backward()
    w32 = w4.astype(np.float32).astype(np.float64)  # the device path's weights are float32
    np.testing.assert_allclose(tp1.grad.cpu().numpy(), plan_adjoint_at(plan, pos, mass, w32)[:, :3],
                               rtol=0, atol=0)
    np.testing.assert_allclose(tp2.grad.cpu().numpy(), plan_adjoint_at(plan, pos2, mass, w32)[:, :3],
                               rtol=0, atol=0)
    scale = np.abs(ref1[:, :3]).max()
    np.testing.assert_allclose(tp1.grad.cpu().numpy(), ref1[:, :3], rtol=0, atol=1e-5 * scale)
    np.testing.assert_allclose(tp2.grad.cpu().numpy(), ref2[:, :3], rtol=0, atol=1e-5 * scale)
    plan.close()


def plan_adjoint_at(plan, pos, mass, w4):
    plan.update(pos, mass)
    return plan.adjoint(w4)


@pytest.mark.parametrize("n,kw", [(3, dict(order=4, eps=0.05)), (70, dict(order=4, eps=0.05)),
                                  (6000, dict(order=0)), (6000, dict(order=2)),
                                  (6000, dict(order=4, merge_groups=5, rcb_cell=2048)),
                                  (6000, dict(order=4, mac="tolerance", errtol=0.05))])
def test_adjoint_along_a_direction(gpu_lib, n, kw):
    """Every list kind (cells of orders 0, 2, 4 and bodies), lists shorter than the
    waves that share them and longer: the gradient along a random direction against
    the central difference of the FP64 forward.  With steps h and h/2 combined the
    difference's own error is O(h^4); FP32 products leave a few 1e-7 of the summed
    terms' magnitude, and each body's pair with itself, m w / eps^3 taken with both
    signs, 2^-24 of that (eps keeps it below the bound)."""
    from pgrav import batch, ics
    pos, mass = ics.clustered(n, seed=41, nhalo=4)
    rng = np.random.default_rng(10)
    w4 = rng.normal(size=(n, 4))
    kw = dict(dict(theta=0.6, eps=5e-3, soft="plummer", leaf_max=8), **kw)
    plan = batch.Plan(pos, mass, **kw)
    grad = plan.adjoint(w4)
    dx, dm = rng.normal(size=(n, 3)), rng.normal(size=n) * 0.1

    def loss(h):
        plan.update(pos + h * dx, mass * (1 + h * dm))
        plan.evaluate("f64")
        return (plan.result("f64") * w4).sum()
    h = 2e-5
    d1 = (loss(h) - loss(-h)) / (2 * h)
    d2 = (loss(h / 2) - loss(-h / 2)) / h
    plan.close()
    fd = (4 * d2 - d1) / 3
    terms = np.concatenate([(grad[:, :3] * dx).ravel(), grad[:, 3] * mass * dm])
    assert abs(terms.sum() - fd) < 1e-4 * np.linalg.norm(terms), (terms.sum(), fd, np.linalg.norm(terms))


def test_unsoftened_sink_beside_the_group_centre(gpu_lib):
    """Three bodies in a row, one group: the middle one misses the centre by a rounding
    error, so that anything evaluated at the centre itself (a block's unused entries)
    overflows.  Against the FP64 direct gradient; one pair's FP32 products a few 2^-24."""
    from pgrav import batch
    pos, mass = np.array([[.1, .1, .1], [.4, .1, .1], [.7, .1, .1]]), np.array([.2, .3, .5])
    kw = dict(soft="none", eps=0.0, order=4)
    c = batch.HostPlan(pos, mass, **kw).group(0)[2]
    assert 0 < abs(c[0] - pos[1, 0]) < 1e-15
    w4 = np.random.default_rng(4).normal(size=(3, 4))
    plan = batch.Plan(pos, mass, **kw)
    grad = plan.adjoint(w4)
    plan.close()
    ref = oracle.direct_grad(pos, mass, w4, soft_type=0, eps=0.0)
    assert np.abs(grad - ref).max() < 64 * 2.0 ** -24 * np.abs(ref).max(), (grad, ref)


def _pair(r2, eps):
    """(phi, e, e') of a unit mass at distance sqrt(r2): a = e d, e' = 2 de/d(r2); Dehnen's
    K1 inside eps (0: none).  The pair at zero distance of an unsoftened body is 0."""
    f = np.where(r2 > 0, np.maximum(r2, 1e-300) ** -0.5, 0.0)
    phi, e, de = -f, -f ** 3, 3 * f ** 5
    if eps:
        u, near = r2 / eps ** 2 - 1, r2 <= eps ** 2
        phi = np.where(near, (((45 / 32 * u - 3 / 8) * u + 0.5) * u - 1) / eps, phi)
        e = np.where(near, ((-135 / 16 * u + 1.5) * u - 1) / eps ** 3, e)
        de = np.where(near, (-135 / 4 * u + 3) / eps ** 5, de)
    return phi, e, de


def _pair_gradients(d, m, w, eps):
    """J w - v a of pairs at d = sink - source; w the sinks' weights (w, v)."""
    _, e, de = _pair((d * d).sum(-1), eps)
    q = (d * w[..., :3]).sum(-1)
    return (m * e)[..., None] * (w[..., :3] - w[..., 3:] * d) + (m * de * q)[..., None] * d


@pytest.mark.parametrize("soft,eps", [("k1", 5e-3), ("none", 0.0)])
def test_k1_and_unsoftened_gradients(gpu_lib, soft, eps):
    """As the Plummer-softened test, against the FP64 direct sum: the tree's own error at
    theta 0.4, order 4 (K1: eps such that a body's pair with itself, 11 m w / eps^3, leaves
    less than that behind: 2^-24 x 2e4 beside gradients of 1e2)."""
    from pgrav import batch, ics
    n = 4096
    pos, mass = ics.clustered(n, seed=32, nhalo=8)
    w4 = np.random.default_rng(6).normal(size=(n, 4))
    plan = batch.Plan(pos, mass, theta=0.4, order=4, eps=eps, soft=soft)
    grad = plan.adjoint(w4)
    plan.close()
    ref = np.zeros((n, 4))
    for i in range(0, n, 256):
        d = pos[i:i + 256, None] - pos[None]
        p = _pair_gradients(d, mass[None], w4[i:i + 256, None], eps)
        ref[i:i + 256, :3] += p.sum(1)
        ref[:, :3] -= p.sum(0)
        phi, e, _ = _pair((d * d).sum(-1), eps)
        ref[:, 3] += (e * (d * w4[i:i + 256, None, :3]).sum(-1) + phi * w4[i:i + 256, None, 3]).sum(0)
    dx = np.linalg.norm(grad[:, :3] - ref[:, :3], axis=1) / np.linalg.norm(ref[:, :3], axis=1)
    dm = np.abs(grad[:, 3] - ref[:, 3]) / np.abs(ref[:, 3])
    assert np.median(dx) < 1e-3 and np.median(dm) < 1e-3, (np.median(dx), np.median(dm))


def test_adjoint_adds_in_its_stated_order(gpu_lib):
    """A sink's FP32 sum takes its cells, then its bodies, each in list order.  Softened
    closely, a body's pair with itself (11 m w / eps^3, K1) is larger than all others by
    1e7 until its source side cancels it, so that what is left depends on that order: the
    same sum in numpy, for one weighted sink at a time, whose gradient is then its own sum
    less that pair.  Every term after the own pair rounds on the pair's grid, a fifth of
    the terms; no body has another inside eps, so that the pair terms' 1e-7 hardly ever
    moves such a rounding, while another order moves three in ten of the sums.  (Masses and
    eps are powers of two and weights short, so that the own pair is exact, fused or not.)"""
    from pgrav import batch
    eps, f32, n = 2.0 ** -9, np.float32, 729
    rng = np.random.default_rng(3)
    pos = (np.stack(np.meshgrid(*[np.arange(9)] * 3, indexing="ij"), -1).reshape(-1, 3) +
           rng.uniform(0.3, 0.7, (n, 3))) / 9
    mass = np.full(n, 2.0 ** -10)
    kw = dict(theta=0.7, order=0, eps=eps, soft="k1", leaf_max=8, group_max=32)
    host = batch.HostPlan(pos, mass, **kw)
    perm, spos = host.sorted()
    w4 = np.round(rng.normal(size=(n, 4)) * 256) / 256
    plan = batch.Plan(pos, mass, **kw)
    same = []
    for g in range(host.stats()["ngroups"]):
        first, cnt, c = host.group(g)
        cells, bodies = [host.cell(k) for k in host.list(g, "mono")], host.list(g, "body")
        assert len(cells) and len(host.list(g, "hexa")) == 0
        for i in {first, first + cnt // 2}:
            w = w4[i]

            def terms(p, m, e):
                d = ((spos[i] - c[:3]).astype(f32) - (p - c[:3]).astype(f32)).astype(np.float64)
                return _pair_gradients(d, m.astype(f32).astype(np.float64), w, e).astype(f32)
            pc = terms(np.array([k["cofm"] for k in cells]), np.array([k["raw"][0] for k in cells]), 0)
            pb = terms(spos[bodies], mass[perm[bodies]], float(f32(eps)))
            own = pb[np.flatnonzero(bodies == i)[0]]
            want = np.zeros(3, f32)
            for t in np.concatenate([pc, pb]):
                want = want + t
            want = want - own
            one = np.zeros((n, 4))
            one[perm[i]] = w
            got = plan.adjoint(one)[perm[i], :3]
            same += list(np.abs(got - want) < 0.5 * np.spacing(np.abs(own)))
    plan.close()
    assert np.mean(same) > 0.93, np.mean(same)

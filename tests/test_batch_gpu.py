"""Parity of the batched path (pgrav_plan_*) on the GPU.

1. The exact lists of sampled groups are re-evaluated by the FP64 oracle (cell
   records rebuilt from each cell's bodies); the kernel variants must agree:
   FP64 to 1e-10, FP32 group-relative to 3e-6 (relative per sink, |da|/|a|).
2. The library's FP64 direct sum equals the oracle's FP64 direct sum (1e-12).
3. Graph replays, the persistent grid and the one-launch-per-group FP64
   dispatch reproduce the eager batched result.
"""
import numpy as np
import pytest

import listoracle
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup(gpu_lib):
    from pgrav import batch, ics
    pos, mass = ics.clustered(40000, seed=21, nhalo=24)
    return batch, ics, pos, mass


def _group_errors(batch, pos, mass, plan_kw, variants, ngroups=12, seed=0):
    plan = batch.Plan(pos, mass, **plan_kw)
    H = batch.HostPlan(pos, mass, **plan_kw)
    perm, spos = H.sorted()
    smass = mass[perm]
    out = {}
    for v in variants:
        plan.evaluate(v)
        out[v] = plan.result(v)[perm]  # back to sorted order
    st = H.stats()
    rng = np.random.default_rng(seed)
    errs = {v: [] for v in variants}
    for g in rng.choice(st["ngroups"], ngroups, replace=False):
        first, ref = listoracle.group_reference(H, int(g), spos, smass,
                                                soft=plan_kw.get("soft", "plummer"),
                                                eps=plan_kw.get("eps", 1e-4),
                                                G=plan_kw.get("G", 1.0))
        slots = H.group_slots(int(g))  # a run of bodies, or a bisection group's body set
        for v in variants:
            got = out[v][slots]
            da = np.linalg.norm(got[:, :3] - ref[:, :3], axis=1) / np.linalg.norm(ref[:, :3], axis=1)
            dp = np.abs(got[:, 3] - ref[:, 3]) / np.abs(ref[:, 3])
            errs[v].append(max(da.max(), dp.max()))
    plan.close()
    return {v: max(e) for v, e in errs.items()}


@pytest.mark.parametrize("soft,eps,mode", [("plummer", 1e-3, 1), ("k1", 2e-3, 1), ("none", 0.0, 1),
                                           ("plummer", 1e-3, 5), ("k1", 2e-3, 5)])
def test_batched_variants_match_oracle_on_same_lists(setup, soft, eps, mode):
    """Every variant against the oracle's FP64 evaluation of the group's own
    lists; mode 5: sink groups from coordinate bisection (body sets, read and
    written through the slot table)."""
    batch, ics, pos, mass = setup
    kw = dict(theta=0.6, order=4, eps=eps, soft=soft, G=1.0, merge_groups=mode, leaf_max=32,
              rcb_cell=4096)
    e = _group_errors(batch, pos, mass, kw, ["rel32c", "rel32", "f64", "abs32"])
    assert e["f64"] < 1e-10, e
    # FP32 sums of ~4000 terms per sink: a few 1e-6 relative
    assert e["rel32c"] < 1e-5, e
    assert e["rel32"] < 1e-5, e
    assert e["abs32"] < 1e-3, e  # absolute FP32 coordinates: the precision loss the
    #                             group-relative path removes


@pytest.mark.parametrize("mode", [1, 5])
def test_tolerance_mac_lists_match_oracle(setup, mode):
    """Lists of the error-tolerance acceptance (cells at orders 0, 2 and 4 mixed
    by their critical radii, nln/mac.c:1776-1800): every variant against the
    oracle's FP64 evaluation of the same lists."""
    batch, ics, pos, mass = setup
    kw = dict(order=4, eps=1e-3, soft="plummer", G=1.0, merge_groups=mode, leaf_max=32,
              rcb_cell=4096, mac="tolerance", errtol=0.1, frac_tol=0.02)
    st = batch.HostPlan(pos, mass, **kw).stats()
    assert min(st["pairs_hexa"], st["pairs_quad"], st["pairs_mono"]) > 0, st
    e = _group_errors(batch, pos, mass, kw, ["rel32c", "f64"])
    assert e["f64"] < 1e-10 and e["rel32c"] < 1e-5, e


def test_tolerance_mac_error_bound_on_gpu(setup):
    """Each sink's error against the FP64 direct sum stays below (cells listed) x
    errtol: every accepted cell's expansion error is within errtol."""
    batch, ics, pos, mass = setup
    errtol = 0.05
    kw = dict(order=4, eps=1e-3, soft="plummer", leaf_max=32, mac="tolerance", errtol=errtol,
              merge_groups=5, rcb_cell=4096)
    plan = batch.Plan(pos, mass, **kw)
    H = batch.HostPlan(pos, mass, **kw)
    plan.evaluate("rel32c")
    got = plan.result("rel32c")
    sample = np.random.default_rng(8).choice(pos.shape[0], 512, replace=False)
    ref = plan.direct(sample)
    plan.close()
    # cells listed for each sampled body's group
    perm, _ = H.sorted()
    inv = np.empty_like(perm)
    inv[perm] = np.arange(perm.size)
    off, slots = H.group_slot_table()
    group_of = np.empty(perm.size, np.int64)
    group_of[slots] = np.repeat(np.arange(off.size - 1), np.diff(off))
    ncell = sum(np.diff(H.csr(k)[0]) for k in ("hexa", "quad", "mono"))
    n_s = ncell[group_of[inv[sample]]]
    err = np.linalg.norm(got[sample, :3] - ref[:, :3], axis=1)
    # FP32 rounding adds ~1e-6 of |a| on top of the truncation bound
    assert np.all(err <= n_s * errtol + 1e-5 * np.linalg.norm(ref[:, :3], axis=1)), \
        (err / (n_s * errtol)).max()


@pytest.mark.parametrize("order", [2, 0])
def test_lower_orders_match_oracle(setup, order):
    batch, ics, pos, mass = setup
    kw = dict(theta=0.5, order=order, eps=1e-3, soft="plummer", G=2.0)
    e = _group_errors(batch, pos, mass, kw, ["rel32c", "f64"], ngroups=8)
    assert e["f64"] < 1e-10 and e["rel32c"] < 1e-5, e


def test_direct_sum_matches_oracle(setup):
    batch, ics, pos, mass = setup
    for soft, st, eps in (("plummer", 1, 1e-3), ("k1", 4, 3e-3), ("none", 0, 0.0)):
        plan = batch.Plan(pos, mass, eps=eps, soft=soft, G=1.5)
        sample = np.arange(0, pos.shape[0], 997)
        got = plan.direct(sample)
        ref = 1.5 * oracle.direct(pos[sample], pos, mass, soft_type=st, eps=eps)
        np.testing.assert_allclose(got, ref, rtol=1e-11, atol=0)
        plan.close()


def test_accuracy_against_direct_sum(setup):
    """Order-4 cells at theta = 0.5: the force error is the expansion error."""
    batch, ics, pos, mass = setup
    plan = batch.Plan(pos, mass, theta=0.5, order=4, eps=1e-4)
    plan.evaluate("rel32c")
    acc = plan.result("rel32c")
    sample = np.random.default_rng(3).choice(pos.shape[0], 1024, replace=False)
    da, dp = batch.rel_errors(acc[sample], plan.direct(sample))
    assert np.median(da) < 1e-4, np.median(da)
    assert np.percentile(da, 99) < 2e-3
    plan.close()


def test_graph_persistent_and_plain_dispatch_reproduce_eager(setup):
    batch, ics, pos, mass = setup
    plan = batch.Plan(pos, mass, theta=0.6, order=4, eps=1e-4)
    plan.evaluate("rel32c")
    eager = plan.result("rel32c")
    plan.graph_capture("rel32c")
    for rep in range(3):
        plan.evaluate("f64")  # unrelated eager work between replays
        plan.synchronize()
        plan.graph_launch()
        np.testing.assert_array_equal(plan.result("rel32c"), eager)
    plan.close()
    pers = batch.Plan(pos, mass, theta=0.6, order=4, eps=1e-4, persistent_blocks=-1)
    for rep in range(2):
        pers.evaluate("rel32c")
        np.testing.assert_array_equal(pers.result("rel32c"), eager)
    pers.graph_capture("rel32c")
    for rep in range(3):
        pers.graph_launch()
        np.testing.assert_array_equal(pers.result("rel32c"), eager)
    pers.evaluate("f64")
    f64 = pers.result("f64")
    pers.evaluate("plain64")
    plain = pers.result("plain64")
    np.testing.assert_allclose(plain, f64, rtol=1e-12, atol=1e-12 * np.abs(f64).max())
    pers.close()


@pytest.mark.parametrize("mode", [1, 5])
def test_unroll_variants_give_identical_results(setup, mode):
    """The autotuner's unroll choices (order-0 and body loops of rel32c) and the
    dispatch orders are the same arithmetic in the same order per group:
    bit-identical results, eager and from a graph, persistent (with its work
    stealing across XCD slices) and one workgroup per group."""
    batch, ics, pos, mass = setup
    plan = batch.Plan(pos, mass, theta=0.6, order=4, eps=1e-4, merge_groups=mode, rcb_cell=4096,
                      mac="tolerance", errtol=0.1)  # lists with order-0, 2, 4 cells and bodies
    st = plan.stats()
    assert min(st["pairs_mono"], st["pairs_body"]) > 0
    plan.evaluate("rel32c")
    want = plan.result("rel32c")
    for bu in (2, 8, 4):
        plan.set_unroll(bu)
        for pb in (0, -1):
            plan.set_launch(pb)
            plan.evaluate("rel32c")
            np.testing.assert_array_equal(plan.result("rel32c"), want)
    # the group orders (global longest-first; XCD slices ordered longest-first,
    # Morton, costliest-first then Morton) change only who evaluates a group when
    for mode in (0, 1, 3, 2):
        plan.set_dispatch(mode)
        plan.evaluate("rel32c")
        np.testing.assert_array_equal(plan.result("rel32c"), want)
    plan.set_unroll(8)
    plan.graph_capture("rel32c")
    for rep in range(2):
        plan.evaluate("f64")
        plan.synchronize()
        plan.graph_launch()
        np.testing.assert_array_equal(plan.result("rel32c"), want)
    from pgrav._lib import PgravError
    with pytest.raises(PgravError):
        plan.set_unroll(3)
    plan.close()


@pytest.mark.parametrize("mode,periodic", [(1, 0), (5, 0), (1, 2)])
def test_tile_variants(setup, mode, periodic):
    """The autotuner's tile (list entries per LDS round: 32, 64, 128) changes only
    where the compensated tile sums are folded: every tile matches the FP64
    evaluation of the same lists to FP32 accuracy, repeats bit for bit, eager and
    from a graph, and the periodic-1 kernels keep their 64."""
    batch, ics, pos, mass = setup
    kw = dict(order=4, eps=1e-3, merge_groups=mode, leaf_max=32, rcb_cell=4096, mac="tolerance",
              errtol=0.1, frac_tol=0.02)
    if periodic:
        p = (pos - pos.min(0)) / (np.ptp(pos, 0).max() * 1.001)
        kw.update(periodic="images", nimage=1, box=1.0)
    else:
        p = pos
    plan = batch.Plan(p, mass, **kw)
    plan.evaluate("f64")
    ref = plan.result("f64")
    out, err = {}, {}
    for tile in (32, 128, 64):
        plan.set_tile(tile)
        for pb in (0, -1):
            plan.set_launch(pb)
            plan.evaluate("rel32c")
            r = plan.result("rel32c")
            if tile in out:
                np.testing.assert_array_equal(r, out[tile])
            out[tile] = r
        da, _ = batch.rel_errors(out[tile], ref)
        dp = np.abs(out[tile][:, 3] - ref[:, 3]) / np.median(np.abs(ref[:, 3]))
        err[tile] = (np.percentile(da, 99.9), da.max(), dp.max())
    print("tile errors against f64 (99.9th pct and max |da|/|a|, max |dphi| / median |phi|):",
          err, flush=True)
    # every body (not sampled groups): the largest relative error sits at a sink
    # whose pull nearly cancels, the same body and size for every tile (the periodic
    # potential crosses zero, hence its scale)
    for tile, e in err.items():
        assert e[0] < 1e-5 and e[1] < 1e-4 and e[2] < 1e-5, (tile, err)
        assert e[1] < 1.5 * err[64][1] + 1e-6, (tile, err)
    plan.set_tile(128)
    plan.graph_capture("rel32c")
    for rep in range(2):
        plan.evaluate("f64")
        plan.synchronize()
        plan.graph_launch()
        np.testing.assert_array_equal(plan.result("rel32c"), out[128])
    from pgrav._lib import PgravError
    with pytest.raises(PgravError):
        plan.set_tile(96)
    plan.close()


def test_plan_rejects_bad_input(gpu_lib):
    from pgrav import batch
    from pgrav._lib import PgravError
    pos = np.random.default_rng(0).uniform(size=(100, 3))
    with pytest.raises(PgravError):
        batch.Plan(pos, np.full(100, 0.01), soft="plummer", eps=0.0)
    with pytest.raises(PgravError):
        batch.Plan(pos, np.full(100, 0.01), soft=3)


@pytest.mark.parametrize("n", [2, 65, 4095, 4096, 32767, 32768])
def test_shared_lists_match_oracle(setup, n):
    """Lists shared by 16, 8 or 4 waves of a workgroup, by the number of groups
    (one-body groups here: n of them, at each side of the rule's steps on 256 CUs),
    some lists shorter than the waves: FP32 and FP64 against the oracle's FP64
    evaluation of the same lists, and one launch shape bit for bit as the other."""
    batch, ics, _, _ = setup
    pos, mass = ics.clustered(n, seed=5, nhalo=8)
    kw = dict(theta=1.0, order=2, eps=1e-3, group_max=1, leaf_max=4, merge_groups=0)
    e = _group_errors(batch, pos, mass, kw, ["rel32c", "f64"], ngroups=min(n, 12))
    # FP32 offsets and a few hundred terms per sink, as above
    assert e["f64"] < 1e-10 and e["rel32c"] < 1e-5, e
    plan = batch.Plan(pos, mass, **kw)
    plan.evaluate("rel32c")
    want = plan.result("rel32c")
    plan.set_launch(0)
    plan.evaluate("rel32c")
    np.testing.assert_array_equal(plan.result("rel32c"), want)
    plan.close()


def _far_pays(st, ewald):
    # the rule of pgrav_plan.hip for 256 CUs (the Ewald kernel's too), by the lists' lengths;
    # of the work listed by the plans here 0.3 and more is far, where the rule asks for 0.2
    return 38 * st["entries_hexa"] + 8 * st["entries_quad"] > 6500 * st["ngroups"] + 4000 * 8192 \
        and (not ewald or st["ngroups"] >= 2 * 8192)


@pytest.mark.parametrize("kw", [
    dict(order=4, soft="plummer", eps=1e-3, merge_groups=1),
    dict(order=4, soft="plummer", eps=1e-3, merge_groups=5, rcb_cell=4096),
    dict(order=4, soft="none", eps=0.0, merge_groups=1),
    dict(order=4, soft="k1", eps=2e-3, merge_groups=1),
    dict(order=2, theta=0.3, soft="plummer", eps=1e-3, merge_groups=1),
    dict(order=4, soft="plummer", eps=1e-3, mac="tolerance", errtol=5e-4, quad_ncut=10,
         hexa_ncut=10, leaf_max=8),
    dict(order=4, theta=0.4, soft="plummer", eps=1e-3, periodic="images", nimage=1, box=1.0),
    dict(order=4, soft="plummer", eps=1e-3, periodic="ewald", box=1.0, group_max=4),
], ids=["plummer", "bisection", "unsoftened", "k1", "order2", "tolerance", "images", "ewald"])
def test_far_cells_match_the_pairs(gpu_lib, kw):
    """Plans whose far cells go through local expansions: FP32 against the batched FP64
    evaluation of the same lists (which takes every cell in pairs), on the plan's bodies
    and after they moved by a few group radii, where the far distance has to follow; and
    bit for bit the same from a graph and from either launch shape."""
    from pgrav import batch, ics
    pos, mass = ics.clustered(60000, seed=21, nhalo=24)
    pos = (pos - pos.min(0)) / (np.ptp(pos, 0).max() * 1.001)
    kw = dict(dict(theta=0.6, group_max=8, leaf_max=16), **kw)
    plan = batch.Plan(pos, mass, **kw)
    assert _far_pays(plan.stats(), kw.get("periodic") == "ewald"), plan.stats()
    rng = np.random.default_rng(3)
    for move in (0.0, 1e-3):
        if move:
            plan.update(pos + rng.normal(0, move, pos.shape), mass)
        plan.evaluate("f64")
        ref = plan.result("f64")
        for var in ("rel32c", "rel32"):
            plan.evaluate(var)
            got = plan.result(var)
            # an FP32 pair kernel's error: a few 1e-7 of the pulls' sum, which the
            # periodic images' partial cancellation raises against the result
            da = np.linalg.norm(got[:, :3] - ref[:, :3], axis=1)
            scale = np.linalg.norm(ref[:, :3], axis=1) + np.median(np.linalg.norm(ref[:, :3], axis=1))
            dp = np.abs(got[:, 3] - ref[:, 3]) / np.median(np.abs(ref[:, 3]))
            tol = 3e-5 if kw.get("periodic") else 3e-6
            assert np.percentile(da / scale, 99) < tol and np.percentile(dp, 99) < tol, \
                (var, move, np.percentile(da / scale, [50, 99, 100]), dp.max())
    plan.evaluate("rel32c")
    want = plan.result("rel32c")
    plan.set_launch(0)
    plan.evaluate("rel32c")
    np.testing.assert_array_equal(plan.result("rel32c"), want)
    plan.graph_capture("rel32c")
    for _ in range(3):
        plan.evaluate("f64")
        plan.synchronize()
        plan.graph_launch()
        np.testing.assert_array_equal(plan.result("rel32c"), want)
    plan.close()


@pytest.mark.parametrize("kw,edge", [
    (dict(order=4, soft="plummer", eps=1e-3, merge_groups=1, theta=0.7), (None, 64)),
    (dict(order=4, soft="plummer", eps=1e-3, merge_groups=5, rcb_cell=4096), None),
    (dict(order=4, soft="none", eps=0.0, merge_groups=1), None),
    (dict(order=4, soft="k1", eps=2e-3, merge_groups=1), None),
    (dict(order=2, theta=0.3, soft="plummer", eps=1e-3, merge_groups=1), None),
    (dict(order=4, soft="plummer", eps=1e-3, mac="tolerance", errtol=5e-4, quad_ncut=10, hexa_ncut=10,
          leaf_max=8), (1, 32)),
    (dict(order=4, theta=0.4, soft="plummer", eps=1e-3, periodic="images", nimage=1, box=1.0), None),
    (dict(order=4, soft="plummer", eps=1e-3, periodic="ewald", box=1.0, group_max=4), None),
], ids=["plummer", "bisection", "unsoftened", "k1", "order2", "tolerance", "images", "ewald"])
def test_far_cells_of_every_sink(gpu_lib, kw, edge):
    """The same plans, every sink's error: a few of 10,000 groups gone wrong are not in a
    percentile.  The far cells' truncation is below 1.4e-3 of a cell's pull at worst
    (test_local_expansion_cpu.py) and 1e-6 of the pulls here; beside it stands an FP32 pair
    kernel's error, largest where a sink has a neighbour
    much closer than its group's radius, unsoftened most of all (as in pairs: 1e-5, and the
    potential 3e-4 after a move).  `edge`: a list kind (or all cells) and the count at
    which the kernel's choice changes, which the groups' lists lie on both sides of."""
    from pgrav import batch, ics
    pos, mass = ics.clustered(60000, seed=21, nhalo=24)
    pos = (pos - pos.min(0)) / (np.ptp(pos, 0).max() * 1.001)
    kw = dict(dict(theta=0.6, group_max=8, leaf_max=16), **kw)
    if edge:
        host = batch.HostPlan(pos, mass, **kw)
        kind, at = edge
        n = sum(np.diff(host.csr(k)[0]) for k in (range(3) if kind is None else [kind]))
        assert all((n == at + d).sum() >= 5 for d in (-1, 0, 1)), [(n == at + d).sum() for d in (-1, 0, 1)]
    plan = batch.Plan(pos, mass, **kw)
    assert _far_pays(plan.stats(), kw.get("periodic") == "ewald"), plan.stats()
    soft = kw["soft"] == "plummer"
    rng = np.random.default_rng(3)
    for move in (0.0, 1e-3):
        if move:
            plan.update(pos + rng.normal(0, move, pos.shape), mass)
        plan.evaluate("f64")
        ref = plan.result("f64")
        a = np.linalg.norm(ref[:, :3], axis=1)
        for var in ("rel32c", "rel32"):
            plan.evaluate(var)
            got = plan.result(var)
            da = np.linalg.norm(got[:, :3] - ref[:, :3], axis=1) / (a + np.median(a))
            dp = np.abs(got[:, 3] - ref[:, 3]) / np.median(np.abs(ref[:, 3]))
            worst = (var, move, da.max(), dp.max())
            assert da.max() < (5e-6 if soft else 5e-5) and dp.max() < (1e-5 if soft else 1e-3), worst
    plan.close()


@pytest.mark.parametrize("size", [0.0, 1e-44, 1e-41, 1e-30, 1e-19, 1e-9])
def test_far_cells_of_a_vanishing_group(gpu_lib, size):
    """Eight bodies closer to one another than FP32 can tell, in a group of their own, among
    many: their results against FP64's (a few 1e-7 of the pulls' sum, as above)."""
    from pgrav import batch, ics
    pos, mass = ics.clustered(60000, seed=21, nhalo=24)
    pos = (pos - pos.min(0)) / (np.ptp(pos, 0).max() * 1.001)
    pos = np.concatenate([pos + 0.001, size * np.arange(8.0)[:, None] * [[1.0, 0.5, 0.25]]])
    plan = batch.Plan(pos, np.append(mass, np.full(8, mass[0])), theta=0.4, order=4, eps=1e-3,
                      group_max=8, leaf_max=16)
    assert _far_pays(plan.stats(), False)
    plan.evaluate("f64")
    ref = plan.result("f64")[-8:]
    for var in ("rel32c", "rel32"):
        plan.evaluate(var)
        got = plan.result(var)[-8:]
        np.testing.assert_allclose(got, ref, rtol=0, atol=3e-6 * np.abs(ref[:, :3]).max())
    plan.close()


def test_plans_that_expansions_do_not_pay_for(gpu_lib):
    """Groups of one body have no expansion, and a softening of the system's size no far
    cell (none is nearer than 100 eps).  Seen by the memory a plan takes: the expansions'
    workspace repeats the cell lists."""
    import torch
    from pgrav import batch, ics
    pos, mass = ics.clustered(80000, seed=21, nhalo=24)
    kw = dict(theta=0.4, order=4, leaf_max=16, merge_groups=0, fp64=False)

    def took(gmax, eps):
        free = torch.cuda.mem_get_info()[0]
        plan = batch.Plan(pos, mass, group_max=gmax, eps=eps, **kw)
        used, st = free - torch.cuda.mem_get_info()[0], plan.stats()
        plan.close()
        return used, st
    batch.Plan(pos[:1000], mass[:1000], **kw).close()  # the library's own start-up
    whole, st = took(8, 1e-3)
    lists = 4 * sum(st["entries_" + k] for k in ("hexa", "quad", "mono"))
    less, _ = took(8, 0.03)  # the same lists
    # (each allocation takes whole units of 2 MB)
    assert abs(whole - less - lists - 32 * st["n"]) < 16 * 2 ** 20, (whole, less, lists)
    one, st = took(1, 1e-3)
    lists = 4 * sum(st["entries_" + k] for k in ("hexa", "quad", "mono"))
    base = 4 * st["entries_body"] + lists + 48 * st["n"] + 96 * st["ngroups"] + 256 * st["nnodes"]
    assert one < base + 0.5 * lists, (one, base, lists)


def test_results_stay_whole_under_the_next_evaluation(gpu_lib):
    """A result read on one stream while the same bodies are evaluated again on another:
    the result array holds whole sums only, so every read gives the first one's values."""
    import torch
    from pgrav import batch, ics
    pos, mass = ics.clustered(60000, seed=21, nhalo=24)
    plan = batch.Plan(pos, mass, theta=0.6, order=4, eps=1e-3, group_max=8, leaf_max=16)
    assert _far_pays(plan.stats(), False)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    acc = torch.empty((8, 60000, 4), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    plan.evaluate("rel32c", stream=s1.cuda_stream)
    want = plan.result("rel32c")
    for k in range(8):
        plan.result_device("rel32c", acc[k].data_ptr(), stream=s2.cuda_stream)
        plan.evaluate("rel32c", stream=s1.cuda_stream)
    torch.cuda.synchronize()
    got = acc.cpu().numpy()
    plan.close()
    for k in range(8):
        np.testing.assert_array_equal(got[k], want.astype(np.float32))


@pytest.mark.parametrize("soft,eps", [("plummer", 1e-3), ("k1", 1e-3), ("none", 0.0)])
def test_fp64_source_beyond_the_range_of_its_square(gpu_lib, soft, eps):
    """A body so far that the FP64 square of its distance is infinite pulls with nothing,
    in the direct sum and in the batched and per-group FP64 kernels: the other bodies'
    results are those of a plan without it, up to the order of 48 terms."""
    from pgrav import batch
    rng = np.random.default_rng(6)
    pos = np.concatenate([rng.uniform(size=(48, 3)), [[3e154, 0.0, 0.0]]])
    mass = np.full(49, 1.0 / 49)
    got, want = [], []
    for out, n in ((got, 49), (want, 48)):
        plan = batch.Plan(pos[:n], mass[:n], order=0, pcut=1000, soft=soft, eps=eps, group_max=48)
        out.append(plan.direct(np.arange(n)))
        for v in ("f64", "plain64"):
            plan.evaluate(v)
            out.append(plan.result(v))
        plan.close()
    scale = np.abs(want[0]).max()
    for a, b in zip(got, want):
        np.testing.assert_allclose(a[:48], b, rtol=0, atol=1e-13 * scale)
        np.testing.assert_array_equal(a[48, :3], np.zeros(3))


@pytest.mark.parametrize("ns", [1, 15, 16, 17, 65, 1025])
def test_direct_sum_sample_sizes(setup, ns):
    """The FP64 direct sum for samples around the sizes of its blocks (16 sinks summed
    per workgroup, 64 evaluated), against the oracle: each of n = 40,000 terms carries a
    few rounding errors of 2^-53 and the sums' are below n 2^-53 of the summed pulls."""
    batch, ics, pos, mass = setup
    plan = batch.Plan(pos, mass, theta=0.8, order=0, eps=1e-3, fp64=False)
    sample = np.random.default_rng(ns).choice(pos.shape[0], ns, replace=False)
    got = plan.direct(sample)
    plan.close()
    ref = oracle.direct(pos[sample], pos, mass, soft_type=1, eps=1e-3)
    pull = np.abs(ref).max()
    assert np.abs(got - ref).max() < 4e4 * 2.0 ** -53 * pull, np.abs(got - ref).max() / pull

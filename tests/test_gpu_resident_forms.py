"""The resident propagation where a launch, a tiling or a batch takes another form than in
test_gpu_resident.py.

Checkpoints, kept units and the batch's split cut the same time steps of the same arithmetic
into other launches, so those comparisons are bit for bit.
"""
import numpy as np
import pytest
import torch

import cases
from conftest import gpu_available
from test_gpu_resident import _with_outside_receiver
from test_resident_plan import EXACT_FORMS, FP64_FORMS, STEP_FORMS

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.fixture(scope="module")
def O():
    from oracle import oracle as O_
    O_.load("oracle")
    return O_


@pytest.fixture(scope="module")
def psv():
    from fwi_cuda_amd import psv as P
    return P


def _obs(c, seed=5):
    """Observed rows of about the synthetics' size."""
    n = len(c["z_rec"]) * int(c["nshot"])
    rng = np.random.default_rng(seed)
    t = np.arange(int(c["nt"]))
    w = np.exp(-(((t - 0.4 * c["nt"]) / (0.1 * c["nt"] + 1)) ** 2))
    return [1e-13 * rng.standard_normal((n, 1)) * w for _ in range(2)]


def _ran(sim, kind, want):
    """The context takes the tiling that the form is there for (on 256 compute units)."""
    t = sim.resident_tiling(kind=kind)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert {k: t[k] for k in want} == want, t
    assert t["shots"] > 0


# nz, nx, order, shots: several tiles of the one-exchange kernel, a last unit of one step
ONE_STEP = [(90, 140, 8, 2), (91, 139, 10, 3), (201, 401, 8, 1), (97, 133, 12, 1), (233, 32, 12, 6)]


@pytest.mark.parametrize("nt", [1, 2, 61])
@pytest.mark.parametrize("form", ONE_STEP, ids=lambda f: f"{f[0]}x{f[1]}-o{f[2]}x{f[3]}")
def test_one_step_launches_bitwise(psv, O, form, nt):
    """Launches of a single time step (a last unit of one step, units of one step, a record of
    one step) give the bits of one launch over all steps."""
    nz, nx, order, ns = form
    c = cases.small_case(O, nz=nz, nx=nx, nt=nt, fdorder=order, nshot=ns, snap_dt=1)
    obs = _obs(c)
    out = []
    for kw in (dict(storage=psv._lib.STORE_FULL), dict(storage=psv._lib.STORE_CHECKPOINT, ckpt_interval=12, ckpt_keep=1),
               dict(storage=psv._lib.STORE_CHECKPOINT, ckpt_interval=1, ckpt_keep=1),
               dict(storage=psv._lib.STORE_CHECKPOINT, ckpt_interval=4, ckpt_keep=2, ckpt_slots=3)):
        with psv.Simulation(c, **kw) as sim:
            for kind in ("step", "exact_forward"):
                _ran(sim, kind, dict(cells=0))
            seis = sim.forward()
            wf = sim.wavefield(0, "szx")
            sim.set_observed(*obs)
            m = sim.gradient()
            out.append((*seis, wf, m, *sim.get_gradient(), *sim.misfit_gradient(*obs), *sim.misfit_gradient_exact(*obs)))
        print(f"{form} nt {nt} {kw}", flush=True)
    assert nt < 61 or all(np.abs(a).max() > 0 for a in out[0])
    for o in out[1:]:
        for i, (a, b) in enumerate(zip(o, out[0])):
            np.testing.assert_array_equal(a, b, err_msg=str(i))


def test_tuned_once_per_context(psv, O):
    """The stencil kernel is tuned once: batches of other sizes (11 shots as 4 + 4 + 3, sub-ranges)
    keep the choice, also after a context with a pinned variant has tuned the same sizes."""
    c = cases.small_case(O, nz=89, nx=143, nt=20, nshot=11, snap_dt=1)
    with psv.Simulation(c, batch=4, work_order=1) as sim:   # a pinned order: launch by launch
        sim.set_observed(*_obs(c))
        sim.forward()
        log = sim.tuning()[1]
        assert log.startswith("chosen") and log.count("o0/v5/tz16/d1 ") == 1
        for other in (1, 2):   # one of them at least is not its choice
            with psv.Simulation(c, batch=4, kernel_variant=other) as pinned:
                pinned.forward(0, 3)
                pinned.forward(0, 4)
            for call in (lambda: sim.forward(0, 3), lambda: sim.gradient(0, 4), lambda: sim.gradient(), lambda: sim.misfit()):
                call()
                assert sim.tuning()[1] == log


@pytest.mark.parametrize("first", ["forward", "gradient"])
def test_two_batches_tune_once_each(psv, O, first):
    """Where a forward pass takes more shots at once than a gradient, each of the two batches is
    tuned once, whichever comes first, for kernels whose misfits compare exactly."""
    c = cases.small_case(O, nz=500, nx=700, nt=40, nshot=8, snap_dt=1)
    obs = _obs(c)
    with psv.Simulation(c, storage=psv._lib.STORE_FULL, kernel_variant=5) as sim:
        budget = int(0.6 * sim.plan()["device_bytes"])
    with psv.Simulation(c, mem_budget=budget, work_order=1) as sim:   # a pinned order: launch by launch
        p = sim.plan()
        assert p["gradient_batch"] < p["batch"] and sim.resident_tiling()["shots"] == 0
        sim.set_observed(*obs)
        heads = {}
        for k in range(2):
            for what in (first, *{"forward", "gradient"} - {first}):
                m = sim.gradient() if what == "gradient" else sim.misfit()
                if what == "gradient":
                    total = sum(m.tolist())
                else:
                    misfit = m
                head, *log = sim.tuning()[1].split("; ")
                assert heads.setdefault(what, head) == head
            if k == 0:
                timed = log
        assert total == misfit
        for call in (lambda: sim.forward(0, 3), lambda: sim.gradient(0, 2), lambda: sim.forward()):
            call()
            assert sim.tuning()[1].split("; ")[1:] == timed
        one_pass = [int(h.split("/v")[1].split("/")[0]) in (4, 7, 8, 9) for h in heads.values()]
        assert one_pass[0] == one_pass[1]
        print(first, heads, len(timed), flush=True)


def test_gradient_batch_smaller_than_forward_batch(psv, O):
    """With storage and batch left open and memory for part of the snapshots, a gradient runs in
    smaller batches than a forward pass: same bits as contexts whose one batch holds all shots or
    that number of shots, and the misfit of a gradient is that of a forward pass."""
    c = cases.small_case(O, nz=500, nx=700, nt=40, nshot=8, snap_dt=1)
    kw = dict(kernel_variant=5, tile_tz=16, work_order=1)
    full = dict(storage=psv._lib.STORE_FULL)
    with psv.Simulation(c, **kw, **full) as sim:
        total = sim.plan()["device_bytes"]
        sim.set_model(1.05 * c["lam"], 1.05 * c["mu"], c["rho"])
        obs = sim.forward()
    adj = _obs(c)

    def run(**opts):
        with psv.Simulation(c, **opts) as sim:
            plan = sim.plan()
            seis = sim.forward()
            sim.set_observed(*obs)
            m = sim.gradient()
            assert sum(m.tolist()) == sim.misfit()
            G, mg = sim.get_gradient(), sim.misfit_gradient(*adj)
            raw = sim.gradient_raw(*adj)
            sim.zero_gradient()
            try:   # its outcome, a step or the search's "no step" exit, and the misfit there
                it = sim.fwi_iteration()
            except psv._lib.FwiError as e:
                it = e.status
            return (*seis, m, *G, *mg, *raw), plan, (it, sim.misfit())

    for part in (0.9, 0.8, 0.7, 0.6, 0.5):
        budget = int(part * total)
        with psv.Simulation(c, mem_budget=budget, **kw) as sim:
            plan = sim.plan()
        print(part, plan, flush=True)
        if plan["gradient_batch"] < plan["batch"] and plan["storage"] == "full":
            break
    assert plan["gradient_batch"] < plan["batch"] and plan["device_bytes"] <= budget
    bg = plan["gradient_batch"]
    out, p, it = run(mem_budget=budget, **kw)
    assert p == plan
    for opts in (full, dict(full, batch=bg), dict(storage=psv._lib.STORE_CHECKPOINT, batch=3)):
        ref, rp, rit = run(**kw, **opts)
        assert rp["gradient_batch"] == rp["batch"] and it == rit
        for i, (a, b) in enumerate(zip(out, ref)):
            np.testing.assert_array_equal(a, b, err_msg=f"{opts} output {i}")
    out, p, it = run(mem_budget=budget)   # tuned kernel
    assert p == plan
    np.testing.assert_allclose(out[2], ref[2], rtol=1e-5)


def test_gradient_batch_over_budgets(psv, O):
    """The planner's choices over a range of budgets, smaller batches that still checkpoint among
    them: the bits of one fully stored batch, within the budget."""
    c = cases.small_case(O, nz=500, nx=700, nt=100, nshot=16, snap_dt=1)
    obs = _obs(c)
    kw = dict(kernel_variant=5, tile_tz=16, work_order=1)
    with psv.Simulation(c, storage=psv._lib.STORE_FULL, **kw) as sim:
        total = sim.plan()["device_bytes"]
        sim.set_observed(*obs)
        want = (sim.gradient(), *sim.get_gradient())
    seen = set()
    for k in range(25, 60):
        budget = int(0.01 * k * total)
        try:
            sim = psv.Simulation(c, mem_budget=budget, **kw)
        except psv._lib.FwiError as e:
            assert e.status == -2
            continue
        with sim:
            p = sim.plan()
            key = (p["gradient_batch"], p["batch"], p["storage"])
            if key in seen:
                continue
            seen.add(key)
            print(k, p, flush=True)
            assert p["device_bytes"] <= budget
            sim.set_observed(*obs)
            got = (sim.gradient(), *sim.get_gradient())
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b, err_msg=str(p))
    assert {s for g, b, s in seen if g < b} == {"full", "checkpoint"}


def test_exact_workspace_counted_and_within_budget(psv, O):
    """The exact adjoint's workspace stays within mem_budget, is counted by plan(), and a kept one
    changes neither the next call's result nor its size."""
    c = cases.small_case(O, nz=90, nx=140, nt=300, nshot=3, snap_dt=1)
    adj = _obs(c)
    with psv.Simulation(c) as sim:
        before = sim.plan()["device_bytes"]
        a = sim.misfit_gradient_exact(*adj)
        held = sim.plan()["device_bytes"]
        assert held - before > 5 * 4 * 90 * 140 * 300 * 3   # the intermediates of every step
        b = sim.misfit_gradient_exact(*adj)
        assert sim.plan()["device_bytes"] == held
    budget = before + (65 << 20)   # the planner's reserve, and less than the workspace
    with psv.Simulation(c, mem_budget=budget) as sim:
        d = sim.misfit_gradient_exact(*adj)
        assert sim.plan()["device_bytes"] <= budget
    for x, y, z in zip(a, b, d):
        assert np.abs(x).max() > 0
        np.testing.assert_array_equal(y, x)
        np.testing.assert_array_equal(z, x)


# nz, nx, order, shots, steps, free surface: calls on 1, 2, ... of the shots take tilings of their
# own; the waves are inside the CPML strips before the record ends
TILINGS = [(246, 335, 8, 6, 250, True), (246, 335, 8, 3, 250, False), (301, 601, 4, 5, 150, False),
           (90, 140, 12, 3, 300, False), (91, 139, 2, 2, 300, True), (89, 131, 6, 2, 300, False),
           (93, 121, 10, 2, 300, True), (800, 1400, 8, 1, 100, True)]


@pytest.mark.parametrize("form", TILINGS, ids=lambda f: f"{f[0]}x{f[1]}-o{f[2]}-{'surface' if f[5] else 'cpml'}")
def test_results_do_not_depend_on_the_tiling(psv, O, form):
    """One shot beside others (adjoint sources of the first shot only), alone, and by variant 5's
    launches: seismograms, fields, correlation sums and misfit derivative bit for bit, the exact
    gradient over the tilings."""
    nz, nx, order, ns, nt, surf = form
    c = cases.small_case(O, nz=nz, nx=nx, nt=nt, fdorder=order, nshot=ns, surface=surf, snap_dt=2)
    n = len(c["z_rec"])
    obs = _obs(c)
    ref = None
    for v in (0, 5):
        with psv.Simulation(c, kernel_variant=v) as sim:
            for k in range(1, ns + 1) if v == 0 else (ns,):
                adj = [np.concatenate([o[:n], np.zeros((n * (k - 1), nt))]) for o in obs]
                out = [s[:n] for s in sim.forward(0, k)]
                out += [sim.wavefield(0, f) for f in ("vz", "vx", "szz", "szx", "sxx", "We")]
                out += [*sim.gradient_raw(*adj, 0, k), *sim.misfit_gradient(*adj, 0, k)]
                out += [*sim.misfit_gradient_exact(*adj, 0, k)]
                ref = ref or out
                for i, (a, b) in enumerate(zip(out, ref)):
                    assert np.abs(b).max() > 0
                    np.testing.assert_array_equal(a, b, err_msg=f"variant {v}, {k} shots, output {i}: {cases.rel_l2(a, b):.1e}")
                print(f"{form} variant {v} {k} shots", flush=True)


# nz, nx, shots, steps whose intermediates take more than the 8 GiB that stay with a context, and
# the shots asked for
GROUPED = [(246, 335, 3, 2500, (3, 2)), (90, 140, 7, 8000, (7, 5))]


@pytest.mark.parametrize("form", GROUPED, ids=lambda f: f"{f[0]}x{f[1]}x{f[2]}")
def test_exact_grouped_shots_and_segments(psv, O, form):
    """Records that exceed the kept workspace run in segments and in batches of shots that share
    launches: the workspace stays bounded, and every call gives the bits of the unsegmented sweep."""
    nz, nx, ns, nt, counts = form
    c = cases.small_case(O, nz=nz, nx=nx, nt=nt, nshot=ns, snap_dt=1)
    n = len(c["z_rec"])
    adj = _obs(c)
    kw = dict(storage=psv._lib.STORE_CHECKPOINT, ckpt_keep=1)   # a small context
    out = {}
    with psv.Simulation(c, **kw) as sim:                       # the interval is left open
        base = sim.plan()["device_bytes"]
        for k in (*counts, *counts):
            g = sim.misfit_gradient_exact(*[a[:n * k] for a in adj], 0, k)
            held = sim.plan()["device_bytes"] - base
            print(form, "shots", k, "held", held >> 20, "MiB", flush=True)
            assert 0 < held <= (8 << 30) + (16 << 20)          # its output buffer and edge words beside it
            for a, b in zip(g, out.setdefault(k, g)):
                np.testing.assert_array_equal(a, b)
    with psv.Simulation(c, ckpt_interval=nt, **kw) as sim:
        for k in counts:
            for a, b in zip(sim.misfit_gradient_exact(*[a[:n * k] for a in adj], 0, k), out[k]):
                assert np.abs(a).max() > 0
                np.testing.assert_array_equal(b, a)


def _form_case(O, form, nt):
    nz, nx, order, ns, surf, npml = form
    return cases.small_case(O, nz=nz, nx=nx, nt=nt, fdorder=order, nshot=ns, surface=surf, snap_dt=2,
                            npml=max(npml, order // 2))


def _ids(f):
    return f"{f[0][0]}x{f[0][1]}-o{f[0][2]}x{f[0][3]}"


@pytest.mark.parametrize("form", [f for f in STEP_FORMS if f[1].get("shots") != 0], ids=_ids)
def test_step_forms_equal_variant5(psv, O, form):
    """Every kernel and tiling of the FP32 steps, among them the two-exchange kernel of one cell per
    thread on several tiles, tiles thinner than the frame, a single tile and CPML memories in LDS
    and in memory: forward and adjoint bit for bit variant 5."""
    c = _form_case(O, form[0], 120)
    obs = _obs(c)
    out = []
    for v in (5, 0):
        with psv.Simulation(c, kernel_variant=v) as sim:
            if v == 0:
                _ran(sim, "step", form[1])
            seis = sim.forward()
            fields = [sim.wavefield(0, f) for f in ("vz", "szx", "We")]
            sim.set_observed(*obs)
            m = sim.gradient()
            out.append((*seis, *fields, m, sim.wavefield(int(c["nshot"]) - 1, "We_adj"), *sim.get_gradient(),
                        *sim.misfit_gradient(*obs)))
            assert v == 0 or sim.resident_tiling()["shots"] == 0
    for i, (a, b) in enumerate(zip(*out)):
        assert np.abs(a).max() > 0
        np.testing.assert_array_equal(b, a, err_msg=f"output {i}: {cases.rel_l2(b, a):.1e}")


@pytest.mark.parametrize("form", FP64_FORMS, ids=_ids)
def test_fp64_forms_match_kernels(psv, O, form):
    """Every tiling of the FP64 propagation against its one-thread-per-cell kernels."""
    c = _form_case(O, form[0], 100)
    d, rows, _ = _with_outside_receiver(c)
    with psv.Simulation(c, seis_fp64=1) as sim:
        _ran(sim, "fp64", form[1])
        a = sim.forward()
    with psv.Simulation(d, seis_fp64=1) as sim:
        assert sim.resident_tiling(kind="fp64")["shots"] == 0
        b = sim.forward()
    for x, y in zip(a, b):
        assert np.linalg.norm(y[rows]) > 0 and cases.rel_l2(x, y[rows]) < 1e-12


@pytest.mark.parametrize("form", EXACT_FORMS, ids=_ids)
def test_exact_forms_match_kernels(psv, O, form):
    """Every tiling of the exact adjoint's reverse sweep against its one-thread-per-cell kernels."""
    c = _form_case(O, form[0], 60)
    d, rows, n = _with_outside_receiver(c)
    obs = _obs(c)
    ext = [np.zeros((n, int(c["nt"]))) for _ in range(2)]
    for e, o in zip(ext, obs):
        e[rows] = o
    with psv.Simulation(c) as sim:
        _ran(sim, "exact", form[1])
        a = sim.misfit_gradient_exact(*obs)
    with psv.Simulation(d) as sim:
        assert sim.resident_tiling(kind="exact")["shots"] == 0
        b = sim.misfit_gradient_exact(*ext)
    for i, (x, y) in enumerate(zip(a, b)):
        print(f"{form[0]} part {i}: {cases.rel_l2(x, y):.2e}", flush=True)
        assert np.linalg.norm(y) > 0 and cases.rel_l2(x, y) < 1e-5


def test_outgrown_edge_words_are_given_back(psv, O):
    """A context that has run ever more shots at once holds the memory of one that ran them all."""
    c = cases.small_case(O, nz=246, nx=335, nt=20, nshot=6, snap_dt=1)
    held = []
    for counts in ((1, 2, 3, 6), (6,)):
        with psv.Simulation(c) as sim:
            for k in counts:
                out = sim.forward(0, k)
            held.append((sim.plan()["device_bytes"], out))
    assert held[0][0] == held[1][0]
    for a, b in zip(held[0][1], held[1][1]):
        np.testing.assert_array_equal(a, b)


def test_without_the_finite_check(psv, O):
    """check_finite 0 leaves the results of every pass as they are."""
    c = cases.small_case(O, nz=90, nx=140, nt=150, nshot=3, snap_dt=1)
    obs = _obs(c)
    out = []
    for on in (1, 0):
        with psv.Simulation(c, check_finite=on, seis_fp64=1) as sim:
            sim.set_observed(*obs)
            out.append((*sim.forward(), sim.wavefield(1, "vz"), sim.gradient(), *sim.get_gradient(), sim.misfit(),
                        *sim.misfit_gradient(*obs), *sim.misfit_gradient_exact(*obs)))
    for a, b in zip(*out):
        np.testing.assert_array_equal(b, a)


def test_contexts_on_several_threads(psv, O):
    """Contexts that run resident launches at the same time, each on its own thread and stream,
    beside one that goes launch by launch: the results of one after the other."""
    import threading
    forms = [(90, 140, 8, 2, {}), (246, 335, 8, 3, {}), (301, 601, 4, 2, {}), (90, 140, 8, 2, dict(kernel_variant=5))]
    work = []
    for nz, nx, order, ns, kw in forms:
        c = cases.small_case(O, nz=nz, nx=nx, nt=150, fdorder=order, nshot=ns, snap_dt=1)
        work.append((psv.Simulation(c, **kw), _obs(c)))

    def run(sim, obs):
        sim.set_observed(*obs)
        sim.zero_gradient()
        return (*sim.forward(), sim.gradient(), *sim.get_gradient(), *sim.misfit_gradient_exact(*obs))

    want = [run(*w) for w in work]
    got, errors = [[] for _ in work], []

    def loop(i):
        try:
            for _ in range(4):
                got[i].append(run(*work[i]))
        except Exception as e:   # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=loop, args=(i,)) for i in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for sim, _ in work:
        sim.close()
    assert not errors, errors
    for w, runs in zip(want, got):
        assert len(runs) == 4
        for r in runs:
            for a, b in zip(r, w):
                np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("stf_type", [0, 1])
@pytest.mark.parametrize("form", [(90, 140, 8, 3), (246, 335, 8, 2), (246, 335, 4, 3), (321, 611, 4, 5)],
                         ids=lambda f: f"{f[0]}x{f[1]}-o{f[2]}x{f[3]}")
def test_points_of_any_number_and_place(psv, O, form, stf_type):
    """Shots with several sources and receivers of their own, some in one cell, some on the first and
    last cells of the interior and of tiles: bit for bit variant 5, units of one step included."""
    nz, nx, order, ns = form
    N = order // 2
    c = cases.small_case(O, nz=nz, nx=nx, nt=61, fdorder=order, nshot=ns, snap_dt=1)
    rng = np.random.default_rng(nz + order + stf_type)
    with psv.Simulation(c) as sim:
        t = sim.resident_tiling()
    edge_z = [N, nz - N - 1, min(N + t["rows"], nz - N - 1), min(N + t["rows"] - 1, nz - N - 1)]
    edge_x = [N, nx - N - 1, min(N + t["cols"], nx - N - 1), min(N + t["cols"] - 1, nx - N - 1)]
    z, x, fire, zr, xr, off = [], [], [], [], [], [0]
    for s in range(ns):
        z += [N + 3 + s, N + 3 + s, *edge_z[:3], int(rng.integers(N, nz - N))]
        x += [nx // 2, nx // 2, *edge_x[1:], int(rng.integers(N, nx - N))]
        fire += [s] * 6
        zr += [N + 3 + s, N + 3 + s, *edge_z, N + 1][s:]   # shot s has 7 - s receivers
        xr += [nx // 2, nx // 2, *edge_x, nx // 2 + 2][s:]
        off.append(len(zr))
    w = rng.uniform(-1.0, 1.0, (2, len(z), 1)) * c["stf_z"][:1]
    c.update(z_src=np.array(z, np.int32), x_src=np.array(x, np.int32), shot_to_fire=np.array(fire, np.int32),
             stf_z=np.ascontiguousarray(w[0]), stf_x=np.ascontiguousarray(w[1]), stf_type=stf_type,
             z_rec=np.array(zr, np.int32), x_rec=np.array(xr, np.int32), rec_off=np.array(off, np.int32))
    obs = [1e-13 * rng.standard_normal((off[-1], 61)) for _ in range(2)]
    out = []
    for kw in (dict(kernel_variant=5), {}, dict(storage=psv._lib.STORE_CHECKPOINT, ckpt_interval=12, ckpt_keep=1)):
        with psv.Simulation(c, **kw) as sim:
            assert (sim.resident_tiling()["shots"] > 0) == ("kernel_variant" not in kw)
            seis = sim.forward()
            sim.set_observed(*obs)
            out.append((*seis, sim.gradient(), *sim.get_gradient(), *sim.misfit_gradient(*obs),
                        *sim.misfit_gradient_exact(*obs)))
    for o in out[1:]:
        for i, (a, b) in enumerate(zip(o, out[0])):
            assert np.abs(b).max() > 0
            np.testing.assert_array_equal(a, b, err_msg=f"output {i}")

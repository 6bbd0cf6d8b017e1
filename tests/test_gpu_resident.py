"""The resident propagation (one launch per range of time steps) against the launch-by-launch
kernels of the same library.

The stencil arithmetic is variant 5's, so seismograms, snapshots and fields are compared with
that variant at the tolerance between two variants of one stencil, rel-L2 1e-6 (FP32 rounding
of differently contracted sums), and gradients and misfit-derivative sums at 1e-4; the FP64
propagation against its one-thread-per-cell kernels at 1e-12, the exact adjoint's sweep
against its kernels at 1e-5 (FP32 states over the same operations).  Where a kernel cannot be
pinned, a receiver outside the interior (which the resident kernels do not take) selects the
other path; it records zero and its residual is zero.  Sizes reach every number of cells
per thread, tiles with short last rows and columns, a single tile, several launches per batch
and CPML memory in registers, LDS and memory.
"""
import numpy as np
import pytest

import cases
from conftest import gpu_available

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
    """Observed rows of about the synthetics' size (any rows do: both paths get the same)."""
    n = int(np.asarray(c["rec_off"])[-1]) if "rec_off" in c else len(c["z_rec"]) * int(c["nshot"])
    rng = np.random.default_rng(seed)
    t = np.arange(int(c["nt"]))
    w = np.exp(-(((t - 0.4 * c["nt"]) / (0.1 * c["nt"])) ** 2))
    return [1e-13 * rng.standard_normal((n, 1)) * w for _ in range(2)]


# nz, nx, order, shots, steps, free surface, snapshot strides: what the tiling gives on 256 CUs
FORMS = [
    (17, 23, 8, 2, 90, True, (1, 1, 1)),        # one small tile, strips that meet
    (90, 140, 2, 2, 150, True, (2, 1, 1)),      # 1 cell per thread, orders 2 to 12
    (90, 140, 6, 2, 150, False, (3, 1, 1)),
    (91, 139, 10, 3, 150, True, (2, 2, 3)),
    (97, 133, 12, 1, 150, False, (1, 3, 2)),
    (246, 335, 8, 3, 120, True, (3, 1, 1)),     # 2
    (321, 611, 4, 5, 80, False, (2, 1, 1)),     # 4, more than one launch per batch
    (800, 1400, 8, 1, 70, True, (3, 1, 1)),     # 8, CPML memory in LDS
]


def _case(O, nz, nx, order, ns, nt, surf, snap):
    npml = 6 if nz < 40 else 12
    c = cases.small_case(O, nz=nz, nx=nx, nt=nt, fdorder=order, nshot=ns, surface=surf, npml=max(npml, order // 2))
    s = list(c["snap"])
    s[4:7] = snap
    s[1] -= (s[1] - s[0]) % snap[1]
    s[3] -= (s[3] - s[2]) % snap[2]
    c["snap"] = type(c["snap"])(s) if isinstance(c["snap"], (tuple, list)) else np.asarray(s, np.int32)
    return c


@pytest.mark.parametrize("form", FORMS, ids=lambda f: f"{f[0]}x{f[1]}-o{f[2]}x{f[3]}")
def test_resident_steps_match_variant5(psv, O, form):
    c = _case(O, *form)
    snap = form[6]
    obs = _obs(c)
    out = {}
    for v in (5, 0):
        with psv.Simulation(c, kernel_variant=v, storage=psv._lib.STORE_FULL) as sim:
            seis = sim.forward()
            wf = sim.wavefield(0, "szx")
            _, snaps = sim.forward_snapshots(0)
            sim.set_observed(*obs)
            m = sim.gradient()
            G = sim.get_gradient()
            mg = sim.misfit_gradient(*obs) if snap[1:] == (1, 1) else ()
            out[v] = (*seis, wf, *(snaps[k] for k in sorted(snaps)), *G, *mg), m, len(snaps)
            assert v == 5 or sim.tuning()[1] == ""   # nothing was tuned: the resident kernels ran
    n = 3 + out[5][2]
    np.testing.assert_allclose(out[0][1], out[5][1], rtol=1e-5)
    for i, (a, b) in enumerate(zip(out[0][0], out[5][0])):
        e = cases.rel_l2(a, b)
        print(f"{form} output {i}: {e:.2e}", flush=True)
        assert e < (1e-6 if i < n else 1e-4), (i, e)


@pytest.mark.parametrize("form", [FORMS[1], FORMS[5], FORMS[6]], ids=lambda f: f"{f[0]}x{f[1]}")
def test_resident_storage_modes_bitwise(psv, O, form):
    """A range cut at checkpoints and kept units gives the bits of one uncut range."""
    c = _case(O, *form[:4], 150, *form[5:])
    obs = _obs(c)
    res = []
    sdt = form[6][0]
    for kw in (dict(storage=psv._lib.STORE_FULL), dict(storage=psv._lib.STORE_CHECKPOINT, ckpt_interval=12 * sdt, ckpt_keep=2),
               dict(storage=psv._lib.STORE_CHECKPOINT, ckpt_interval=7 * sdt, ckpt_slots=2, use_graph=1)):
        with psv.Simulation(c, **kw) as sim:
            sim.set_observed(*obs)
            m = sim.gradient()
            res.append((m, *sim.get_gradient()))
    for r in res[1:]:
        for a, b in zip(r, res[0]):
            np.testing.assert_array_equal(a, b)


def _with_outside_receiver(c):
    """The case with one more receiver per shot at cell (0, 0), outside the interior."""
    d = dict(c)
    ns = int(c["nshot"])
    off = np.asarray(c["rec_off"]) if "rec_off" in c else np.arange(ns + 1) * len(c["z_rec"])
    zr, xr = np.asarray(c["z_rec"]), np.asarray(c["x_rec"])
    if "rec_off" not in c:
        zr, xr = np.tile(zr, ns), np.tile(xr, ns)
    z, x, o, rows = [], [], [0], []
    for s in range(ns):
        z += [*zr[off[s]:off[s + 1]], 0]
        x += [*xr[off[s]:off[s + 1]], 0]
        rows += list(range(len(z) - 1 - (off[s + 1] - off[s]), len(z) - 1))
        o.append(len(z))
    d["z_rec"], d["x_rec"], d["rec_off"] = np.asarray(z, np.int32), np.asarray(x, np.int32), np.asarray(o, np.int32)
    return d, np.asarray(rows), o[-1]


FP64_FORMS = [FORMS[0], FORMS[1], FORMS[3], FORMS[5], (321, 611, 8, 3, 60, True, (2, 1, 1)),
              (600, 1100, 8, 1, 60, False, (2, 1, 1))]


@pytest.mark.parametrize("form", FP64_FORMS, ids=lambda f: f"{f[0]}x{f[1]}-o{f[2]}x{f[3]}")
def test_resident_fp64_matches_kernels(psv, O, form):
    c = _case(O, *form)
    d, rows, _ = _with_outside_receiver(c)
    with psv.Simulation(c, seis_fp64=1) as sim:
        a = sim.forward()
    with psv.Simulation(d, seis_fp64=1) as sim:
        b = sim.forward()
    for i in range(2):
        e = cases.rel_l2(a[i], b[i][rows])
        print(f"{form} component {i}: {e:.2e}", flush=True)
        assert e < 1e-12


EXACT_FORMS = [FORMS[0], FORMS[1], FORMS[3], FORMS[4], (246, 335, 8, 3, 60, True, (1, 1, 1)),
               (301, 601, 4, 5, 50, False, (1, 1, 1)), (500, 900, 8, 1, 50, True, (1, 1, 1))]


@pytest.mark.parametrize("interval", [0, 13])
@pytest.mark.parametrize("form", EXACT_FORMS, ids=lambda f: f"{f[0]}x{f[1]}-o{f[2]}x{f[3]}")
def test_resident_exact_adjoint_matches_kernels(psv, O, form, interval):
    """The reverse sweep in one launch, with all intermediates held or segments of 13 steps
    recomputed, against the kernels that run where a receiver lies outside the interior."""
    c = _case(O, *form[:6], (form[6][0], 1, 1))
    d, rows, n = _with_outside_receiver(c)
    obs = _obs(c)
    ext = [np.zeros((n, int(c["nt"]))) for _ in range(2)]
    for e, o in zip(ext, obs):
        e[rows] = o
    kw = dict(storage=psv._lib.STORE_CHECKPOINT, ckpt_interval=interval) if interval else {}
    with psv.Simulation(c, **kw) as sim:
        a = sim.misfit_gradient_exact(*obs)
    with psv.Simulation(d) as sim:
        b = sim.misfit_gradient_exact(*ext)
    for i in range(3):
        e = cases.rel_l2(a[i], b[i])
        print(f"{form} interval {interval} part {i}: {e:.2e}", flush=True)
        assert np.linalg.norm(b[i]) > 0 and e < 1e-5

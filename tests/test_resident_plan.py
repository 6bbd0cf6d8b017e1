"""The rule that splits a grid for the resident propagation (no device needed): every tiling holds
what the kernels assume of it, and the forms that the GPU tests name take the kernels they name.
"""
import random
import sys

import numpy as np
import pytest

from conftest import ROOT

# nz, nx, order, shots, free surface, CPML cells: cells per thread on 256 compute units, and more of
# the tiling where a test is there for it
STEP_FORMS = [
    ((17, 23, 8, 2, True, 6), dict(cells=1, tiles_z=1, tiles_x=1)),       # a single tile
    ((90, 140, 2, 2, True, 12), dict(cells=0)),                           # one exchange per step
    ((90, 140, 6, 2, False, 12), dict(cells=0)),
    ((91, 139, 10, 3, True, 12), dict(cells=0)),
    ((97, 133, 12, 1, False, 12), dict(cells=0)),
    ((28, 104, 10, 2, False, 12), dict(cells=0, rows=1)),                 # tiles thinner than the frame
    ((233, 32, 12, 6, True, 12), dict(cells=0, cols=10)),
    ((246, 335, 8, 2, True, 12), dict(cells=1, tiles_z=11, tiles_x=11)),  # two exchanges
    ((301, 601, 8, 1, False, 12), dict(cells=1, tiles_z=13, tiles_x=19)),
    ((246, 335, 8, 3, True, 12), dict(cells=2, shots=3)),
    ((246, 335, 8, 6, True, 12), dict(cells=4, shots=6, psi_lds=1)),
    ((321, 611, 4, 5, False, 12), dict(cells=4, shots=5)),
    ((440, 597, 12, 3, True, 40), dict(cells=4, shots=3, psi_lds=0)),     # CPML memory in memory
    ((800, 1400, 8, 1, True, 12), dict(cells=8, psi_lds=1)),
    ((600, 1100, 8, 8, True, 12), dict(shots=0)),                         # the batched kernels are as fast
    ((1001, 2001, 8, 1, True, 12), dict(shots=0)),                        # does not fit
]
FP64_FORMS = [
    ((17, 23, 8, 2, True, 6), dict(cells=1, tiles_z=1, tiles_x=1)),
    ((90, 140, 2, 2, True, 12), dict(cells=1, shots=2)),
    ((91, 139, 10, 3, True, 12), dict(cells=1, shots=3)),
    ((246, 335, 8, 3, True, 12), dict(cells=2)),
    ((321, 611, 8, 3, True, 12), dict(cells=1, shots=1)),                 # three launches
    ((399, 1183, 8, 1, True, 12), dict(cells=4, psi_lds=1)),
    ((600, 1100, 8, 1, False, 12), dict(cells=4, psi_lds=0)),
]
EXACT_FORMS = [
    ((17, 23, 8, 2, True, 6), dict(cells=1, tiles_z=1, tiles_x=1)),
    ((90, 140, 2, 2, True, 12), dict(cells=1, shots=2)),
    ((91, 139, 10, 3, True, 12), dict(cells=1, shots=3)),
    ((97, 133, 12, 1, False, 12), dict(cells=1)),
    ((246, 335, 8, 3, True, 12), dict(cells=2, shots=3)),
    ((301, 601, 4, 5, False, 12), dict(cells=2, shots=2)),
    ((500, 900, 8, 1, True, 12), dict(cells=2)),
    ((560, 1000, 8, 1, True, 12), dict(cells=4)),                         # carries in LDS
]


def strips(nz, nx, N, top, npml):
    """Strip numbers of the CPML's rows at the bottom, and at the top, and of its columns."""
    z, x = np.full(nz, -1, np.int32), np.full(nx, -1, np.int32)
    zi = [i for i in range(N, nz - N) if (top and i < npml) or i >= nz - N - npml - 1]
    xi = [i for i in range(N, nx - N) if i < npml or i >= nx - N - npml - 1]
    z[zi], x[xi] = np.arange(len(zi)), np.arange(len(xi))
    return z, x


@pytest.mark.parametrize("kind,forms", [("step", STEP_FORMS), ("fp64", FP64_FORMS), ("exact", EXACT_FORMS)])
def test_forms_take_the_kernels_they_name(kind, forms):
    from fwi_cuda_amd import psv
    for (nz, nx, order, ns, surf, npml), want in forms:
        z, x = strips(nz, nx, order // 2, not surf, npml)
        t = psv.plan_tiling(nz, nx, order, ns, kind, 256, z, x)
        assert {k: t[k] for k in want} == want, (nz, nx, order, ns, t)


def test_tilings_hold_what_the_kernels_assume():
    """Random grids, orders, shots, strips and device sizes, against the limits the kernels are
    written for: a block per tile and compute unit, threads for every cell, tiles of at least N
    rows and columns where only neighbours are read, at most four edge values (two cells of the
    frame) per thread, LDS that holds the fields and the strips' memories."""
    from fwi_cuda_amd import psv
    r = random.Random(3)
    count = {}
    for _ in range(6000):
        N = r.randint(1, 6)
        nz, nx = (max(2 * N + 1, int((2 * N + 1) * (top / (2 * N + 1)) ** r.random())) for top in (1100, 1600))
        ns, cus, npml, top = r.randint(1, 9), r.choice((256, 256, r.randint(1, 304))), r.randint(0, 40), r.random() < 0.5
        kind = r.choice(("step", "fp64", "exact_forward", "exact"))
        z, x = strips(nz, nx, N, top, npml)
        t = psv.plan_tiling(nz, nx, 2 * N, ns, kind, cus, z, x)
        if t["shots"] == 0:
            continue
        at = (kind, nz, nx, N, ns, cus, npml, top, t)
        cells, TZ, TX, ntz, ntx, thr = (t[k] for k in ("cells", "rows", "cols", "tiles_z", "tiles_x", "threads"))
        count[kind, cells] = count.get((kind, cells), 0) + 1
        iz, ix, elt = nz - 2 * N, nx - 2 * N, 8 if kind == "fp64" else 4
        lastz, lastx = iz - (ntz - 1) * TZ, ix - (ntx - 1) * TX
        assert 1 <= t["shots"] <= ns and t["shots"] * ntz * ntx <= cus and thr % 64 == 0 and thr <= 1024, at
        assert 0 < lastz <= TZ and 0 < lastx <= TX and t["lds"] <= 160 * 1024, at
        if cells == 0:
            assert kind in ("step", "exact_forward") and ntz * ntx > 1, at
            assert TX + 2 * N <= 32 and 32 * (TZ + 2 * N) <= thr and (TX + 4 * N) * (TZ + 4 * N) <= 2 * thr, at
            assert t["lds"] >= 4 * (2 * (32 + 2 * N) * (TZ + 4 * N) + (3 * 32 + 6) * (TZ + 2 * N)), at
            continue
        lanes = 64 if cells >= 4 and elt == 4 else 32
        assert cells in ((1, 2, 4) if kind in ("fp64", "exact") else (1, 2, 4, 8)), at
        assert TX <= lanes and TZ % cells == 0 and lanes * TZ // cells <= thr, at
        assert (ntz == 1 or min(TZ, lastz) >= N) and (ntx == 1 or min(TX, lastx) >= N), at
        assert (4 * N * TX if ntz > 1 else 0) + (4 * N * TZ if ntx > 1 else 0) <= 4 * thr, at
        rows = max(int((z[a:min(a + TZ, nz - N)] >= 0).sum()) for a in range(N, nz - N, TZ))
        cols = max(int((x[a:min(a + TX, nx - N)] >= 0).sum()) for a in range(N, nx - N, TX))
        need = elt * ((4 if kind == "exact" else 5) * (lanes + 2 * N) * (TZ + 2 * N) + 6 * TZ) + 4 * TZ
        if t["psi_lds"]:
            assert t["psi_rows"] >= rows and t["psi_cols"] >= cols, at
            need += 4 * elt * (t["psi_rows"] * TX + t["psi_cols"] * TZ)
        assert t["lds"] >= need, at
    reached = {("exact_forward", c) for c in (0, 1, 2, 4, 8)} | {(k, c) for k in ("fp64", "exact") for c in (1, 2, 4)}
    assert reached <= set(count), count


def test_plan_tiling_refuses_bad_arguments():
    from fwi_cuda_amd import _lib, psv
    for args in ((8, 40, 8, 1), (40, 8, 8, 1), (40, 40, 7, 1), (40, 40, 14, 1), (40, 40, 8, 0)):
        with pytest.raises(_lib.FwiError) as e:
            psv.plan_tiling(*args)
        assert e.value.status == -1
    with pytest.raises(_lib.FwiError):
        psv.plan_tiling(40, 40, 8, 1, cus=0)


def test_bench_reports_resident_launches_per_time_step():
    """bench.py makes no HBM bandwidth of launches that keep their fields on the chip: it names the
    resident kernel and gives the time of a time step."""
    sys.path.insert(0, str(ROOT))
    import bench
    t = dict(cells=0, shots=2)
    r = bench.resident_report(t, 4, 6.8, 10, 5, 20000)
    assert r["instantiation"] == "k_resident1<4, *>" and r["us_per_time_step"] == 3.4 and r["tiling"] is t
    assert r["achieved"] is r["frac"] is r["peak"] is None
    for cells, name in ((1, "k_resident<float, 6, 1, 32, *>"), (4, "k_resident<float, 6, 4, 64, *>")):
        assert bench.resident_report(dict(t, cells=cells), 6, 1.0, 1, 1, 100)["instantiation"] == name

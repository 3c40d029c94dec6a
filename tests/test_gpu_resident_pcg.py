"""The resident PCG (one launch per refinement) against the two-kernel form
(taken for iteration caps above 16384), on the same systems, each side in the
form that its size and cap ask for: one workgroup and several, one and four
slots per wave around the sizes where the layout changes (2048 slots with
MIC(0), 3072 with Jacobi), rows of a wave and waves of a workgroup that hold
no slot, one to three waves per SIMD and both register budgets, and one slot
more than fits (both are then the two-kernel form).  Both solve to the same
FP64 residual; with the same rounding of every vector update they take the
same iterations up to the last few, and their pressures differ by the solver's
tolerance times a factor for the operator's condition, far below 1e-4."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MOST = 11264  # slots that fit the chip: 256 CUs, eleven waves of four slots


def _bricks(n, seed):
    """Grid and particles (one per cell, a few cells left empty) of n bricks
    stacked x, y, z in a box that holds them, the last layer partly filled."""
    side = max(1, int(np.ceil(n ** (1 / 3))))
    rng = np.random.default_rng(seed)
    b = np.arange(n)
    bx, by, bz = b % side, (b // side) % side, b // (side * side)
    c = np.arange(512)
    i = (bx[:, None] * 8 + (c & 7)).reshape(-1)
    j = (by[:, None] * 8 + ((c >> 3) & 7)).reshape(-1)
    k = (bz[:, None] * 8 + (c >> 6)).reshape(-1)
    size = 8 * side
    h = np.float32(1.0 / size)
    keep = rng.random(i.size) > 0.05
    pos = [((a[keep] + 0.5) * h).astype(np.float32) for a in (i, j, k)]
    vel = [rng.uniform(-1, 1, pos[0].size).astype(np.float32) for _ in range(3)]
    return (0.0, 0.0, 0.0, size, size, size, 1.0 / size), pos, vel


@pytest.mark.parametrize("prec", ["jacobi", "mic0"])
@pytest.mark.parametrize("n", [1, 4, 5, 16, 17, 63, 1000, 1025, 2048, 2049, 3072, 3073, 4096, 4101, 8192, 8195, 11264, 11265])
def test_resident_matches_two_kernel_form(flip2, n, prec):
    grid, pos, vel = _bricks(n, n)
    got = []
    for cap in (4000, 20000):
        sim = flip2.FluidSim(pos[0].size, grid, preconditioner=prec, max_iterations=cap)
        sim.set_particles(*pos, *vel)
        print(f"resident PCG: {n} bricks, {prec}, cap {cap}", flush=True)
        for stage in ("transfer_prepare", "system"):
            sim.stage(stage)
        resident = n <= MOST and cap == 4000
        s = sim.solve_with(prec)
        form = sim.solve_form()
        assert form == {"resident_refinements": s["refinements"] if resident else 0, "give_ups": 0}, form
        again = sim.solve_with(prec)
        assert sim.solve_form() == form
        assert s["active_bricks"] == n and s["converged"] and s["rel_residual"] <= 1e-6
        assert again["iterations"] == s["iterations"] and again["rel_residual"] == s["rel_residual"]  # deterministic
        got.append((s, sim.get("p")))
        sim.close()
    (a, p), (b, q) = got
    assert a["refinements"] == b["refinements"]
    assert abs(a["iterations"] - b["iterations"]) <= 2 + 0.03 * b["iterations"], (a, b)
    assert np.linalg.norm(p - q) <= 1e-4 * np.linalg.norm(q)


@pytest.mark.parametrize("prec", ["jacobi", "mic0"])
def test_resident_iteration_cap(flip2, prec):
    """The cap ends a refinement within the launch, as in the two-kernel form."""
    grid, pos, vel = _bricks(100, 3)
    got = []
    for cap in (7, 20000):
        sim = flip2.FluidSim(pos[0].size, grid, preconditioner=prec, max_iterations=cap, tolerance=1e-6)
        sim.set_particles(*pos, *vel)
        for stage in ("transfer_prepare", "system"):
            sim.stage(stage)
        got.append(sim.solve_with(prec))
        assert (sim.solve_form()["resident_refinements"] > 0) == (cap == 7)
        sim.close()
    assert got[0]["iterations"] == 7 and not got[0]["converged"]
    assert got[1]["converged"] and got[1]["iterations"] > 7


def test_resident_on_threads(flip2):
    """Simulations solving on threads of one process: their resident launches
    take turns (each fits the chip by itself, not all together), every solve
    stays resident, and each gives the iterations and pressure of the same
    solve alone, bit for bit."""
    sims, alone = [], []
    for n, prec in ((64, "mic0"), (3100, "jacobi"), (900, "jacobi"), (2100, "mic0")):
        grid, pos, vel = _bricks(n, n)
        sim = flip2.FluidSim(pos[0].size, grid, preconditioner=prec)
        sim.set_particles(*pos, *vel)
        for stage in ("transfer_prepare", "system"):
            sim.stage(stage)
        s = sim.solve_with(prec)
        assert s["converged"] and sim.solve_form()["resident_refinements"] == s["refinements"]
        sims.append((sim, prec))
        alone.append((s["iterations"], sim.get("p")))
    got = [[] for _ in sims]

    def work(k):
        sim, prec = sims[k]
        for _ in range(8):
            s = sim.solve_with(prec)
            got[k].append((s["iterations"], s["refinements"], sim.solve_form(), sim.get("p")))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(sims))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, (iterations, p) in enumerate(alone):
        assert len(got[k]) == 8
        for its, refinements, form, q in got[k]:
            assert its == iterations and np.array_equal(q, p)
            assert form == {"resident_refinements": refinements, "give_ups": 0}
    for sim, _ in sims:
        sim.close()

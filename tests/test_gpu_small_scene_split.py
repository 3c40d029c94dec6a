"""Transfer + prepare and G2P + RK2 where the scene has fewer bricks than the
chip holds workgroups (one face component per workgroup, a brick's particles
over several) against the unfused stages, bit for bit: one brick, a few with
uneven loads (an empty one among them), and a grid whose bricks number just
below and above the switch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(dims, fill, seed):
    h = np.float32(1.0 / max(dims))
    rng = np.random.default_rng(seed)
    n = int(fill * dims[0] * dims[1] * dims[2]) + 1
    pos = [(rng.random(n) * d * h * 0.999).astype(np.float32) for d in dims]
    heavy = rng.random(n) < 0.5  # half of them in one corner brick
    pos = [np.where(heavy, (rng.random(n) * 8 * h).astype(np.float32), p) for p in pos]
    vel = [rng.uniform(-3, 3, n).astype(np.float32) for _ in range(3)]
    return (0.0, 0.0, 0.0, *dims, float(h)), pos, vel


@pytest.mark.parametrize("dims,fill", [((8, 8, 8), 3.0), ((16, 8, 24), 0.02), ((24, 16, 24), 6.0), ((64, 64, 64), 0.5),
                                       ((80, 64, 64), 0.3), ((96, 96, 64), 0.2)])
def test_small_scene_stages(flip2, dims, fill):
    grid, pos, vel = _scene(dims, fill, sum(dims))
    sims = [flip2.FluidSim(pos[0].size, grid, preconditioner="mic0") for _ in range(2)]
    for s in sims:
        s.set_particles(*pos, *vel)
    a, b = sims
    for _ in range(2):
        for st in ("transfer_prepare", "system", "solve", "project"):
            a.stage(st)
        for st in ("transfer", "prepare", "system", "solve", "project"):
            b.stage(st)
        for name in ("U", "V", "W", "U0", "V0", "W0"):
            assert np.array_equal(a.get(name).view(np.uint32), b.get(name).view(np.uint32)), name
        a.stage("g2p_advect")
        b.stage("g2p")
        b.stage("advect")
        for p, q in zip(a.particles(), b.particles()):
            assert np.array_equal(p.view(np.uint32), q.view(np.uint32))


@pytest.mark.parametrize("dims,fill", [((8, 8, 8), 3.0), ((24, 16, 24), 6.0), ((64, 64, 64), 0.5), ((96, 96, 64), 0.2)])
def test_small_scene_transfer_matches_oracle(flip2, oracle, dims, fill):
    """Positions in 64ths of a unit cell: coordinates, weights (multiples of
    2^-18, up to 1) and their fixed-point sums are exact, so a face carries
    the roundings of vel * scale * weight (two) and of the result: 3 * 2^-24 of
    the largest speed."""
    _, pos, vel = _scene(dims, fill, 7 + sum(dims))
    pos = [(np.floor(p * max(dims) * 64) / 64).astype(np.float32) for p in pos]
    grid = (0.0, 0.0, 0.0, *dims, 1.0)
    *U, _ = flip2.transfer(*pos, *vel, grid)
    for a, b, v in zip(U, oracle.ns_p2g(*pos, *vel, grid), vel):
        assert np.max(np.abs(a.astype(np.float64) - b)) <= 3 * 2.0**-24 * np.max(np.abs(v))

"""The SOR's quotient and the G2P's (component, particle) pairs where they can
go wrong.

An SOR iteration is linear, and a power of two scales every step of it without
rounding: with divU scaled by 2^-940 every quotient takes the division (the
corrected product is for |q| above 2^-900), unscaled none does, and the two
pressures are equal bit for bit up to the scale.  G2P: a node with one
particle, one whose pairs fill the workgroup once (64) and just more (65), and
several times (300), against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DOM = (0.0, 0.0, 0.0, 8, 8, 8, 0.125)
DT = 1.0 / 240.0


def _pair(flip2, oracle, counts, seed):
    rng = np.random.default_rng(seed)
    cells = [(1, 1, 1), (3, 4, 5), (0, 7, 0), (7, 0, 7)]
    pos = [np.concatenate([(c[d] + rng.random(n)) * 0.125 for c, n in zip(cells, counts)]) for d in range(3)]
    vel = [rng.uniform(-1, 1, pos[0].size) for _ in range(3)]
    out = []
    for s in (flip2.Particles(pos[0].size), oracle.OracleParticles(pos[0].size)):
        s.setDomain(*DOM)
        s.set_positions(*pos)
        s.set_velocities(*vel)
        s.initialize()
        out.append(s)
    return out


@pytest.mark.parametrize("iters", [1, 2])
def test_sor_quotient_matches_division(flip2, oracle, iters):
    got = []
    for scale in (1.0, 2.0**-940):
        g, o = _pair(flip2, oracle, (300, 200, 65, 20), 3)
        o.particleVelToVoxels()
        o.applyGravity(DT)
        o.calcDivU()
        g.set("divU", o.get("divU") * scale)
        g.gsIterations(DT, iters)
        got.append((g.get("p") / scale, g.get("residuals")))
    assert np.any(got[0][0] != 0.0)
    assert np.array_equal(got[0][0], got[1][0])


@pytest.mark.parametrize("counts", [(1, 1, 1, 1), (64, 65, 1, 300), (21, 22, 63, 129)])
def test_g2p_pairs(flip2, oracle, counts):
    g, o = _pair(flip2, oracle, counts, sum(counts))
    o.particleVelToVoxels()
    for n in ("voxelsUx", "voxelsUy", "voxelsUz"):
        g.set(n, o.get(n))
    g.voxelVelsToParticles()
    o.voxelVelsToParticles()
    for n in ("vx", "vy", "vz"):
        a, b = g.get(n), o.get(n)
        # 64 FP64 products and sums of one sign in the weights: far below 1e-12
        assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b)), n

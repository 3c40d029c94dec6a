"""The weight gradient's tiles (16 x 4 x 4 voxels, workgroups that walk several
tiles, channel pairs of every layer) where they do not divide the grid: levels
of 40, 20 and 10 voxels (partial tiles on every axis, more tiles than
workgroups on level 0) and of 24, 12 and 6, against the FP64 oracle's gradient
of the same bf16-rounded forward pass, at the tolerance of the other gradient
checks."""
import pytest

pytestmark = pytest.mark.gpu

from oracle import unet_oracle as uo
from tests.test_gpu_unet import GRAD_TOL, biased_params, check_gradients
from tests.unet_cases import synthetic_system


@pytest.mark.parametrize("n", [24, 40])
def test_gradient_matches_oracle_ragged(flip2, n):
    net = flip2.UNet(n, seed=9)
    net.set_smoothing(0.0)
    p = biased_params(net, 70 + n)
    b, coef = synthetic_system(n, 71 + n)
    loss, g = net.loss_grad(b, coef)
    Lo, go = uo.Net(n, p, bf16=True).loss_grad(b, coef)
    assert abs(loss - Lo) <= 1e-2 * Lo, (loss, Lo)
    check_gradients(g, go, GRAD_TOL)

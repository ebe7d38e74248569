"""The 768-point transforms (radix 12, whose LDS layouts are swizzled instead
of padded) along either grid axis and along both, for one and two coil blocks,
against the float64 arithmetic model."""

import numpy as np
import pytest

from gpu_util import dev, need_gpu, rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coils", [3, 11])
@pytest.mark.parametrize("image", [(384, 32), (64, 384), (384, 384)])
def test_radix_12(image, coils):
    need_gpu()
    from oracle.solver import KbOperator
    from trajsparsenufft_amd import pack, synth
    from trajsparsenufft_amd.recon import build_plan
    grid = (2 * image[0], 2 * image[1])
    traj = synth.radial(13, 211)
    packs = pack.prepare_trajectory(traj, image, grid)
    smaps = synth.coil_maps(coils, *image)
    cols, re, im = packs.kb.arrays()
    model = KbOperator(cols, re, im, smaps, packs.apod, image, grid, "fp32", "fp32")
    plan = build_plan(packs, dev(smaps), "fp32")
    x = dev(synth.phantom(*image, seed=coils))
    rng = np.random.default_rng(coils)
    m = traj.shape[0]
    y = (rng.standard_normal((coils, m)) + 1j * rng.standard_normal((coils, m))).astype(np.complex64)
    assert rel_l2(plan.forward(x).cpu().numpy(), model.forward(x.cpu().numpy())) <= 2e-6
    assert rel_l2(plan.adjoint(dev(y)).cpu().numpy(), model.adjoint(y)) <= 2e-6

"""Plan operators read and write a caller's row-major images in place: for
non-square shapes the results match the float64 arithmetic model, and a normal
operator whose output is its input image gives the same bits as one that
writes elsewhere."""

import numpy as np
import pytest

from gpu_util import dev, need_gpu, rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coils", [1, 7, 12])
@pytest.mark.parametrize("image", [(32, 128), (64, 32)])
@pytest.mark.parametrize("precision,tol", [("fp32", 2e-6), ("split16", 2e-5)])
def test_row_major_images(image, coils, precision, tol):
    need_gpu()
    from oracle.solver import KbOperator
    from trajsparsenufft_amd import pack, synth
    from trajsparsenufft_amd.recon import build_plan
    grid = (2 * image[0], 2 * image[1])
    traj = synth.radial(31, 97)
    packs = pack.prepare_trajectory(traj, image, grid)
    smaps = synth.coil_maps(coils, *image)
    cols, re, im = packs.kb.arrays()
    modes = ("fp32", "fp32") if precision == "fp32" else ("fp16", "split2")
    model = KbOperator(cols, re, im, smaps, packs.apod, image, grid, *modes)
    plan = build_plan(packs, dev(smaps), precision)
    x = dev(synth.phantom(*image, seed=coils))
    rng = np.random.default_rng(coils)
    m = traj.shape[0]
    y = (rng.standard_normal((coils, m)) + 1j * rng.standard_normal((coils, m))).astype(np.complex64)
    assert rel_l2(plan.forward(x).cpu().numpy(), model.forward(x.cpu().numpy())) <= tol
    assert rel_l2(plan.adjoint(dev(y)).cpu().numpy(), model.adjoint(y)) <= tol
    ref = plan.normal(x, 0.5, 0.25)
    same = x.clone()
    plan.normal(same, 0.5, 0.25, out=same)
    assert torch.equal(torch.view_as_real(ref), torch.view_as_real(same))
    expect = 0.5 * model.adjoint(model.forward(x.cpu().numpy())) + 0.25 * x.cpu().numpy()
    assert rel_l2(ref.cpu().numpy(), expect) <= tol

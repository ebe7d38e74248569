"""Sample layout kernels at the edges of their row tiles: the split of raw
samples into half panels matches numpy bit for bit, and the row-major copies
behind the FP32 adjoint and the fused data consistency match the float64
arithmetic model."""

import numpy as np
import pytest

from gpu_util import dev, need_gpu, rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coils", [1, 8, 9, 16])
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 300])
def test_split_panel(rows, coils):
    need_gpu()
    from trajsparsenufft_amd import device
    rng = np.random.default_rng(rows + coils)
    y = (rng.standard_normal((coils, rows)) + 1j * rng.standard_normal((coils, rows))).astype(np.complex64)
    scale = np.float32(0.75)
    hi, res = (t.cpu().numpy() for t in device.split_panel(dev(y), coils, float(scale)))
    blocks = (coils + 7) // 8
    v = np.zeros((blocks, rows, 16), np.float32)
    for c in range(coils):
        v[c // 8, :, c % 8] = y[c].real * scale
        v[c // 8, :, c % 8 + 8] = y[c].imag * scale
    h = v.astype(np.float16)
    assert np.array_equal(hi.reshape(v.shape), h)
    assert np.array_equal(res.reshape(v.shape), (v - h.astype(np.float32)).astype(np.float16))


@pytest.mark.parametrize("coils", [1, 5, 16])
@pytest.mark.parametrize("samples", [1, 127, 128, 130])
@pytest.mark.parametrize("precision,tol", [("fp32", 2e-6), ("split16", 2e-5)])
def test_sample_rows(samples, coils, precision, tol):
    need_gpu()
    from oracle.solver import KbOperator
    from trajsparsenufft_amd import pack, synth
    from trajsparsenufft_amd.recon import build_plan
    image, grid = (32, 32), (64, 64)
    traj = synth.radial(3, 64)[:samples]
    packs = pack.prepare_trajectory(traj, image, grid)
    smaps = synth.coil_maps(coils, *image)
    cols, re, im = packs.kb.arrays()
    modes = ("fp32", "fp32") if precision == "fp32" else ("fp16", "split2")
    model = KbOperator(cols, re, im, smaps, packs.apod, image, grid, *modes)
    plan = build_plan(packs, dev(smaps), precision)
    rng = np.random.default_rng(samples + coils)
    y = (rng.standard_normal((coils, samples)) + 1j * rng.standard_normal((coils, samples))).astype(np.complex64)
    x = (rng.standard_normal(image) + 1j * rng.standard_normal(image)).astype(np.complex64)
    assert rel_l2(plan.adjoint(dev(y)).cpu().numpy(), model.adjoint(y)) <= tol
    dc = plan.data_consistency(dev(x), dev(y), measurement_scale=1.0).cpu().numpy()
    assert rel_l2(dc, model.adjoint(model.forward(x) - y)) <= tol

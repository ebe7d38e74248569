"""FP32 interpolation through LDS-staged column blocks: coil counts off the
lane width, non-square grids, sparse spirals (few shared columns) and dense
centres (groups cut into column chunks) against the float64 product, and
non-finite inputs staying with the rows that name them."""

import numpy as np
import pytest

from gpu_util import dev, need_gpu, rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# image shape, trajectory kind, interleaves / spokes, readout
CASES = {"sparse spiral": ((64, 32), "spiral", 3, 331), "dense radial": ((32, 32), "radial", 301, 63),
         "one spoke": ((32, 64), "radial", 1, 77)}


def _case(name):
    from trajsparsenufft_amd import pack, synth
    image, kind, n, readout = CASES[name]
    traj = synth.radial(n, readout) if kind == "radial" else synth.spiral(n, readout, turns=5.0)
    kb = pack.KbMatrix.build(traj, image, (2 * image[0], 2 * image[1]))
    return kb, *kb.arrays()


@pytest.mark.parametrize("view", ["G", "G_T"])
@pytest.mark.parametrize("coils", [1, 5, 9, 13])
@pytest.mark.parametrize("name", list(CASES))
def test_csr_blocks_match_oracle(name, coils, view):
    need_gpu()
    from oracle.solver import apply_csr, apply_csr_adjoint
    from trajsparsenufft_amd import device
    kb, cols, re, im = _case(name)
    d = device.Direction.csr(kb, view)
    rng = np.random.default_rng(coils)
    x = (rng.standard_normal((d.cols, coils)) + 1j * rng.standard_normal((d.cols, coils))).astype(np.complex64)
    x64 = x.astype(np.complex128)
    ref = apply_csr(cols, re, im, x64) if view == "G" else apply_csr_adjoint(cols, re, im, x64, d.rows)
    out = torch.full((d.rows, coils), float("nan"), dtype=torch.complex64, device="cuda")
    device.interp_f32(d, dev(x), out, coils=coils, conjugate=view == "G_T", layout="row_major")
    assert rel_l2(out.cpu().numpy(), ref) <= 1e-6
    # non-finite inputs reach exactly the rows that name them
    bad = np.array([0, d.cols // 2])
    y = x.copy()
    y[bad] = np.array([np.inf, np.nan])[:, None]
    hit = np.zeros(d.rows, dtype=bool)
    if view == "G":
        hit = np.isin(cols, bad).any(axis=1)
    else:
        hit[cols[bad].ravel()] = True
    got = torch.full_like(out, float("nan"))
    device.interp_f32(d, dev(y), got, coils=coils, conjugate=view == "G_T", layout="row_major")
    g, o = got.cpu().numpy(), out.cpu().numpy()
    assert np.array_equal(g[~hit].view(np.uint32), o[~hit].view(np.uint32))
    assert not np.isfinite(g[hit]).any()

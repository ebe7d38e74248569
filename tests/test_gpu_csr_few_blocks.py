"""FP32 interpolation of directions of few blocks (coils split over blocks of
four, fewer rows a block) and of many (all coils in each): a sample's value has
the same bits in both, and both match the float64 product at coil counts off
the lane width."""

import numpy as np
import pytest

from gpu_util import dev, need_gpu, rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

IMAGE, GRID = (64, 64), (128, 128)


def _run(d, x, coils, layout, conjugate=False, accumulate=False):
    from trajsparsenufft_amd import device
    shape = (d.rows, coils) if layout == "row_major" else (coils, d.rows)
    out = torch.full(shape, 2 - 1j if accumulate else float("nan"), dtype=torch.complex64, device="cuda")
    device.interp_f32(d, dev(x), out, coils=coils, conjugate=conjugate, accumulate=accumulate, layout=layout)
    return out.cpu().numpy() if layout == "row_major" else out.T.cpu().numpy()


@pytest.mark.parametrize("coils", [1, 4, 5, 8, 9, 13, 16])
def test_few_and_many_blocks(coils):
    need_gpu()
    from oracle.solver import apply_csr, apply_csr_adjoint
    from trajsparsenufft_amd import device, pack, synth
    traj = synth.radial(300, 128)  # at least 600 blocks of 64 samples; most grid rows are long
    many = pack.KbMatrix.build(traj, IMAGE, GRID)
    few = pack.KbMatrix.build(traj[:1777], IMAGE, GRID)
    rng = np.random.default_rng(coils)

    def data(rows):
        return (rng.standard_normal((rows, coils)) + 1j * rng.standard_normal((rows, coils))).astype(np.complex64)
    g = data(GRID[0] * GRID[1])
    for layout in ("row_major", "coil_major"):
        for conjugate, accumulate in ((False, False), (True, True)):
            a = _run(device.Direction.csr(many, "G"), g, coils, layout, conjugate, accumulate)[:1777]
            b = _run(device.Direction.csr(few, "G"), g, coils, layout, conjugate, accumulate)
            assert np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))
    for kb in (many, few):
        cols, re, im = kb.arrays()
        assert rel_l2(_run(device.Direction.csr(kb, "G"), g, coils, "row_major"),
                      apply_csr(cols, re, im, g.astype(np.complex128))) <= 1e-6
        y = data(len(cols))
        assert rel_l2(_run(device.Direction.csr(kb, "G_T"), y, coils, "row_major", conjugate=True),
                      apply_csr_adjoint(cols, re, im, y.astype(np.complex128), g.shape[0])) <= 1e-6

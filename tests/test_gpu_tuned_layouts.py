"""A direction tuned for 9 to 16 coils keeps one schedule for plans (both coil
blocks of a panel row in one line) and one for calls on a caller's panels
(separate blocks): every launch of either gives the bits of the untuned one,
and a schedule that is set by hand goes to both."""

import numpy as np
import pytest

from gpu_util import dev, need_gpu, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _bits(t):
    torch.cuda.synchronize()
    t = torch.view_as_real(t) if t.is_complex() else t
    return np.ascontiguousarray(t.cpu().numpy()).view(np.uint32)


@pytest.mark.parametrize("coils", [8, 11, 16])
def test_tuned_layouts(coils):
    need_gpu()
    from trajsparsenufft_amd import device, synth
    from trajsparsenufft_amd.recon import build_plan
    traj, packs = small_case(32, 120)  # long groups in the adjoint
    rng = np.random.default_rng(coils)

    def data(rows):
        return dev((rng.standard_normal((coils, rows)) + 1j * rng.standard_normal((coils, rows))).astype(np.complex64))
    plan = build_plan(packs, dev(synth.coil_maps(coils, 32)), "split16")
    fwd, adj = plan._dirs
    x, y = dev(synth.phantom(32, seed=coils)), data(traj.shape[0])
    panels = {d: device.split_panel_il(data(d.cols), coils) for d in (fwd, adj)}

    def outputs():
        out = [plan.forward(x), plan.adjoint(y), plan.normal(x, 1.0, 0.1)]
        for d, conj in ((fwd, False), (adj, True)):
            for layout in ("row_major", "coil_major"):
                o = torch.zeros(d.rows * coils, dtype=torch.complex64, device="cuda")
                out.append(device.interp_il(d, panels[d], o, coils, conjugate=conj, layout=layout))
        o = torch.zeros(device.coil_blocks(coils) * fwd.rows * 16, dtype=torch.int32, device="cuda")
        out.append(device.interp_il(fwd, panels[fwd], o, coils, layout="split_il"))
        return [_bits(o) for o in out]
    ref = outputs()
    for d in (fwd, adj):
        unit, us = d.autotune(coils)
        assert unit in (2, 3, 4, 5, 6, 8, 10, 12, 14, 16) and d.unit_tiles == unit and us > 0
    assert all(np.array_equal(a, b) for a, b in zip(outputs(), ref))
    for d in (fwd, adj):
        d.schedule(3)
        d.coil_waves, d.pipe_depth = 2, 1
        assert (d.unit_tiles, d.coil_waves, d.pipe_depth) == (3, 2, 1)
    assert all(np.array_equal(a, b) for a, b in zip(outputs(), ref))

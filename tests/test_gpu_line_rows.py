"""Plans of 9 to 16 coils keep both coil blocks of a panel row in one 128-byte
line: every operator is bitwise the same whether one wave takes both blocks
(16-byte line loads, either pipeline depth) or one wave takes each block
(4-byte loads of half lines), and matches the up-to-8-coil layout coil by
coil."""

import numpy as np
import pytest

from gpu_util import dev, need_gpu, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _outputs(plan, x, y, density):
    out = [plan.forward(x), plan.adjoint(y), plan.data_consistency(x, y, density), plan.normal(x, 1.0, 0.1)]
    torch.cuda.synchronize()
    return [np.ascontiguousarray(torch.view_as_real(o).cpu().numpy()).view(np.uint32) for o in out]


@pytest.mark.parametrize("precision", ["split16", "splitbf16", "dense16", "hi16"])
@pytest.mark.parametrize("coils", [9, 11, 16])
def test_line_rows_are_bitwise_invariant(coils, precision):
    need_gpu()
    from trajsparsenufft_amd import synth
    from trajsparsenufft_amd.recon import build_plan
    traj, packs = small_case(32, 120)  # 120 spokes: long groups in the adjoint
    rng = np.random.default_rng(coils)
    smaps = synth.coil_maps(coils, 32)
    x = dev(synth.phantom(32, seed=coils))
    m = traj.shape[0]
    y = dev((rng.standard_normal((coils, m)) + 1j * rng.standard_normal((coils, m))).astype(np.complex64))
    density = dev(rng.uniform(0.1, 1.0, m).astype(np.float32))
    plan = build_plan(packs, dev(smaps), precision)
    ref = None
    for waves, depth in ((1, 0), (2, 0), (1, 2)):
        for d in plan._dirs:
            d.coil_waves, d.pipe_depth = waves, depth
        got = _outputs(plan, x, y, density)
        if ref is None:
            ref = got
        assert all(np.array_equal(a, b) for a, b in zip(got, ref)), (waves, depth)
    # the first eight coils alone, in the one-block layout: a coil's samples do not depend on the others
    one = build_plan(packs, dev(smaps[:8]), precision).forward(x)
    torch.cuda.synchronize()
    assert np.array_equal(np.ascontiguousarray(torch.view_as_real(one).cpu().numpy()).view(np.uint32), ref[0][:8])


@pytest.mark.parametrize("precision", ["split16", "splitbf16", "dense16", "hi16"])
@pytest.mark.parametrize("coils", [9, 11, 16])
def test_second_block_of_line_rows_matches_the_one_block_layout(coils, precision):
    """Coils 8 .. are the second half of every line: their samples have the bits
    of a plan that holds them alone in the one-block layout."""

    need_gpu()
    from trajsparsenufft_amd import synth
    from trajsparsenufft_amd.recon import build_plan
    _, packs = small_case(32, 120)
    smaps = synth.coil_maps(coils, 32)
    x = dev(synth.phantom(32, seed=coils))
    both = build_plan(packs, dev(smaps), precision).forward(x)
    second = build_plan(packs, dev(smaps[8:]), precision).forward(x)
    torch.cuda.synchronize()
    assert torch.equal(torch.view_as_real(both[8:]), torch.view_as_real(second))

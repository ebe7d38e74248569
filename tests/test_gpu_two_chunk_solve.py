"""Solves of more than eight coils (two coil chunks share the pixel vectors,
one of them updates x in place): every replay of a captured solve gives the
bits of the enqueued one."""

import pytest

from gpu_util import dev, need_gpu, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coils", [9, 16])
@pytest.mark.parametrize("precision", ["fp32", "split16"])
def test_two_chunk_solves_repeat_bitwise(precision, coils):
    need_gpu()
    from trajsparsenufft_amd import synth
    from trajsparsenufft_amd.recon import build_plan
    n = 32
    _, packs = small_case(n)
    plan = build_plan(packs, dev(synth.coil_maps(coils, n)), precision)
    y = plan.forward(dev(synth.phantom(n, seed=coils))) * (2 * n)
    scale = plan.operator_scale(y)
    ref = torch.view_as_real(plan.cg(y, 6, scale, 1e-4).image).clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        out = plan.capture_cg(y, 6, scale, 1e-4)
        for _ in range(5):
            out.image.zero_()
            plan.replay()
            stream.synchronize()
            assert torch.equal(torch.view_as_real(out.image), ref)

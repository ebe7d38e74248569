"""A normal operator whose output overlaps its input image at an offset (down
to one pixel, up to all but one) gives the same bits as one that writes
elsewhere."""

import pytest

from gpu_util import dev, need_gpu, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coils", [3, 11])
@pytest.mark.parametrize("precision", ["fp32", "split16"])
def test_normal_into_an_overlapping_image(precision, coils):
    need_gpu()
    from trajsparsenufft_amd import synth
    from trajsparsenufft_amd.recon import build_plan
    n = 32
    _, packs = small_case(n)
    plan = build_plan(packs, dev(synth.coil_maps(coils, n)), precision)
    x = dev(synth.phantom(n, seed=coils))
    ref = torch.view_as_real(plan.normal(x, 0.5, 0.25))
    px = n * n
    for offset in (-px, 1 - px, -n, -1, 0, 1, 3, n, px // 2, px - 1, px):
        buf = torch.zeros(2 * px, dtype=torch.complex64, device="cuda")
        a, b = max(0, -offset), max(0, offset)
        image, out = buf[a:a + px].view(n, n), buf[b:b + px].view(n, n)
        image.copy_(x)
        plan.normal(image, 0.5, 0.25, out=out)
        assert torch.equal(torch.view_as_real(out), ref), offset

"""Device planning of spectra (fufft_plan_filter*_device_f32, spectrum kind):
the bit-permuting transpose moves 2^11 points per workgroup, so a tile holds
several small items (the last one partly past the batch), one item, or a part
of one.  A permutation times a power of two: bit-identical to the host
planner, and nothing written past the items."""
import numpy as np
import pytest

from conftest import bits_equal, crandn

pytestmark = pytest.mark.gpu


def _run(dev, spec, plan, host):
    """plan(in, out) on the device against the host planner's rows; a guard row
    behind the output stays as it was."""
    import torch
    count, n = spec.shape
    out = torch.full((count * n + 4096,), 7.0 + 0j, dtype=torch.complex64, device=dev)
    plan(torch.from_numpy(spec).to(dev), out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert bits_equal(got[: count * n].reshape(count, n), np.stack([host(s) for s in spec]))
    assert np.all(got[count * n:] == 7.0)


@pytest.mark.parametrize("layout", ["dr", "lane", "bperm"])
@pytest.mark.parametrize("variant,n,count", [("v16", 256, 1), ("v16", 256, 9), ("v16", 512, 7), ("r8", 512, 5),
                                             ("r8", 1024, 3), ("v16", 2048, 3), ("r8", 2048, 2), ("v16", 4096, 5),
                                             ("r8", 4096, 3), ("v16", 8192, 1), ("r8", 8192, 3), ("v16", 16384, 2),
                                             ("v16", 32768, 2)])
def test_1d(dev, rng, variant, n, count, layout):
    import fufft_amd as ff
    print(f"case plan 1d {variant} n={n} count={count} {layout}", flush=True)
    _run(dev, crandn(rng, (count, n)),
         lambda i, o: ff.plan_filter_device(i, o, n, count=count, variant=variant, layout=layout),
         lambda s: ff.plan_filter(s, n, variant=variant, layout=layout))


@pytest.mark.parametrize("variant", ["v16", "r8"])
@pytest.mark.parametrize("n,count", [(8192, 3), (65536, 2), (131072, 1), (1 << 20, 1)])
def test_large(dev, rng, variant, n, count):
    import fufft_amd as ff
    print(f"case plan large {variant} n={n} count={count}", flush=True)
    _run(dev, crandn(rng, (count, n)),
         lambda i, o: ff.plan_filter_large_device(i, o, n, count=count, variant=variant),
         lambda s: ff.plan_filter_large(s, n, variant=variant))


@pytest.mark.parametrize("layout", ["dr", "lane"])
@pytest.mark.parametrize("h,w,count", [(8, 8, 33), (8, 512, 3), (512, 8, 1), (16, 64, 5), (64, 128, 2), (256, 256, 3),
                                       (512, 512, 2), (2048, 256, 1), (256, 4096, 1), (1024, 8192, 1)])
def test_2d(dev, rng, h, w, count, layout):
    import fufft_amd as ff
    print(f"case plan 2d {h}x{w} count={count} {layout}", flush=True)
    _run(dev, crandn(rng, (count, h * w)),
         lambda i, o: ff.plan_filter2d_device(i, o, h, w, count=count, layout=layout),
         lambda s: ff.plan_filter2d(s, h, w, layout=layout))

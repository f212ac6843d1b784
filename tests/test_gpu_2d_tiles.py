"""The 2D column kernels' tiles: 4, 8 or 16 columns per workgroup by the
points of the launch, the tiles that share cache lines on one XCD.  Every
column is the same transform whatever the tile, so a batch on either side of
each line gives what its images give one at a time (parity of those with the
oracle: test_gpu_2d.py), bit for bit, and nothing behind it is written."""
import pytest

pytestmark = pytest.mark.gpu


def _same(a, b):
    import torch
    return torch.equal(torch.view_as_real(a), torch.view_as_real(b))


# (h, w, images): 4 columns below 1600 columns in the launch, then 8, and at
# h <= 512 16 beyond 2^14 columns
@pytest.mark.parametrize("layout", ["dr", "lane"])
@pytest.mark.parametrize("h,w,batch", [(256, 256, 6), (256, 256, 7), (256, 256, 65), (512, 512, 3), (512, 512, 4),
                                       (512, 512, 33), (1024, 256, 6), (1024, 256, 7), (2048, 512, 3), (2048, 256, 7)])
def test_conv(dev, h, w, batch, layout):
    import torch
    import fufft_amd as ff
    print(f"case conv2d {h}x{w} batch={batch} {layout}", flush=True)
    gen = torch.Generator(device=dev)
    gen.manual_seed(h + w + batch)
    n = h * w
    x = torch.randn(batch * n, dtype=torch.complex64, device=dev, generator=gen)
    f = torch.randn(n, dtype=torch.complex64, device=dev, generator=gen)
    out = torch.full(((batch + 1) * n,), 7.0 + 0j, dtype=torch.complex64, device=dev)
    one = torch.empty(n, dtype=torch.complex64, device=dev)
    spec = torch.empty_like(x)
    ff.conv2d(x, f, out, h, w, batch, layout=layout)
    ff.fwd2d(x, spec, h, w, batch)
    for i in range(batch):
        ff.conv2d(x[i * n: (i + 1) * n], f, one, h, w, 1, layout=layout)
        assert _same(one, out[i * n: (i + 1) * n]), i
        ff.fwd2d(x[i * n: (i + 1) * n], one, h, w, 1)
        assert _same(one, spec[i * n: (i + 1) * n]), i
    assert bool((out[batch * n:] == 7.0).all())


# the split apply: 16 columns and streamed filters beyond 2^22 points
@pytest.mark.parametrize("layout", ["dr", "lane"])
@pytest.mark.parametrize("own_spec", [False, True])
@pytest.mark.parametrize("h,w,batch", [(256, 256, 6), (256, 256, 64), (256, 256, 65), (512, 512, 17), (1024, 1024, 4),
                                       (1024, 512, 9), (2048, 256, 9)])
def test_apply(dev, h, w, batch, layout, own_spec):
    import torch
    import fufft_amd as ff
    print(f"case apply2d {h}x{w} batch={batch} {layout} own_spec={own_spec}", flush=True)
    gen = torch.Generator(device=dev)
    gen.manual_seed(h + w + batch)
    n = h * w
    s = torch.randn((batch if own_spec else 1) * n, dtype=torch.complex64, device=dev, generator=gen)
    f = torch.randn(batch * n, dtype=torch.complex64, device=dev, generator=gen)
    out = torch.full(((batch + 1) * n,), 7.0 + 0j, dtype=torch.complex64, device=dev)
    one = torch.empty(n, dtype=torch.complex64, device=dev)
    ff.apply2d(s, f, out, h, w, batch, spec_stride=n if own_spec else 0, filt_stride=n, layout=layout)
    for i in range(batch):
        si = s[i * n: (i + 1) * n] if own_spec else s
        ff.apply2d(si, f[i * n: (i + 1) * n], one, h, w, 1, spec_stride=0, filt_stride=n, layout=layout)
        assert _same(one, out[i * n: (i + 1) * n]), i
    assert bool((out[batch * n:] == 7.0).all())

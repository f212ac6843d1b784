"""The cache policy of the conv's loads (N <= 8192: signals of up to 80 MiB or
more), of the N = 16384 conv's stores and of the C2C's stores (results of up to
256 MiB, with the filters where each signal has its own, or more) is chosen by
size, each with a kernel of its own.  On both sides of the line, and beside it,
a batch gives what its parts give in small calls (parity of those with the
oracle: test_gpu_conv1d.py, test_gpu_c2c.py), bit for bit, out of place and in
place."""
import pytest

pytestmark = pytest.mark.gpu

PART = 64


def _same(a, b):
    import torch
    return torch.equal(torch.view_as_real(a), torch.view_as_real(b))


def _signals(dev, n, batch):
    import torch
    gen = torch.Generator(device=dev)
    gen.manual_seed(n + batch)
    return torch.randn(batch * n, dtype=torch.complex64, device=dev, generator=gen), gen


@pytest.mark.parametrize("layout", ["dr", "lane", "bperm"])
@pytest.mark.parametrize("n,variant", [(256, "v16"), (512, "r8"), (4096, "v16"), (4096, "r8"), (8192, "v16"),
                                       (8192, "r8")])
@pytest.mark.parametrize("past", [-1, 0, 1])
def test_conv_loads(dev, n, variant, layout, past):
    import torch
    import fufft_amd as ff
    batch = (80 << 20) // (8 * n) + past
    print(f"case conv policy n={n} {variant} {layout} batch={batch}", flush=True)
    x, gen = _signals(dev, n, batch)
    f = torch.randn(n, dtype=torch.complex64, device=dev, generator=gen)
    out = torch.empty_like(x)
    ff.conv(x, f, out, n, batch, mid="conj", variant=variant, layout=layout)
    part = torch.empty(PART * n, dtype=torch.complex64, device=dev)
    for a in (0, batch // 2, batch - PART):
        ff.conv(x[a * n: (a + PART) * n], f, part, n, PART, mid="conj", variant=variant, layout=layout)
        assert _same(part, out[a * n: (a + PART) * n]), a
    ff.conv(x, f, x, n, batch, mid="conj", variant=variant, layout=layout)
    assert _same(x, out)


@pytest.mark.parametrize("own", [False, True])
@pytest.mark.parametrize("layout", ["dr", "bperm"])
@pytest.mark.parametrize("past", [0, 1])
def test_conv_16384_stores(dev, layout, own, past):
    import torch
    import fufft_amd as ff
    n = 16384
    batch = ((128 if own else 256) << 20) // (8 * n) + past
    print(f"case conv policy n={n} {layout} own={own} batch={batch}", flush=True)
    x, gen = _signals(dev, n, batch)
    f = torch.randn(n * (batch if own else 1), dtype=torch.complex64, device=dev, generator=gen)
    stride = n if own else 0
    out = torch.empty_like(x)
    ff.conv(x, f, out, n, batch, filt_stride=stride, layout=layout)
    part = torch.empty(PART * n, dtype=torch.complex64, device=dev)
    for a in (0, batch // 2, batch - PART):
        fp = f[a * n: (a + PART) * n] if own else f
        ff.conv(x[a * n: (a + PART) * n], fp, part, n, PART, filt_stride=stride, layout=layout)
        assert _same(part, out[a * n: (a + PART) * n]), a
    ff.conv(x, f, x, n, batch, filt_stride=stride, layout=layout)
    assert _same(x, out)


@pytest.mark.parametrize("n,variant", [(256, "v16"), (512, "r8"), (4096, "r8"), (16384, "v16")])
@pytest.mark.parametrize("past", [0, 1])
def test_c2c_stores(dev, n, variant, past):
    import torch
    import fufft_amd as ff
    batch = (256 << 20) // (8 * n) + past
    print(f"case c2c policy n={n} {variant} batch={batch}", flush=True)
    x, _ = _signals(dev, n, batch)
    for d in (ff.FORWARD, ff.INVERSE):
        out = torch.empty_like(x)
        ff.c2c(x, out, n, batch, direction=d, variant=variant)
        part = torch.empty(PART * n, dtype=torch.complex64, device=dev)
        for a in (0, batch - PART):
            ff.c2c(x[a * n: (a + PART) * n], part, n, PART, direction=d, variant=variant)
            assert _same(part, out[a * n: (a + PART) * n]), (d, a)
        ff.c2c(x, x, n, batch, direction=d, variant=variant)
        assert _same(x, out)

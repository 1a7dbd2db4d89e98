"""GPU: the trunk's row kernels at the edges of their forms -- embedding ids in
launch arguments (256 a launch, up to 1024) and in a buffer, rows split over
workgroups, norm rows held in registers (up to 8192) and read twice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    from quantibbler_amd import GpuContext

    return GpuContext(0)


@pytest.mark.parametrize("n,d", [(1, 1), (1, 4096), (255, 3), (256, 1025), (257, 64), (1024, 17), (1025, 17)])
def test_embed_rows(ctx, n, d):
    from quantibbler_amd.gpu import embed, embed_dev

    g = torch.Generator(device="cuda")
    g.manual_seed(n + d)
    table = torch.randn((500, d), device="cuda", generator=g)
    ids = np.random.default_rng(n).integers(0, 500, n).astype(np.int32)
    out = torch.empty((n, d), device="cuda")
    dev = torch.empty((n, d), device="cuda")
    it = torch.from_numpy(ids).cuda()
    embed(ctx, table, 500, d, ids, out, torch.cuda.current_stream())
    embed_dev(ctx, table, 500, d, it, n, dev, torch.cuda.current_stream())
    torch.cuda.synchronize()
    want = table[it.long()]
    assert torch.equal(out, want) and torch.equal(dev, want)


@pytest.mark.parametrize("serving", ["bf16", "fp32"])
@pytest.mark.parametrize("rows,d", [(1, 1), (3, 255), (2, 257), (1, 4096), (2, 8191), (2, 8192), (2, 8193), (1, 20000)])
def test_rms_norm_rows(ctx, rows, d, serving):
    """Against float64: the sum of squares has relative error below d eps (a
    tree's is far less), bf16's output half an ulp, 2^-9, more."""
    from quantibbler_amd.gpu import rms_norm_dev

    g = torch.Generator(device="cuda")
    g.manual_seed(rows + d)
    x, w = torch.randn((rows, d), device="cuda", generator=g), torch.rand(d, device="cuda", generator=g) + 0.5
    out = torch.empty((rows, d), device="cuda")
    rms_norm_dev(ctx, x, rows, d, w, 1e-5, out, torch.cuda.current_stream(), serving)
    torch.cuda.synchronize()
    b = (x.bfloat16() if serving == "bf16" else x).double()
    want = b * torch.rsqrt((b * b).mean(-1, keepdim=True) + 1e-5) * w.double()
    tol = (d + 8) * 2.0 ** -24 + (2.0 ** -8 if serving == "bf16" else 0.0)
    assert bool(((out.double() - want).abs() <= tol * want.abs() + 1e-30).all())


@pytest.mark.parametrize("serving", ["bf16", "fp32"])
@pytest.mark.parametrize("rows,d", [(3, 511), (2, 512), (2, 513), (70, 2048), (2, 2049), (2, 4095), (2, 4097)])
def test_rms_norm_rows_at_the_kernels_widths(ctx, rows, d, serving):
    test_rms_norm_rows(ctx, rows, d, serving)


@pytest.mark.parametrize("n,d", [(1280, 1030), (1281, 1030), (3000, 2049)])
def test_embed_many_rows(ctx, n, d):
    """Either side of where a row stops being split over workgroups."""
    test_embed_rows(ctx, n, d)

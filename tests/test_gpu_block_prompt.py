"""GPU: a prompt's prefill through the one-launch GEMM with SwiGLU formed in the
up projection's epilogue and the norms in 16-byte pieces, at the edges of both:
the smallest prompt they take, ragged token groups, widths that are not
multiples of 4 (the general kernels), FFN rows of a multiple of 4 only --
against the oracle's prefill: all rows together to the decoder block's
tolerance (cos >= 0.9999, relative L2 <= 1 %), each row to what its roundings
allow: five bf16 roundings stand between a row and its output (norm, t and u of
a projection, the attention's output, the down projection's z), each at most
2^-9 of the value, and the device and the oracle, whose sums differ in order,
may fall apart at each -- 2 x 5 x 2^-9 = 1.95 %."""
import numpy as np
import pytest

from test_gpu_block import COS_MIN, REL_MAX, metrics, scaled_layer

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,d,ffn", [(256, 256, 512), (261, 132, 300), (300, 256, 514), (257, 250, 512), (65, 256, 512)])
def test_prompt_matches_oracle(orc, n, d, ffn):
    from quantibbler_amd import DecoderBlock, FactorLayer, GpuContext

    print("block prompt", n, d, ffn, flush=True)
    ctx = GpuContext(0)
    H, Hk, hd, theta, eps = 2, 1, 128, 500000.0, 1e-5
    rng = np.random.default_rng(n + d + ffn)
    shapes = [(H * hd, d, 64), (Hk * hd, d, 32), (Hk * hd, d, 32), (d, H * hd, 64), (ffn, d, 96), (ffn, d, 96),
              (d, ffn, 96)]
    layers = [scaled_layer(orc, rng, *s) for s in shapes]
    devs = [FactorLayer.from_rows(ctx, L["dout"], L["din"], L["r"], L["ub"], L["vt"], L["s1"], L["s2"], L["bias"])
            for L in layers]
    bfv = lambda a: orc.bf16_to_f32(orc.f32_to_bf16(a.astype(np.float32)))
    norms = {k: bfv(1.0 + 0.1 * rng.standard_normal(d)) for k in ("input", "post_attention")}
    block = DecoderBlock(ctx, devs, norms["input"], norms["post_attention"], H, Hk, hd, theta, eps, n)
    h = rng.standard_normal((n, d)).astype(np.float32)
    hd_ = torch.from_numpy(h).cuda()
    need = block.prefill_workspace_size(n)
    block.prefill_dev(hd_, n, torch.empty(need, dtype=torch.uint8, device="cuda"), need, torch.cuda.current_stream())
    torch.cuda.synchronize()
    kc, vc = np.zeros((n, Hk * hd), np.float32), np.zeros((n, Hk * hd), np.float32)
    want = orc.block_prefill(layers, norms, h, kc, vc, H, Hk, hd, theta, eps)
    got = hd_.cpu().numpy()
    cos, rel = metrics(got, want)
    assert cos >= COS_MIN and rel <= REL_MAX
    assert max(metrics(got[t], want[t])[1] for t in range(n)) <= 2 * 5 * 2.0 ** -9
    block.close()

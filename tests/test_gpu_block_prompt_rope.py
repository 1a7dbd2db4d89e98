"""GPU: a prompt's RoPE and cache append in 16-byte accesses, sixteen lanes a
head: head counts that leave part of a workgroup idle (4, 5, 15, 48 heads of
q, k and v together, sixteen a workgroup), one row and many, with and without
the q/k norms.  The cache rows against the oracle's, each to what its
roundings allow: four bf16 roundings stand between a row and its cache row
(the norm, t and z of the projection, the q/k norm's operand), a fifth where
the q/k norm rounds its result, each at most 2^-9 of the value; the device and
the oracle may fall apart at each -- 2 x 5 x 2^-9 = 1.95 %."""
import numpy as np
import pytest

from test_gpu_block import metrics, scaled_layer

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,H,Hk,qk_norm", [(1, 2, 1, False), (9, 3, 1, True), (70, 32, 8, True), (67, 13, 1, False)])
def test_prompt_cache_rows(orc, n, H, Hk, qk_norm):
    from quantibbler_amd import DecoderBlock, FactorLayer, GpuContext

    print("prompt rope", n, H, Hk, qk_norm, flush=True)
    ctx = GpuContext(0)
    hd, d, ffn, theta, eps = 128, 256, 256, 500000.0, 1e-5
    rng = np.random.default_rng(100 * n + H)
    shapes = [(H * hd, d, 64), (Hk * hd, d, 32), (Hk * hd, d, 32), (d, H * hd, 64), (ffn, d, 96), (ffn, d, 96),
              (d, ffn, 96)]
    layers = [scaled_layer(orc, rng, *s) for s in shapes]
    devs = [FactorLayer.from_rows(ctx, L["dout"], L["din"], L["r"], L["ub"], L["vt"], L["s1"], L["s2"], L["bias"])
            for L in layers]
    bfv = lambda a: orc.bf16_to_f32(orc.f32_to_bf16(a.astype(np.float32)))
    norms = {k: bfv(1.0 + 0.1 * rng.standard_normal(d)) for k in ("input", "post_attention")}
    heads = {k: bfv(1.0 + 0.1 * rng.standard_normal(hd)) for k in ("q_norm", "k_norm")} if qk_norm else {}
    block = DecoderBlock(ctx, devs, norms["input"], norms["post_attention"], H, Hk, hd, theta, eps, n, **heads)
    h = rng.standard_normal((n, d)).astype(np.float32)
    out = torch.from_numpy(h).cuda()
    need = block.prefill_workspace_size(n)
    block.prefill_dev(out, n, torch.empty(need, dtype=torch.uint8, device="cuda"), need, torch.cuda.current_stream())
    torch.cuda.synchronize()
    kc, vc = np.zeros((n, Hk * hd), np.float32), np.zeros((n, Hk * hd), np.float32)
    want = orc.block_prefill(layers, {**norms, **heads}, h, kc, vc, H, Hk, hd, theta, eps)
    tol = 2 * 5 * 2.0 ** -9
    for ptr, ref in zip(block.cache_ptrs(), (kc, vc)):
        sto = torch._C._construct_storage_from_data_pointer(ptr, torch.device("cuda", 0), n * Hk * hd * 4)
        got = torch.empty(0, dtype=torch.float32, device="cuda").set_(sto, 0, (n, Hk * hd), (Hk * hd, 1)).cpu().numpy()
        assert max(metrics(got[t], ref[t])[1] for t in range(n)) <= tol
    got = out.cpu().numpy()
    assert max(metrics(got[t], want[t])[1] for t in range(n)) <= tol
    block.close()

"""GPU: a prompt's faster kernels against the general ones they stand in for,
bit for bit: norms and RoPE in 16-byte pieces, SwiGLU in the up projection's
epilogue."""
import numpy as np
import pytest

from test_gpu_block import scaled_layer

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def make_block(orc, ctx, seed, d, ffn, H, Hk, capacity, n_seqs=1, qk_norm=False):
    from quantibbler_amd import DecoderBlock, FactorLayer

    hd = 128
    rng = np.random.default_rng(seed)
    shapes = [(H * hd, d, 64), (Hk * hd, d, 32), (Hk * hd, d, 32), (d, H * hd, 64), (ffn, d, 96), (ffn, d, 96),
              (d, ffn, 96)]
    layers = [scaled_layer(orc, rng, *s) for s in shapes]
    devs = [FactorLayer.from_rows(ctx, L["dout"], L["din"], L["r"], L["ub"], L["vt"], L["s1"], L["s2"], L["bias"])
            for L in layers]
    bfv = lambda a: orc.bf16_to_f32(orc.f32_to_bf16(a.astype(np.float32)))
    norms = [bfv(1.0 + 0.1 * rng.standard_normal(d)) for _ in range(2)]
    heads = {k: bfv(1.0 + 0.1 * rng.standard_normal(hd)) for k in ("q_norm", "k_norm")} if qk_norm else {}
    return DecoderBlock(ctx, devs, norms[0], norms[1], H, Hk, hd, 500000.0, 1e-5, capacity, n_seqs=n_seqs, **heads)


def prefill(block, h, shift=0):
    """The prompt's rows after the block, from an h that starts `shift` floats past a 256-byte boundary."""
    n, d = h.shape
    buf = torch.empty(n * d + shift, dtype=torch.float32, device="cuda")
    rows = buf[shift:].view(n, d)
    rows.copy_(torch.from_numpy(h))
    need = block.prefill_workspace_size(n)
    block.prefill_dev(rows, n, torch.empty(need, dtype=torch.uint8, device="cuda"), need, torch.cuda.current_stream())
    torch.cuda.synchronize()
    return rows.cpu().numpy()


@pytest.mark.parametrize("n,d", [(65, 4), (70, 252), (66, 256), (256, 260), (300, 1028), (68, 4096), (67, 4100), (65, 8192)])
def test_norm_in_16_byte_pieces_keeps_the_sums(orc, n, d):
    """A row stream h that is not 16-byte aligned takes the general norm (and the
    element-wise GEMM store): the same prompt leaves the same bits."""
    from quantibbler_amd import GpuContext

    print("prompt norm bits", n, d, flush=True)
    block = make_block(orc, GpuContext(0), n + d, d, 256, 2, 1, n)
    h = np.random.default_rng(n * d).standard_normal((n, d)).astype(np.float32)
    h *= np.exp(np.random.default_rng(d).standard_normal((1, d))).astype(np.float32)
    assert prefill(block, h).tobytes() == prefill(block, h, 1).tobytes()
    block.close()


@pytest.mark.parametrize("n,ffn,r", [(256, 512, 96), (261, 508, 96), (1031, 260, 40), (300, 512, 1100)])
def test_swiglu_in_the_epilogue_is_the_separate_pass(orc, n, ffn, r):
    """The up projection's epilogue forms SwiGLU at an ffn that is a multiple of
    4; two more ffn rows whose gate is 0 (s1 = bias = 0) add zeros to the down
    projection's sums and take the general kernels: f32 rows of gate and up,
    the SwiGLU pass, the down GEMM on f32 rows, the residual's pass."""
    from quantibbler_amd import DecoderBlock, FactorLayer, GpuContext

    print("prompt swiglu bits", n, ffn, r, flush=True)
    ctx, d, H, Hk, hd = GpuContext(0), 256, 2, 1, 128
    rng = np.random.default_rng(n + ffn + r)
    att = [scaled_layer(orc, rng, *s) for s in [(H * hd, d, 64), (Hk * hd, d, 32), (Hk * hd, d, 32), (d, H * hd, 64)]]
    gate, up = scaled_layer(orc, rng, ffn + 2, d, r), scaled_layer(orc, rng, ffn + 2, d, r)
    gate["s1"][ffn:] = gate["bias"][ffn:] = 0.0
    vts = rng.choice([-1, 1], (r, ffn + 2)).astype(np.int8)
    down = scaled_layer(orc, rng, d, ffn + 2, r)
    down["vt"] = orc.pack_bits(vts)
    h = rng.standard_normal((n, d)).astype(np.float32)

    def rows(L, m):
        return dict(L, dout=m, ub=L["ub"][:m], s1=L["s1"][:m], bias=L["bias"][:m])

    outs = []
    for f in (ffn, ffn + 2):
        mlp = [rows(gate, f), rows(up, f),
               dict(down, din=f, vt=orc.pack_bits(np.ascontiguousarray(vts[:, :f])), s2=down["s2"][:f])]
        devs = [FactorLayer.from_rows(ctx, L["dout"], L["din"], L["r"], L["ub"], L["vt"], L["s1"], L["s2"], L["bias"])
                for L in att + mlp]
        ones = np.ones(d, np.float32)
        block = DecoderBlock(ctx, devs, ones, ones, H, Hk, hd, 500000.0, 1e-5, n)
        outs.append(prefill(block, h))
        block.close()
    assert np.isfinite(outs[0]).all() and outs[0].tobytes() == outs[1].tobytes()


@pytest.mark.parametrize("H,Hk,qk_norm", [(2, 1, True), (3, 1, False), (16, 8, True), (13, 1, True)])
def test_rope_in_16_byte_pieces_keeps_the_sums(orc, H, Hk, qk_norm):
    """A prompt's cache rows against those that a batched decode step writes at
    the same positions, one a sequence: its RoPE runs a wave a head, with the
    tree of sums that the prompt's sixteen lanes keep."""
    from quantibbler_amd import GpuContext

    n, d = 8, 256
    print("prompt rope bits", H, Hk, qk_norm, flush=True)
    ctx = GpuContext(0)
    block = make_block(orc, ctx, 10 * H + Hk, d, 256, H, Hk, n, n_seqs=n, qk_norm=qk_norm)
    h = np.random.default_rng(H).standard_normal((n, d)).astype(np.float32)
    width = Hk * 128

    def caches():
        out = []
        for ptr in block.cache_ptrs():
            sto = torch._C._construct_storage_from_data_pointer(ptr, torch.device("cuda", 0), n * n * width * 4)
            out.append(torch.empty(0, dtype=torch.float32, device="cuda")
                       .set_(sto, 0, (n, n, width), (n * width, width, 1)))
        return out

    for c in caches():
        c.zero_()
    prefill(block, h)
    want = [c[0].cpu().numpy() for c in caches()]  # sequence 0's rows 0 .. n - 1
    for c in caches():
        c.zero_()
    block.set_filled(list(range(n)))
    rows = torch.from_numpy(h).cuda()
    need = block.decode_batch_workspace_size(n)
    block.decode_batch_dev(rows, list(range(n)), torch.empty(need, dtype=torch.uint8, device="cuda"), need,
                           torch.cuda.current_stream())
    torch.cuda.synchronize()
    for c, w in zip(caches(), want):
        got = np.stack([c[i, i].cpu().numpy() for i in range(n)])
        assert np.abs(w).sum(axis=1).min() > 0 and got.tobytes() == w.tobytes()
    block.close()


def test_prompt_workspace_holds_two_ffn_rows(orc):
    """The gate projection's f32 rows, and one region for the up projection's or
    the z that its epilogue leaves: 8 bytes for each further ffn row and token."""
    from quantibbler_amd import GpuContext

    ctx, n = GpuContext(0), 300
    need = []
    for ffn in (512, 1024):
        block = make_block(orc, ctx, ffn, 256, ffn, 2, 1, n)
        need.append(block.prefill_workspace_size(n))
        block.close()
    assert need[1] - need[0] == n * 512 * 8

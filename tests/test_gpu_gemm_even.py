"""GPU parity of the prefill FP8 GEMM's 192 x 128, 128 x 192 and 192 x 192
blocks: ragged last blocks in both directions, one to nine k-steps (the
three-stage rings start, fill and wrap), every epilogue.

A row's sums run over K in the same order in every unsplit block, so beside
the oracle (on sampled rows, max |Y - Y_ref| <= 1e-2 x RMS(Y_ref), plus half a
bf16 ulp for bf16 outputs) the whole output must equal, bit for bit, the same
rows computed 64 at a time by the short-prompt blocks.
"""
import numpy as np
import pytest
import torch

from helpers import (activations_bf16, assert_close, bf16_tensor_to_f32,
                     to_torch_bf16)

pytestmark = pytest.mark.gpu

# (block, M, N, K)
CASES = [
    ("192x128", 777, 6144, 128),     # one k-step, last row block of 9 rows
    ("192x128", 768, 6130, 256),     # whole row blocks, ragged N
    ("192x128", 157, 19304, 384),    # one row block, part of it past M
    ("192x128", 385, 10800, 1152),   # last row block of 1 row, ragged N
    ("128x192", 1000, 6100, 1024),   # ragged both ways
    ("192x192", 750, 12200, 1152),   # ragged both ways
]
# The neighbours of the rule's lines keep their blocks.
KEPT = [
    ("256x64", 1024, 4000, 128), ("256x64", 420, 4592, 1152),
    # 200 to 256 tiles of 256 x 64, which 192 x 128 blocks do not beat
    ("256x64", 193, 15000, 1152), ("256x64", 240, 14336, 4096), ("256x64", 512, 8192, 1024),
    ("256x64", 1024, 4096, 4096),
    ("256x128", 1000, 6144, 512), ("256x128", 215, 22512, 1024),
    ("256x192", 750, 12288, 512), ("256x128", 2048, 4096, 1024),
]


def _block(p):
    return f"{p.block_m}x{p.block_n}"


@pytest.mark.parametrize("epi", ["none", "silu", "residual"])
@pytest.mark.parametrize("cfg,m,n,k", CASES)
def test_even_blocks(uh, orc, gpu, cfg, m, n, k, epi):
    w = torch.randn((n, k), generator=torch.Generator().manual_seed(m + n)) * 0.02
    lw = uh.LinearWeight.quantize(w.to(gpu), uh.ENCODING_FP8_E4M3_ROW, gated=epi == "silu")
    q, s = lw.export()
    xb = activations_bf16(orc, m, k, tag=m + 1)
    xq, xs = orc.act_quantize(xb)
    rows = np.unique(np.r_[0, 63, 64, 127, 128, 191, m - 1,
                           np.arange(0, m, 96), np.arange(191, m, 192)].clip(0, m - 1))
    ref = orc.fp8_gemm(xq[rows], xs[rows], q, s)[0]
    res = None
    if epi == "silu":
        ref = orc.silu_mul(ref)
    elif epi == "residual":
        rb = activations_bf16(orc, m, n, tag=m + 2)
        ref = ref + orc.bf16_to_f32(rb[rows])
        res = to_torch_bf16(rb, gpu)
    xq_t, xs_t = torch.from_numpy(xq).to(gpu), torch.from_numpy(xs).to(gpu)
    for dt in (torch.bfloat16, torch.float32):
        y = torch.full((m, ref.shape[1]), float("nan"), dtype=dt, device=gpu)
        r = res if res is None or dt == torch.bfloat16 else res.float()
        kw = {} if r is None else {"residual": r}
        p = lw.plan(xq_t, y, x_scales=xs_t, **kw)
        assert (p.kernel, _block(p), p.split_k) == (uh.KERNEL_GEMM_LDS, cfg, 1)
        assert p.grid == p.tiles <= torch.cuda.get_device_properties(gpu).multi_processor_count
        lw.forward(xq_t, y, x_scales=xs_t, **kw)
        parts = torch.empty_like(y)
        for m0 in range(0, m, 64):
            sl = slice(m0, min(m, m0 + 64))
            kw = {} if r is None else {"residual": r[sl]}
            lw.forward(xq_t[sl], parts[sl], x_scales=xs_t[sl], **kw)
        torch.cuda.synchronize()
        assert torch.equal(y, parts), (cfg, epi, dt)
        got = bf16_tensor_to_f32(y[rows]) if dt == torch.bfloat16 else y[rows].cpu().numpy()
        assert_close(got, ref, bf16_out=dt == torch.bfloat16, what=f"{cfg} {epi} {m}x{n}x{k}")


@pytest.mark.parametrize("cfg,m,n,k", KEPT)
def test_neighbouring_plans(uh, gpu, cfg, m, n, k):
    lw = uh.LinearWeight.quantize(torch.zeros((n, k), device=gpu), uh.ENCODING_FP8_E4M3_ROW)
    x = torch.empty((m, k), dtype=torch.bfloat16, device=gpu)
    y = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    assert _block(lw.plan(x, y, mode=uh.ACT_FP8_PER_TOKEN)) == cfg

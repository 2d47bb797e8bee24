"""GPU parity of the many-row exact products (gemm_wq.hip): bf16 activations
times FP8 or AQ4 weights at M > 16, against the C oracle.

The shapes reach every block configuration (checked through
ullm_linear_forward_plan on a 256-CU device) at the edges where a tile can go
wrong: rows and columns one past a block, K tails of one to three 128-k steps
past the pipeline's four (one to seven where two groups of waves take turns),
an FP8 K that ends inside a step, K shorter than
the waves that split it, strided activations, unaligned outputs, and the fused
epilogues.  Tolerances are the suite's (helpers.assert_close); fp32 outputs
are also held to 1e-5 of their RMS: sums of at most 10752 fp32 products round
to about 1e-7, and AQ4's group offset (16 + z against q) raises that by less
than 30.
"""
import numpy as np
import pytest
import torch

from helpers import (activations_bf16, assert_close, bf16_tensor_to_f32,
                     to_torch_bf16, weights)

pytestmark = pytest.mark.gpu


def _weight(uh, orc, enc, w, gated=False):
    if enc == "fp8":
        enc_w = orc.fp8_quantize_rows(w)
        return uh.LinearWeight.from_fp8(*enc_w, gated=gated), enc_w
    enc_w = orc.aq4_quantize(w)
    return uh.LinearWeight.from_aq4(*enc_w, gated=gated), enc_w


def _ref(orc, enc, xb, enc_w):
    return (orc.fp8_gemv if enc == "fp8" else orc.aq4_gemv)(xb, *enc_w)[0]


def _block(lw, x, y, expect):
    p = lw.plan(x, y)
    assert p.kernel == 3 and p.split_k == 1, "not a block kernel"
    if torch.cuda.get_device_properties(x.device).multi_processor_count == 256:
        assert (p.block_m, p.block_n) == expect, (p.block_m, p.block_n)


# (m, n, k): the block on 256 CUs for (fp8, aq4).
SHAPES = {
    (87, 40, 128): ((32, 32), (16, 32)),
    (33, 129, 64): ((32, 32), (16, 32)),
    (40, 300, 4096): ((16, 32), (16, 32)),
    (70, 1000, 4224): ((16, 32), (16, 32)),
    (38, 4106, 384): ((32, 48), (16, 32)),
    (64, 6000, 2112): ((32, 48), (32, 48)),
    (38, 6855, 640): ((32, 64), (32, 32)),
    (48, 6150, 1280): ((32, 64), (32, 64)),
    (37, 4349, 320): ((32, 48), (16, 32)),
    (129, 4100, 1280): ((32, 128), (32, 48)),
    (67, 6318, 2432): ((32, 96), (32, 96)),
    (38, 9226, 896): ((32, 128), (48, 48)),
    (34, 9188, 1664): ((48, 48), (48, 48)),
    (34, 13626, 1664): ((32, 128), (48, 64)),
    (34, 14658, 2944): ((48, 64), (48, 64)),
    (1162, 806, 1024): ((64, 64), (32, 64)),
    (1167, 770, 1280): ((64, 64), (64, 64)),
    (66, 16580, 256): ((32, 128), (32, 128)),
    (66, 18300, 320): ((32, 128), (32, 128)),
    (38, 6889, 1152): ((32, 64), (32, 64)),
    (38, 5732, 384): ((32, 48), (32, 48)),
    (50, 8524, 2048): ((32, 128), (32, 96)),
    (38, 18311, 256): ((64, 128), (64, 128)),
    (38, 16572, 128): ((32, 128), (64, 128)),
    (38, 17030, 1024): ((64, 128), (64, 128)),
    (38, 17352, 1152): ((64, 128), (64, 128)),
    (37, 16645, 1280): ((64, 128), (64, 128)),
    (38, 17293, 384): ((64, 128), (64, 128)),
    (38, 17463, 640): ((64, 128), (64, 128)),
    (39, 16883, 896): ((64, 128), (64, 128)),
    (37, 17162, 192): ((64, 128), (64, 128)),
    (200, 24661, 256): ((128, 256), (128, 256)),
    (195, 24731, 192): ((128, 256), (128, 256)),
    (321, 27266, 256): ((64, 128), (128, 384)),
    (387, 23495, 384): ((64, 128), (128, 384)),
    # 17 to 32 rows on one round of strips
    (17, 129, 4224): ((16, 32), (16, 32)),
    (31, 4090, 4224): ((16, 32), (16, 32)),
    (32, 480, 10752): ((16, 32), (16, 32)),
    (24, 300, 2048): ((16, 32), (16, 32)),
    (32, 2041, 2176): ((16, 32), (16, 32)),
}
# Calls beside that rule's lines, left to the decode kernels.
DECODE = [(16, 480, 8192), (23, 300, 4096), (24, 300, 1920), (32, 2060, 4096),
          (32, 4100, 4224), (17, 1000, 12288)]


@pytest.mark.parametrize("m,n,k", DECODE)
@pytest.mark.parametrize("enc", ["fp8", "aq4"])
def test_few_rows_stay_decode(uh, gpu, enc, m, n, k):
    lw = uh.LinearWeight.quantize(torch.zeros((n, k), device=gpu), 1 if enc == "fp8" else 2)
    x = torch.empty((m, k), dtype=torch.bfloat16, device=gpu)
    assert lw.plan(x, torch.empty((m, n), device=gpu)).kernel == uh.KERNEL_GEMV


@pytest.mark.parametrize("m,n,k", list(SHAPES))
@pytest.mark.parametrize("enc", ["fp8", "aq4"])
def test_wq_gemm_parity(uh, orc, gpu, enc, m, n, k):
    if enc == "aq4" and k % 128:
        pytest.skip("AQ4 K is a multiple of 128")
    lw, enc_w = _weight(uh, orc, enc, weights(n, k, tag=51))
    xb = activations_bf16(orc, m, k, tag=m + 400)
    y_ref = _ref(orc, enc, xb, enc_w)
    x = to_torch_bf16(xb, gpu)
    y32 = torch.full((m, n), float("nan"), device=gpu)
    lw.forward(x, y32)
    _block(lw, x, y32, SHAPES[(m, n, k)][enc == "aq4"])
    # Bound: the oracle adds K products one after the other in fp32, so its own
    # sums deviate by about 2^-24 sqrt(K / 6) of their RMS (random rounding of
    # partial sums that grow as sqrt(j / K)); 8 x 2^-24 sqrt(K) is 19 of these
    # deviations.  Its largest error against 64-bit sums is 1.28e-5 RMS at
    # 31 x 4090 x 4224 (bound 3.1e-5) and 1.38e-5 at 32 x 480 x 10752 (4.9e-5).
    rel = max(1e-5, 8 * 2.0 ** -24 * k ** 0.5) if m <= 32 else 1e-5
    assert_close(y32.cpu().numpy(), y_ref, rel=rel, what=f"{enc} f32 {m}x{n}x{k}")
    yb = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu)
    lw.forward(x, yb)
    assert_close(bf16_tensor_to_f32(yb), y_ref, bf16_out=True, what=f"{enc} bf16 {m}x{n}x{k}")


# FP8 K of 8 i + 7 tiles of 64: a whole number of four-step rounds whose last
# step is half one.  (m, n, k) for each block of 8 waves.
HALF_STEPS = [
    ((32, 128), 37, 6564, 448), ((32, 128), 40, 8250, 960), ((32, 128), 34, 8255, 1472),
    ((32, 128), 65, 8314, 4032),
    ((64, 128), 37, 17140, 448), ((64, 128), 37, 17117, 960), ((64, 128), 35, 16407, 1472),
    ((64, 128), 40, 19069, 4032),
    ((128, 256), 129, 26336, 448), ((128, 256), 129, 26171, 960), ((128, 256), 130, 26261, 1472),
    ((128, 256), 129, 26266, 4032),
    ((64, 128), 259, 26239, 448), ((64, 128), 258, 26363, 960), ((64, 128), 257, 21942, 1472),
    ((64, 128), 257, 22039, 4032),
]


@pytest.mark.parametrize("block,m,n,k", HALF_STEPS)
def test_wq_gemm_half_last_step(uh, orc, gpu, block, m, n, k):
    """Nothing past K counts: not the next stripe's weights, and neither the
    columns beside a strided x nor the next row (both NaN or inf here)."""
    lw, enc_w = _weight(uh, orc, "fp8", weights(n, k, tag=63))
    xb = activations_bf16(orc, m, k, tag=m + 450)
    rows = np.unique(np.r_[0, 4, 15, 31, 32, np.arange(0, m, 37), m - 2, m - 1])
    y_ref = _ref(orc, "fp8", np.ascontiguousarray(xb[rows]), enc_w)
    x = to_torch_bf16(xb, gpu)
    wide = torch.full((m, k + 64), float("nan"), dtype=torch.bfloat16, device=gpu)
    wide[:, :k] = x
    y = torch.full((m, n), float("nan"), device=gpu)
    _block(lw, x, y, block)
    lw.forward(x, y)
    # The bound of test_wq_gemm_parity.
    rel = max(1e-5, 8 * 2.0 ** -24 * k ** 0.5)
    assert_close(y[rows].cpu().numpy(), y_ref, rel=rel, what=f"{block} {m}x{n}x{k}")
    assert torch.equal(lw.forward(wide[:, :k], out_dtype=torch.float32), y)
    bad = x.clone()
    bad[5], bad[33] = float("nan"), float("inf")
    y2 = lw.forward(bad, out_dtype=torch.float32)
    keep = torch.ones(m, dtype=torch.bool, device=gpu)
    keep[5] = keep[33] = False
    assert torch.equal(y2[keep], y[keep])


@pytest.mark.parametrize("block,m,n,k", [
    ((32, 128), 79, 21001, 12416), ((64, 128), 410, 3813, 14208),
    ((128, 256), 1421, 2873, 12032),
])
def test_wq_gemm_fp8_sum_error(uh, gpu, block, m, n, k):
    """The 8-wave FP8 blocks add up in two levels (four steps of 128 k, then
    these), so their error stays below that of one chain over K.

    An fp32 addition whose result is S rounds by c |S| RMS, c = 2^-24
    sqrt(0.541 / 3) = 2.53e-8 (mean square of an error uniform in half an ulp,
    mantissas uniform in the logarithm).  A chain of j equal parts of a sum S
    costs c^2 S^2 j / 2.  Two levels: K / 512 parts of 4 steps of 4 matrix
    instructions, and two roundings at the end (scale and alpha), c^2
    (K / 1024 + 2 + 2 + 2); one chain of steps instead: c^2 (K / 256 + 2 + 2),
    1.7 times the error at these K.  10 % are allowed for the inputs.
    """
    g = torch.Generator(device=gpu).manual_seed(n)
    w = torch.randn((n, k), generator=g, device=gpu) * 0.02
    x = torch.randn((m, k), generator=g, device=gpu).to(torch.bfloat16)
    s = w.abs().amax(dim=1) / 448.0
    q = (w / s[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    lw = uh.LinearWeight.from_fp8(q.view(torch.uint8), s)
    y = torch.empty((m, n), device=gpu)
    _block(lw, x, y, block)
    lw.forward(x, y)
    rows = torch.arange(0, m, max(1, m // 40), device=gpu)
    ref = x[rows].double() @ (q.double() * s.double()[:, None]).T
    err = float((y[rows].double() - ref).norm() / ref.norm())
    assert err <= 1.1 * 2.53e-8 * (k / 1024 + 6) ** 0.5, err


@pytest.mark.parametrize("m,n", [(50, 1100), (300, 2056)])
@pytest.mark.parametrize("enc", ["fp8", "aq4"])
def test_wq_gemm_strided_and_unaligned(uh, orc, gpu, enc, m, n):
    """x a column slice of a wider buffer whose other columns are NaN, y a
    column slice at an odd offset (no 16-byte rows), values outside both
    untouched; a strip block and an 8-wave block."""
    k = 640
    lw, enc_w = _weight(uh, orc, enc, weights(n, k, tag=53))
    xb = activations_bf16(orc, m, k, tag=m + 410)
    y_ref = _ref(orc, enc, xb, enc_w)
    wide = torch.full((m, k + 24), float("nan"), dtype=torch.bfloat16, device=gpu)
    wide[:, 8:8 + k] = to_torch_bf16(xb, gpu)
    for dt in (torch.bfloat16, torch.float32):
        buf = torch.full((m, n + 5), 7.0, dtype=dt, device=gpu)
        y = buf[:, 3:3 + n]
        _block(lw, wide[:, 8:8 + k], y, (32, 128) if m > 64 else
               (32, 32) if enc == "fp8" else (16, 32))
        lw.forward(wide[:, 8:8 + k], y)
        assert_close(bf16_tensor_to_f32(y.contiguous()), y_ref, bf16_out=dt == torch.bfloat16,
                     what=f"{enc} strided")
        assert torch.all(buf[:, :3] == 7.0) and torch.all(buf[:, 3 + n:] == 7.0)


@pytest.mark.parametrize("m,n", [(37, 1040), (300, 2064)])
@pytest.mark.parametrize("enc", ["fp8", "aq4"])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_wq_gemm_epilogues(uh, orc, gpu, enc, m, n, out):
    """SiLU-gate (F not a multiple of the block) and an in-place residual,
    with alpha, in a strip block and an 8-wave block."""
    k = 384
    w = weights(n, k, tag=57)
    xb = activations_bf16(orc, m, k, tag=m + 420)
    x = to_torch_bf16(xb, gpu)
    lw, enc_w = _weight(uh, orc, enc, w)
    y_ref = 0.5 * _ref(orc, enc, xb, enc_w).astype(np.float64)
    r = torch.randn((m, n), generator=torch.Generator().manual_seed(3)).to(out)
    y = r.clone().to(gpu)
    _block(lw, x, y, (32, 128) if m > 64 else (32, 32) if enc == "fp8" else (16, 32))
    lw.forward(x, y, residual=y, alpha=0.5)
    assert_close(bf16_tensor_to_f32(y), y_ref + r.double().numpy(),
                 bf16_out=out == torch.bfloat16, what=f"{enc} residual")
    lg, enc_g = _weight(uh, orc, enc, w, gated=True)
    p = 0.5 * _ref(orc, enc, xb, enc_g).astype(np.float64)
    g, u = p[:, :n // 2], p[:, n // 2:]
    yg = lg.forward(x, out_dtype=out, alpha=0.5)
    assert_close(bf16_tensor_to_f32(yg), g / (1 + np.exp(-g)) * u,
                 bf16_out=out == torch.bfloat16, what=f"{enc} gated")


# (encoding, block, m, n, k) with rows of 16-byte segments (N and F multiples
# of 8) and part of the last block past M and past N.
SEGMENTS = [
    ("fp8", (32, 128), 300, 2064, 384), ("aq4", (32, 128), 300, 2064, 384),
    ("fp8", (64, 128), 65, 11072, 256), ("aq4", (64, 128), 129, 20000, 640),
    ("aq4", (64, 128), 100, 12000, 640),  # two groups of waves over K
    ("fp8", (128, 256), 200, 24688, 384), ("aq4", (128, 256), 200, 24688, 384),
    ("aq4", (128, 384), 321, 27280, 384),
]


@pytest.mark.parametrize("epi", ["none", "silu", "residual"])
@pytest.mark.parametrize("enc,block,m,n,k", SEGMENTS)
def test_wq_gemm_segment_stores(uh, orc, gpu, enc, block, m, n, k, epi):
    """The 8-wave blocks' bf16 rows leave in 16-byte segments, whole and cut at
    the edges: the same bits as the fp32 output rounded, which is held to the
    oracle on sampled rows, and nothing written beside them."""
    lw, enc_w = _weight(uh, orc, enc, weights(n, k, tag=65), gated=epi == "silu")
    xb = activations_bf16(orc, m, k, tag=m + 460)
    rows = np.unique(np.r_[0, 15, 16, 31, 32, np.arange(0, m, 41), m - 1].clip(0, m - 1))
    ref = 0.5 * _ref(orc, enc, np.ascontiguousarray(xb[rows]), enc_w).astype(np.float64)
    x = to_torch_bf16(xb, gpu)
    cols = n
    if epi == "silu":
        cols = n // 2
        ref = ref[:, :cols] / (1 + np.exp(-ref[:, :cols])) * ref[:, cols:]
    buf = torch.full((m + 1, cols + 8), 7.0, dtype=torch.bfloat16, device=gpu)
    y = buf[:m, :cols]
    y32 = torch.full((m, cols), float("nan"), device=gpu)
    kw, kw32 = {}, {}
    if epi == "residual":
        y.copy_(torch.randn((m, n), generator=torch.Generator().manual_seed(m)))
        kw, kw32 = {"residual": y}, {"residual": y.float()}
        ref = ref + y[rows].double().cpu().numpy()
    _block(lw, x, y, block)
    lw.forward(x, y32, alpha=0.5, **kw32)
    lw.forward(x, y, alpha=0.5, **kw)
    assert_close(y32[rows].cpu().numpy(), ref, what=f"{enc} {block} {epi}")
    assert torch.equal(y, y32.to(torch.bfloat16))
    assert torch.all(buf[:, cols:] == 7.0) and torch.all(buf[m] == 7.0)


@pytest.mark.parametrize("enc", ["fp8", "aq4"])
def test_wq_gemm_captured(uh, orc, gpu, enc):
    """No scratch: workspace_size is 0, and a captured launch replays on new
    inputs."""
    m, n, k = 70, 528, 1024
    lw, _ = _weight(uh, orc, enc, weights(n, k, tag=59))
    assert lw.workspace_size(m) == 0
    x = torch.zeros((m, k), dtype=torch.bfloat16, device=gpu)
    y = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        lw.forward(x, y)
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            lw.forward(x, y)
    for i in range(3):
        x.copy_(to_torch_bf16(activations_bf16(orc, m, k, tag=i + 430), gpu))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, lw.forward(x))


@pytest.mark.parametrize("enc", ["fp8", "aq4"])
def test_wq_gemm_rows_are_independent(uh, orc, gpu, enc):
    """A row of inf or NaN leaves the other rows' results as they are."""
    for m, n in ((40, 300), (260, 2000)):
        k = 512
        lw, _ = _weight(uh, orc, enc, weights(n, k, tag=61))
        x = to_torch_bf16(activations_bf16(orc, m, k, tag=440), gpu)
        y = lw.forward(x)
        x2 = x.clone()
        x2[5, 17], x2[33, 100] = float("inf"), float("nan")
        y2 = lw.forward(x2)
        keep = torch.ones(m, dtype=torch.bool, device=gpu)
        keep[5] = keep[33] = False
        assert torch.equal(y[keep], y2[keep])
        assert not torch.any(torch.isfinite(y2[33].float()))

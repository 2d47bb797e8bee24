"""GPU: quantize, pack, export and dequantize of whole wave tiles, bit for bit
against the C oracle, where those kernels change path: K at and past each
register depth of the FP8 quantizer (1024, 2048, 4096 and longer), K that does
not fill a tile or a 16-byte access, sources and results that are not 16-byte
aligned, gated-pair rows with padding in the middle, and rows that leave the
plain encode (inf, NaN, subnormal scales)."""
import numpy as np
import pytest
import torch

from helpers import weights

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("n,k", [(16, 1024), (17, 1088), (5, 2048), (33, 2052), (16, 4096),
                                 (31, 4100), (40, 4097), (20, 9000)])
@pytest.mark.parametrize("gated", [False, True])
def test_fp8_tiles(uh, orc, gpu, n, k, gated):
    n += n % 2 if gated else 0
    w = weights(n, k, tag=71)
    w[1 % n] *= 1e-30
    q_ref, s_ref = orc.fp8_quantize_rows(w)
    src = torch.empty(n * k + 1, device=gpu)
    for off in (0, 1):  # aligned, and one float past it
        v = src[off:off + n * k].view(n, k)
        v.copy_(torch.from_numpy(w))
        lw = uh.LinearWeight.quantize(v, uh.ENCODING_FP8_E4M3_ROW, gated=gated)
        q, s = lw.export()
        assert np.array_equal(q, q_ref) and np.array_equal(_bits(s), _bits(s_ref))
    d_ref = _bits(orc.fp8_dequantize(q_ref, s_ref))
    assert np.array_equal(_bits(lw.dequantize().cpu()), d_ref)
    # encoded bytes in device memory, aligned or not
    buf = torch.empty(n * k + 1, dtype=torch.uint8, device=gpu)
    sd = torch.from_numpy(s_ref).to(gpu)
    for off in (0, 1):
        b = buf[off:off + n * k].view(n, k)
        b.copy_(torch.from_numpy(q_ref))
        l2 = uh.LinearWeight.from_fp8(b, sd, gated=gated)
        assert np.array_equal(_bits(l2.dequantize().cpu()), d_ref)


@pytest.mark.parametrize("n,k", [(16, 128), (15, 384), (18, 4096), (40, 1152)])
@pytest.mark.parametrize("gated", [False, True])
def test_aq4_tiles(uh, orc, gpu, n, k, gated):
    n += n % 2 if gated else 0
    w = weights(n, k, tag=73)
    w[0, :128] = -0.5                       # constant group
    w[n - 1, :128] = np.linspace(0, 1e-7, 128)  # scale near the f16 subnormals
    p_ref, s_ref, z_ref = orc.aq4_quantize(w)
    src = torch.empty(n * k + 1, device=gpu)
    for off in (0, 1):
        v = src[off:off + n * k].view(n, k)
        v.copy_(torch.from_numpy(w))
        lw = uh.LinearWeight.quantize(v, uh.ENCODING_AQ4_G128, gated=gated)
        p, s, z = lw.export()
        assert np.array_equal(p, p_ref) and np.array_equal(s, s_ref)
        assert np.array_equal(z, z_ref)
    l2 = uh.LinearWeight.from_aq4(p_ref, s_ref, z_ref, gated=gated)
    d_ref = _bits(orc.aq4_dequantize(p_ref, s_ref, z_ref))
    assert np.array_equal(_bits(l2.dequantize().cpu()), d_ref)
    assert np.array_equal(_bits(lw.dequantize().cpu()), d_ref)


def test_fp8_rows_off_the_plain_encode(uh, orc, gpu):
    """Rows with inf or NaN, a subnormal scale (quotients past 449), exact
    ties and values one rounding past 448 encode as the oracle does."""
    k = 320
    w = weights(8, k, tag=75)
    w[0, 3], w[0, 4] = np.inf, -1.0
    w[1, 100] = np.nan
    w[2] = np.nan
    w[3] = np.float32(1e-45) * np.arange(k) * 3
    w[4] = np.float32(1e-38) * np.linspace(-1, 1, k)
    w[5, :16] = [448, -448, 447.99997, 440, 432, 424, 17, 19, 0.0029296875, -0.0009765625,
                 0.015625, 0.0146484375, 1e-9, -1e-9, 0.0, -0.0]
    w[5, 16:] = 0.0
    w[6] = 0.0
    with np.errstate(all="ignore"):
        q_ref, s_ref = orc.fp8_quantize_rows(w)
    lw = uh.LinearWeight.quantize(torch.from_numpy(w).to(gpu), uh.ENCODING_FP8_E4M3_ROW)
    q, s = lw.export()
    assert np.array_equal(_bits(s), _bits(s_ref))
    assert np.array_equal(q, q_ref)


@pytest.mark.parametrize("n,k,gated", [(16, 128, False), (15, 384, False), (4096, 1024, False),
                                       (18, 256, True), (1000, 4096, True)])
def test_device_bytes(uh, gpu, n, k, gated):
    """A weight holds its padded rows once: half a byte (AQ4) or a byte (FP8)
    per element, and a scale|zero word per group or a scale per row."""
    n16 = 2 * -(-(n // 2) // 8) * 8 if gated else -(-n // 16) * 16
    w = torch.zeros((n, k), device=gpu)
    for enc, expect in ((uh.ENCODING_AQ4_G128, n16 * k // 2 + n16 * (k // 128) * 4),
                        (uh.ENCODING_FP8_E4M3_ROW, n16 * k + n16 * 4)):
        assert uh.LinearWeight.quantize(w, enc, gated=gated).info().device_bytes == expect

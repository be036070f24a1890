"""GPU parity of the block-scaled linear operators against the oracle.

lin_pq   src/ext/mxfp4_decode.cu:135-170   (grouped GEMV for M <= 16, MFMA GEMM above)
forward  src/ext/mxfp4_linear.cu:106-198   (fp16 rounding + quantize + GEMM)

Tolerances: per-op (same quantized operands) cos >= 0.99999, max-rel <= 1e-4
(tests/gpu_helpers.py), tighter than the north-star cos >= 0.999 / 1e-2.
"""
import numpy as np
import pytest
import torch

from oracle import mxfp4 as fmt
from oracle import ops
from moe_fused_inference_amd import _lib
from tests.gpu_helpers import DEV, assert_close, log, np_

pytestmark = pytest.mark.gpu


def _w(dext, N, K, seed):
    rng = np.random.default_rng(seed)
    W = rng.standard_normal((N, K)).astype(np.float32)
    W *= np.power(2.0, rng.integers(-1, 2, size=(N, 1))).astype(np.float32)
    wq, ws = fmt.quantize_rows(W)
    return torch.from_numpy(wq).to(DEV), torch.from_numpy(ws).to(DEV), wq, ws


# shapes of tests/correctness/test_mxfp4_decode.py:78-79 plus GEMM-path shapes
LIN_SHAPES = [(1, 32, 64), (1, 768, 2048), (1, 2048, 768), (3, 128, 100), (1, 4096, 2048),
              (2, 2048, 2048), (16, 64, 96), (17, 64, 256), (128, 128, 256), (200, 300, 1000),
              (129, 257, 40), (512, 1536, 2048), (300, 520, 768), (2048, 2048, 768),
              (2048, 4096, 512), (2000, 4000, 768),   # these two on the 256 x 256 tile GEMM
              # ragged edges on the 128 x 128 ring (192 tiles) and the 4-stage 64 x 64 ring (270 tiles);
              # (512, 1536, 2048), (17, 64, 256) and (300, 520, 768) run on the 8-stage 64 x 64 ring
              (1000, 3000, 512), (1100, 900, 1024),
              # small-M split-K GEMV: K in 16 / 8 / 4 parts, unsplit with 4 row tiles, odd step count
              (1, 128, 2048), (1, 2048, 4096), (1, 5120, 2048), (3, 20000, 2048), (5, 1000, 4160),
              (8, 136, 2048), (40, 48, 96)]


@pytest.mark.parametrize("M,N,K", LIN_SHAPES)
def test_lin_pq_vs_oracle(dext, M, N, K):
    rng = np.random.default_rng(M + N + K)
    wp, wsc, wq, ws = _w(dext, N, K, seed=N * 31 + K)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32) * 0.5).to(DEV).bfloat16()
    xq, xs = dext.prequant(x)
    y = dext.lin_pq(xq, xs, wp, wsc, M, N, K)
    torch.cuda.synchronize()
    ref = ops.lin_pq_ref(np_(xq), np_(xs), wq, ws)
    assert y.shape == (M, N) and y.dtype == torch.float32
    assert_close(np_(y), ref, what=f"lin_pq M={M} N={N} K={K}")


# shapes of tests/correctness/test_mxfp4_mma.py:74-100 plus config-3 shapes
FWD_SHAPES = [(16, 8, 64), (16, 8, 100), (16, 8, 40), (1, 8, 64), (1, 32, 64), (16, 32, 64),
              (32, 32, 64), (8, 64, 2048), (1, 768, 2048), (8, 2048, 768), (2048, 2048, 768)]


# M > 16 with Kp % 256 != 0: one block and one short of a step, scale rows that start at any byte of a dword,
# a tail after full steps on each tile size (64 x 64; 64 x 128 from (1100, 900) on; 128 x 128 and 256 x 256 the last two)
RAGGED_SHAPES = [(17, 33, 32), (65, 127, 224), (333, 1000, 2080), (100, 129, 1312 + 256), (200, 64, 2048 + 96),
                 (1100, 900, 544), (1500, 2100, 800), (3000, 3100, 288), (2600, 4100, 1568)]


# the tile rule's other sides: M up to one and just past one 64- and 128-row tile with many columns, 144 and 160 tiles of
# 256 x 256, K on both sides of 1024 and 1536
@pytest.mark.parametrize("M,N,K", [(64, 5000, 512), (65, 10300, 512), (129, 5300, 1024), (2300, 4000, 1536), (2500, 4090, 1536),
                                   (2300, 2500, 1280), (520, 5121, 2048),
                                   # a long K with one 128 x 128 a CU: full tiles, ragged ones, one XCD short of them; 135 tiles of
                                   # 256 x 256 without padding; two stages of 128 x 128 below 160 tiles
                                   (1024, 4096, 2048), (1000, 4001, 2304), (500, 5900, 3072), (2304, 3840, 3072), (1500, 1300, 512)])
def test_lin_pq_tile_rule_vs_oracle(dext, M, N, K):
    test_lin_pq_vs_oracle(dext, M, N, K)


@pytest.mark.parametrize("M,N,K", RAGGED_SHAPES)
def test_lin_pq_ragged_k_vs_oracle(dext, M, N, K):
    test_lin_pq_vs_oracle(dext, M, N, K)


# the streaming GEMV of a many-row weight: its smallest sizes at each K, a last tile of one row, waves with a tile fewer,
# one to sixteen activation rows; `part`: rows of a slice that is too short to stream and long enough to leave K whole
# (1024 tiles and more; at K = 4096 so many stream)
@pytest.mark.parametrize("M,N,K,part", [(1, 32784, 2048, 16384), (3, 32768, 2048, 16384), (8, 131089, 1024, 65536),
                                        (16, 22001, 3072, 16384), (5, 16400, 4096, None), (1, 40001, 4096, None)])
def test_lin_pq_streamed_rows(dext, M, N, K, part):
    """Equal, bit for bit, to the same rows as slices of fewer rows, which
    take the kernel of a tile per wave (its unsplit instance: the same MFMA
    chain); the last slice ends at N.  Where there is none, every row against
    the oracle."""
    g = torch.Generator(device=DEV)
    g.manual_seed(M + N)
    wp, wsc = dext.prequant(torch.randn((N, K), generator=g, device=DEV).bfloat16())
    xq, xs = dext.prequant(torch.randn((M, K), generator=g, device=DEV).bfloat16())
    y = dext.lin_pq(xq, xs, wp, wsc, M, N, K)
    if part:
        for n0 in [*range(0, N - part, part), N - part]:   # (N - part: any row may be a slice's first)
            n1 = n0 + part
            assert torch.equal(dext.lin_pq(xq, xs, wp[n0:n1].contiguous(), wsc[n0:n1].contiguous(), M, part, K), y[:, n0:n1])
        rows = torch.cat((torch.arange(0, 300), torch.arange(N - 300, N))).to(DEV)
    else:
        rows = torch.arange(N, device=DEV)
    # against fp32 products of the same operands, summed in fp64
    want = ops.lin_pq_ref_chunked(np_(xq), np_(xs), np_(wp[rows]), np_(wsc[rows]))
    assert_close(np_(y[:, rows]), want, what=f"lin_pq streamed {M}x{N}x{K}")


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_lin_pq_ragged_scales_at_any_byte(dext, shift):
    """Scale tensors that start inside a dword give the bits of aligned ones."""
    M, N, K = 70, 150, 1120
    wp, wsc, _, _ = _w(dext, N, K, seed=71)
    g = torch.Generator(device=DEV)
    g.manual_seed(72)
    xq, xs = dext.prequant(torch.randn((M, K), generator=g, device=DEV).bfloat16())

    def moved(t, by):
        buf = torch.zeros(t.numel() + 8, dtype=torch.uint8, device=DEV)
        v = buf[by:by + t.numel()].view(t.shape)
        v.copy_(t)
        return v

    want = dext.lin_pq(xq, xs, wp, wsc, M, N, K)
    assert torch.equal(dext.lin_pq(xq, moved(xs, shift), wp, moved(wsc, 4 - shift), M, N, K), want)


@pytest.mark.parametrize("M,N,K", FWD_SHAPES)
@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16])
def test_forward_vs_oracle(lext, M, N, K, xdt):
    rng = np.random.default_rng(M * 3 + N * 5 + K)
    wp, wsc, wq, ws = _w(None, N, K, seed=N + K)
    x = rng.standard_normal((M, K)).astype(np.float32) * 0.5
    x[rng.random((M, K)) < 0.005] *= 4.0
    xt = torch.from_numpy(x).to(DEV).to(xdt)
    y = lext.forward(xt, wp, wsc)
    torch.cuda.synchronize()
    ref = ops.forward_ref(np_(xt.float()), wq, ws)
    assert_close(np_(y), ref, what=f"forward {xdt} M={M} N={N} K={K}")


def test_forward_equals_prequant_then_lin_pq(dext, lext):
    """Structural: forward == quantize(fp16(x)) then lin_pq, bit for bit."""
    rng = np.random.default_rng(9)
    M, N, K = 64, 512, 2048
    wp, wsc, _, _ = _w(dext, N, K, seed=5)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(DEV).half()
    y1 = lext.forward(x, wp, wsc)
    lib = _lib.load()
    Kp = 2048
    xq = torch.empty((M, Kp // 2), dtype=torch.uint8, device=DEV)
    xs = torch.empty((M, Kp // 32), dtype=torch.uint8, device=DEV)
    assert lib.mxfp4_quantize_rows(x.data_ptr(), 1, 1, K, M, K, Kp, xq.data_ptr(), xs.data_ptr(),
                                   torch.cuda.current_stream().cuda_stream) == 0
    y2 = dext.lin_pq(xq, xs, wp, wsc, M, N, K)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2)


def test_config3_largest_gemm_north_star(lext):
    """(4096, 4096, 2048), activations bf16 N(0,1) quantized on the fly, weights
    MXFP4 from bf16 N(0,0.02): per-op tolerance against the oracle."""
    M, N, K = 4096, 4096, 2048
    g = torch.Generator(device=DEV)
    g.manual_seed(30)
    x = torch.randn((M, K), generator=g, device=DEV).bfloat16()
    w = (torch.randn((N, K), generator=g, device=DEV) * 0.02).bfloat16()
    wq, ws = fmt.quantize_rows(np_(w.float()))
    y = lext.forward(x, torch.from_numpy(wq).to(DEV), torch.from_numpy(ws).to(DEV))
    torch.cuda.synchronize()
    ref = ops.forward_ref(np_(x.float()), wq, ws)
    assert_close(np_(y), ref, what="forward 4096x4096x2048")

"""The GEMM on 16x16 and 32x32 tiles whose waves share the reduction
(csrc/gemm_small.hip), against the oracle's fp32 product of the same
dequantized operands (dnn/layers/fully_connected_layer.cu:14-65) at the
path's bar (1e-4), on every row.

Shapes: one value short of, on and past the tile edges (16, 32) in M and N;
K within one step, on a step's edge, one 16-byte chunk past it, not a
multiple of 16, fewer steps than waves; more than one round of steps (a wave's
slab written again after it was read) for each tiling and wave count, whole
rounds and a partial last one; outputs whose rows are not 16-byte aligned.
The operands' leading dimensions hold codes past K that must not be read.
"""
import numpy as np
import pytest
import torch

import deepfuse_amd as df
from deepfuse_amd import Fmt, synth
from oracle import pyoracle as orc
from test_gpu_gemm import TOL, band_rows, check_bf16_image, quant_operand

pytestmark = pytest.mark.gpu

# M, N, K, the tile and the waves of a block
CASES = [(1, 1, 5, 16, 4), (1, 17, 128, 16, 4), (15, 16, 144, 16, 4), (16, 33, 127, 16, 4), (17, 1601, 272, 32, 4),
         (8, 1600, 1600, 16, 4), (8, 640, 6400, 16, 4), (31, 2049, 640, 32, 4), (32, 2048, 512, 32, 4),
         (33, 3072, 784, 32, 4), (64, 3072, 768, 32, 4), (63, 1600, 3072, 16, 4), (97, 130, 2064, 16, 4),
         (512, 768, 768, 32, 4), (300, 257, 1040, 32, 8), (300, 130, 1024, 16, 4), (2048, 640, 2048, 32, 4),
         (512, 768, 3072, 32, 4), (1000, 771, 1037, 32, 4), (512, 512, 3088, 32, 8), (255, 769, 3072, 32, 8),
         (102, 1808, 12112, 32, 8), (102, 200, 12112, 16, 4)]


@pytest.mark.parametrize("M,N,K,tile,waves", CASES)
@pytest.mark.parametrize("fa,fb", [(Fmt.E4M3, Fmt.E4M3), (Fmt.E5M2, Fmt.E4M3)])
def test_small_tiles_match_oracle(dev, M, N, K, tile, waves, fa, fb):
    seed = synth.SEED_BASE + 31 * M + 7 * N + K
    A = synth.normal((M, K), 1.0, seed=seed)
    B = synth.normal((N, K), 0.02, seed=seed + 1)
    bb = synth.f32_to_bf16_bits(synth.normal((N,), 0.1, seed=seed + 2))
    aq, _, sa, Ad = quant_operand(A, fa, dev)
    bq, _, sb, Bd = quant_operand(B, fb, dev)
    # wider rows, filled with a non-zero code behind K's 16-byte granule
    kp = df.round16(K)
    wide = [torch.full((t.shape[0], kp + 48), 0x38, dtype=torch.uint8, device=dev) for t in (aq, bq)]
    for dst, src in zip(wide, (aq, bq)):
        dst[:, :kp].copy_(src)
    aq, bq = wide[0][:, :kp], wide[1][:, :kp]
    bd = torch.from_numpy(bb.view(np.int16)).to(dev).view(torch.bfloat16)
    plan = df.gemm_plan(M, N, K, aq.stride(0), bq.stride(0), bd, 1 << 30)
    assert plan == (df.GemmKernel.SMALL_16 if tile == 16 else df.GemmKernel.SMALL_32, waves), f"plan {plan!r}"
    Y = df.gemm_nt(aq, fa, bq, fb, K, sa, sb, bias=bd)
    ref = orc.fc_forward(Ad, Bd, orc.bf16_to_f32(bb))
    err = orc.rel_err(Y.cpu().numpy(), ref)
    assert err <= TOL, f"M={M} N={N} K={K}: rel err {err:.3e}"
    check_bf16_image(Y, df.gemm_nt(aq, fa, bq, fb, K, sa, sb, bias=bd, out_dtype=torch.bfloat16))
    # binary16: the RNE image too (an f16 output takes an fp32 bias of the same values)
    b32 = torch.from_numpy(orc.bf16_to_f32(bb)).to(dev)
    Y16 = df.gemm_nt(aq, fa, bq, fb, K, sa, sb, bias=b32, out_dtype=torch.float16)
    img = orc.convert(np.ascontiguousarray(Y.cpu().numpy()), 0, 1).reshape(M, N)
    assert np.array_equal(Y16.view(torch.int16).cpu().numpy().view(np.uint16), img)
    # no bias, and a second call gives the same bits
    n1 = df.gemm_nt(aq, fa, bq, fb, K, sa, sb)
    assert orc.rel_err(n1.cpu().numpy(), orc.fc_forward(Ad, Bd, None)) <= TOL
    assert torch.equal(n1, df.gemm_nt(aq, fa, bq, fb, K, sa, sb))


def test_output_rows_apart(dev):
    """ldc > N: the columns between rows are left alone."""
    M, N, K, ldc = 40, 50, 300, 67
    A, B = synth.normal((M, K), 1.0, seed=3), synth.normal((N, K), 0.02, seed=4)
    aq, _, sa, Ad = quant_operand(A, Fmt.E4M3, dev)
    bq, _, sb, Bd = quant_operand(B, Fmt.E4M3, dev)
    C = torch.full((M, ldc), 7.0, device=dev)
    df.call("df_fp8_gemm_nt", 0, aq.data_ptr(), aq.stride(0), 0, bq.data_ptr(), bq.stride(0), M, N, K, sa.data_ptr(),
            sb.data_ptr(), 0, None, 0, C.data_ptr(), ldc, None, 0, torch.cuda.current_stream().cuda_stream)
    assert orc.rel_err(C[:, :N].cpu().numpy(), orc.fc_forward(Ad, Bd, None)) <= TOL
    assert bool((C[:, N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(4001, 999, 640), (4001, 1000, 768), (9001, 130, 1024)])
def test_256x128_tiles_at_their_edges(dev, M, N, K):
    """Ragged shapes too large for the small tiles run the persistent
    kernel's 256x128 tiles unsplit: rows and columns ending inside a wave's
    64x64 part, an odd-length bf16 bias, rows that are not 16-byte aligned."""
    seed = synth.SEED_BASE + 700 + M + N + K
    A = synth.normal((M, K), 1.0, seed=seed)
    B = synth.normal((N, K), 0.02, seed=seed + 1)
    bb = synth.f32_to_bf16_bits(synth.normal((N,), 0.1, seed=seed + 2))
    aq, _, sa, Ad = quant_operand(A, Fmt.E4M3, dev)
    bq, _, sb, Bd = quant_operand(B, Fmt.E4M3, dev)
    bd = torch.from_numpy(bb.view(np.int16)).to(dev).view(torch.bfloat16)
    assert df.gemm_plan(M, N, K, aq.stride(0), bq.stride(0), bd, 1 << 30) == (df.GemmKernel.PERSISTENT_NARROW, 1)
    Y = df.gemm_nt(aq, Fmt.E4M3, bq, Fmt.E4M3, K, sa, sb, bias=bd)
    check_bf16_image(Y, df.gemm_nt(aq, Fmt.E4M3, bq, Fmt.E4M3, K, sa, sb, bias=bd, out_dtype=torch.bfloat16))
    rows = band_rows(M, seed)
    err = orc.rel_err(Y.cpu().numpy()[rows], orc.fc_forward(Ad[rows], Bd, orc.bf16_to_f32(bb)))
    assert err <= TOL, f"M={M} N={N} K={K}: rel err {err:.3e}"

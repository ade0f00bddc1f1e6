"""GPU parity: the wave-split-K kernel (csrc/gemm_ks.hip) behind the linear and
P5 entry points, at the edges of its row blocks (16 rows), its tiles, its K
units (64: fewer units than wavefronts, ragged last group) and its range.

Against the CPU oracle (double accumulation, one rounding): the kernel's fp32
sums differ from it in order only, so all but a few outputs agree to one bf16
ulp, and none is off by more than the GEMM bar.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch
from helpers import bf16_randn, bits, from_bits, max_rel_err, rel_err, ulp

import oracle
from umic.kernels import fused_ffn, linear

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 2e-2


def _check(out, ref_bits):
    d = ulp(bits(out), ref_bits)
    assert (d <= 1).mean() > 0.999, np.bincount(d.ravel())[:8]
    ref = from_bits(ref_bits)
    assert max_rel_err(out, ref) <= TOL and rel_err(out, ref) <= TOL


@pytest.mark.parametrize("M,N,K", [(3, 8, 64), (8, 1032, 576), (9, 264, 640), (16, 24, 4096),
                                   (17, 4104, 128), (33, 1000, 1024), (64, 4096, 192),
                                   (100, 520, 704), (257, 328, 1280), (515, 1032, 2112)])
@pytest.mark.parametrize("act,code,bias", [(None, 0, False), ("gelu_tanh", 2, True)])
def test_linear_vs_oracle(M, N, K, act, code, bias):
    print(f"split-K linear M={M} N={N} K={K} act={act}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    x, w = bf16_randn(M, K + 8, gen=g), bf16_randn(N, K, scale=0.05, gen=g)
    b = bf16_randn(N, scale=0.5, gen=g) if bias else None
    y = linear.linear_hip(x.to(DEV)[:, :K], w.to(DEV), None if b is None else b.to(DEV), act=act)
    torch.cuda.synchronize()
    _check(y, oracle.linear(bits(x[:, :K]), bits(w), None if b is None else bits(b), code,
                            fused=True))


@pytest.mark.parametrize("M,N,K", [(3, 8, 64), (16, 1000, 320), (33, 3072, 1024), (65, 104, 640),
                                   (130, 776, 192)])
def test_gate_silu_mul_vs_oracle(M, N, K):
    print(f"split-K P5 M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    x = bf16_randn(M, K, gen=g)
    wg, wu = bf16_randn(N, K, scale=0.05, gen=g), bf16_randn(N, K, scale=0.05, gen=g)
    y = fused_ffn.gate_silu_mul_hip(x.to(DEV), wg.to(DEV).t(), wu.to(DEV).t())
    torch.cuda.synchronize()
    _check(y, oracle.gate_silu_mul(bits(x), bits(wg), bits(wu), fused=True))


def test_streamed_weights_and_nan_rows():
    """Weights past the streaming size (non-temporal loads), and a NaN row and
    an infinite row that must stay in their own output rows."""
    g = torch.Generator(device=DEV).manual_seed(3)
    M, N, K = 40, 8200, 4096
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    w = (0.02 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    x[7, 100] = float("nan")
    x[39] = 0.0
    x[39, 5] = float("inf")
    y = linear.linear_hip(x, w)
    torch.cuda.synchronize()
    ref = x.float() @ w.float().t()
    keep = [i for i in range(M) if i not in (7, 39)]
    assert max_rel_err(y[keep], ref[keep]) <= TOL and rel_err(y[keep], ref[keep]) <= TOL
    assert y[7].isnan().all()
    assert torch.equal(y[39].float().nan_to_num(nan=3.0), ref[39].nan_to_num(nan=3.0))

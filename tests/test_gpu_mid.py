"""GPU parity: the tiled kernels below 256 x 256 (csrc/gemm_mid.hip) behind the
linear and P5 entry points, at ragged edges of their tiles (96 to 256 rows
by 128 columns), with an odd number of K stages (64 each; the one-tile schedule
gives odd ones to its second group of waves) and each epilogue.

Against the CPU oracle (double accumulation, one rounding) at small sizes and an
fp32 torch evaluation at the larger: the kernel's fp32 sums differ from either in
order only, so all but a few outputs agree to one bf16 ulp.
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


def _close(y, ref):
    d = ulp(bits(y), bits(ref.to(torch.bfloat16)))
    # the fp32 reference's own sums are in another order: a few more one-ulp ties
    assert (d <= 1).mean() > 0.999, np.bincount(d.ravel())[:8]
    assert max_rel_err(y, ref) <= TOL and rel_err(y, ref) <= TOL


# one tile per CU (128 and 96 rows), several per CU, 256-row tiles (GELU): rows
# and columns off the tile, an odd stage count
@pytest.mark.parametrize("M,N,K,act", [(1000, 4088, 1984, None), (700, 3848, 1344, None),
                                       (2047, 3848, 1216, None), (1500, 4104, 704, "gelu_tanh"),
                                       (16129, 2568, 320, "gelu"), (16384, 5120, 192, "gelu_tanh"),
                                       # the ring of stages of the one-tile kernels, 96 to 256
                                       # rows: fewer, as many and more stages than its slots
                                       (3137, 1000, 64, None), (2900, 1000, 128, None),
                                       (2900, 1000, 192, None), (1500, 4088, 256, None),
                                       (1409, 4088, 320, None), (2047, 4088, 64, None),
                                       (2045, 4096, 128, None), (1793, 4088, 192, None),
                                       (2048, 4096, 1088, None), (1000, 5112, 1280, "gelu")])
def test_linear_vs_fp32(M, N, K, act):
    print(f"mid linear M={M} N={N} K={K} act={act}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K + 64, generator=g, device=DEV).to(torch.bfloat16)[:, :K]
    w = (0.02 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16) if act else None
    y = linear.linear_hip(x, w, b, act=act)
    ref = x.float() @ w.float().t()
    if act:
        ref = torch.nn.functional.gelu(ref + b.float(),
                                       approximate="tanh" if act == "gelu_tanh" else "none")
    torch.cuda.synchronize()
    _close(y, ref)


@pytest.mark.parametrize("M,N,K", [(641, 12280, 320), (150, 6136, 1088),
                                   # one tile per CU: 128 and 256 rows by 64 gate columns
                                   (500, 3064, 1024), (257, 6136, 2112), (769, 3064, 1088),
                                   (350, 6136, 2048), (250, 12280, 2112)])
def test_gate_silu_mul_vs_fp32(M, N, K):
    print(f"mid P5 M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    wg = (0.02 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    wu = (0.02 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    y = fused_ffn.gate_silu_mul_hip(x, wg.t(), wu.t())
    gate = x.float() @ wg.float().t()
    ref = torch.nn.functional.silu(gate) * (x.float() @ wu.float().t())
    torch.cuda.synchronize()
    _close(y, ref)


def test_linear_vs_oracle():
    """128 x 128 tiles, several per CU, at a K the oracle can afford."""
    M, N, K = 4224, 1160, 64
    g = torch.Generator().manual_seed(5)
    x, w = bf16_randn(M, K, gen=g), bf16_randn(N, K, scale=0.1, gen=g)
    b = bf16_randn(N, scale=0.5, gen=g)
    y = linear.linear_hip(x.to(DEV), w.to(DEV), b.to(DEV), act="gelu_tanh")
    torch.cuda.synchronize()
    ref = oracle.linear(bits(x), bits(w), bits(b), 2, fused=True)
    d = ulp(bits(y), ref)
    assert (d <= 1).mean() > 0.999, np.bincount(d.ravel())[:8]
    assert max_rel_err(y, from_bits(ref)) <= TOL and rel_err(y, from_bits(ref)) <= TOL

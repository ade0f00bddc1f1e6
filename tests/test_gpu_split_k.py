"""GPU parity: the wave-split-K kernel (csrc/gemm_ks.hip) behind the linear and
P5 entry points: every tile of its tables, at ragged edges of the tile and of
its K units (64 each: fewer units than wavefronts, a ragged last group), and
the ends of its range.  Each case names the kernel it is for and asserts that
the dispatch runs it (``kernel_of``).

Against the CPU oracle (double accumulation, one rounding) at small sizes and
an fp32 torch evaluation at the larger: the kernel's fp32 sums differ from
either in order only, so all but a few outputs agree to one bf16 ulp, and none
is off by more than the GEMM bar.
"""

from __future__ import annotations

import pytest
import torch
from helpers import bf16_randn, bits, check_one_ulp, kernel_of, max_rel_err, rel_err

import oracle
from umic.kernels import fused_ffn, linear

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 2e-2

ORACLE = [(28016016, 3, 8, 64), (28016016, 8, 1032, 576), (28016016, 9, 264, 640),
          (28016016, 16, 24, 4096), (28032032, 17, 4104, 128), (28016016, 33, 1000, 1024),
          (28032032, 64, 4096, 192), (28016016, 100, 520, 704), (28016032, 257, 328, 1280),
          (28048064, 515, 1032, 2112)]
# 17 units of K: two or three to each of eight waves, four or five to each of four
TILES = [(28016016, 5, 8, 1088), (28016032, 5, 4104, 1088), (28032016, 4099, 8, 1088),
         (28032032, 17, 4104, 1088), (28032064, 9, 8200, 1088), (28048032, 8200, 8, 1088),
         (28048064, 33, 8200, 1088), (28064032, 4099, 72, 1088), (28064064, 49, 8200, 1088),
         (28064096, 9, 16392, 1088), (28080064, 65, 8200, 1088), (28096064, 81, 12440, 1088),
         (24048064, 130, 8200, 1088), (24064064, 97, 12440, 1088), (24080064, 130, 12280, 1088)]
P5_ORACLE = [(28016032, 3, 8, 64), (28016032, 16, 1000, 320), (28032064, 33, 3072, 1024),
             (28016032, 65, 104, 640), (28032032, 130, 776, 192)]
P5_TILES = [(28016032, 5, 8, 1088), (28016096, 5, 4104, 1088), (28032032, 4099, 8, 1088),
            (28032064, 9, 4104, 1088), (28032096, 33, 4104, 1088), (28048096, 8200, 8, 1088),
            (28064096, 49, 7176, 1088), (24032064, 9, 12440, 1088), (24064064, 33, 12440, 1088),
            (24048096, 9, 16392, 1088),
            # weights past the streaming size, one row tile: non-temporal loads
            (28032064, 29, 4104, 4096), (28064096, 61, 12280, 4096)]


@pytest.mark.parametrize("kernel,M,N,K", ORACLE)
@pytest.mark.parametrize("act,code,bias", [(None, 0, False), ("gelu_tanh", 2, True)])
def test_linear_vs_oracle(kernel, M, N, K, act, code, bias):
    print(f"split-K linear M={M} N={N} K={K} act={act}", flush=True)
    assert kernel_of(M, N, K, act) == kernel
    g = torch.Generator().manual_seed(M + N + K)
    x, w = bf16_randn(M, K + 8, gen=g), bf16_randn(N, K, scale=0.05, gen=g)
    b = bf16_randn(N, scale=0.5, gen=g) if bias else None
    y = linear.linear_hip(x.to(DEV)[:, :K], w.to(DEV), None if b is None else b.to(DEV), act=act)
    torch.cuda.synchronize()
    check_one_ulp(y, oracle.linear(bits(x[:, :K]), bits(w), None if b is None else bits(b), code,
                                   fused=True))


@pytest.mark.parametrize("kernel,M,N,K", TILES)
@pytest.mark.parametrize("act", [None, "gelu"])
def test_every_linear_tile_vs_fp32(kernel, M, N, K, act):
    print(f"split-K tile {kernel} M={M} N={N} K={K} act={act}", flush=True)
    assert kernel_of(M, N, K, act) == kernel
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K + 64, generator=g, device=DEV).to(torch.bfloat16)[:, :K]
    w = (0.05 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16) if act else None
    y = linear.linear_hip(x, w, b, act=act)
    ref = x.float() @ w.float().t()
    if act:
        ref = torch.nn.functional.gelu(ref + b.float())
    torch.cuda.synchronize()
    check_one_ulp(y, bits(ref.to(torch.bfloat16)))


@pytest.mark.parametrize("kernel,M,N,K", P5_ORACLE)
def test_gate_silu_mul_vs_oracle(kernel, M, N, K):
    print(f"split-K P5 M={M} N={N} K={K}", flush=True)
    assert kernel_of(M, N, K, p5=True) == kernel
    g = torch.Generator().manual_seed(M + N + K)
    x = bf16_randn(M, K, gen=g)
    wg, wu = bf16_randn(N, K, scale=0.05, gen=g), bf16_randn(N, K, scale=0.05, gen=g)
    y = fused_ffn.gate_silu_mul_hip(x.to(DEV), wg.to(DEV).t(), wu.to(DEV).t())
    torch.cuda.synchronize()
    check_one_ulp(y, oracle.gate_silu_mul(bits(x), bits(wg), bits(wu), fused=True))


@pytest.mark.parametrize("kernel,M,N,K", P5_TILES)
def test_every_p5_tile_vs_fp32(kernel, M, N, K):
    print(f"split-K P5 tile {kernel} M={M} N={N} K={K}", flush=True)
    assert kernel_of(M, N, K, p5=True) == kernel
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    wg, wu = ((0.05 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
              for _ in range(2))
    y = fused_ffn.gate_silu_mul_hip(x, wg.t(), wu.t())
    ref = torch.nn.functional.silu(x.float() @ wg.float().t()) * (x.float() @ wu.float().t())
    torch.cuda.synchronize()
    check_one_ulp(y, bits(ref.to(torch.bfloat16)))


def test_streamed_weights_and_nan_rows():
    """Weights past the streaming size (non-temporal loads), and a NaN row and
    an infinite row that must stay in their own output rows."""
    g = torch.Generator(device=DEV).manual_seed(3)
    M, N, K = 40, 8200, 4096
    assert kernel_of(M, N, K) == 28048064
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

"""GPU parity: the tiled kernels below 256 x 256 (csrc/gemm_mid.hip) behind the
linear and P5 entry points, at ragged edges of their tiles (96 to 256 rows
by 128 columns), with an odd number of K stages (64 each; the one-tile schedule
gives odd ones to its second group of waves) and each epilogue; and ragged shapes
that the 256 x 256 tiles of csrc/gemm.hip keep, one per epilogue and for few
stages.  Each case names the kernel it is for and asserts that the dispatch
runs it (``kernel_of``).

Against the CPU oracle (double accumulation, one rounding) at small sizes and an
fp32 torch evaluation at the larger: the kernel's fp32 sums differ from either in
order only, so all but a few outputs agree to one bf16 ulp.
"""

from __future__ import annotations

import pytest
import torch
from helpers import bf16_randn, bits, check_one_ulp, kernel_of

import oracle
from umic.kernels import fused_ffn, linear

pytestmark = pytest.mark.gpu
DEV = "cuda"

# one tile per CU (96 to 256 rows), several per CU, 256-row tiles: rows and
# columns off the tile, an odd stage count
LINEAR = [(38128128, 1000, 4088, 1984, None), (38096128, 700, 3848, 1344, None),
          (38256128, 2047, 3848, 1216, None), (34128128, 1500, 4104, 704, "gelu_tanh"),
          (34128128, 16129, 2568, 320, "gelu"), (34256128, 16384, 5120, 192, "gelu_tanh"),
          (34256128, 1200, 16392, 192, None), (34128128, 257, 16392, 1088, None),
          # the ring of stages of the one-tile kernels, four slots for up to 192 rows
          # and three for 256: fewer, as many and more stages than slots, where the
          # dispatch takes them for so few (never a single stage, and 256 rows
          # from four)
          (38096128, 2900, 1000, 128, None), (38096128, 2900, 1000, 192, None),
          (38096128, 81, 16392, 256, None), (38128128, 97, 16392, 128, None),
          (38128128, 97, 16392, 192, None), (38128128, 97, 16392, 256, None),
          (38192128, 32800, 120, 128, None), (38192128, 130, 16392, 192, None),
          (38192128, 1500, 4088, 256, None), (38192128, 1409, 4088, 320, None),
          (38256128, 200, 16392, 256, None), (38256128, 200, 16392, 320, None),
          (38256128, 2048, 4096, 1088, None), (38192128, 1000, 5112, 1280, "gelu")]
# the 256 x 256 tiles of four waves, and of eight where K % 64 != 0
LARGE = [(44256256, 3137, 1000, 64, None), (44256256, 2047, 4088, 64, None),
         (44256256, 2045, 4096, 128, None), (44256256, 1793, 4088, 192, None),
         (44256256, 400, 16392, 576, None), (44256256, 641, 16392, 576, "gelu"),
         (44256256, 641, 16392, 576, "gelu_tanh"), (48256256, 520, 4104, 96, "gelu"),
         (48256256, 300, 1000, 1056, "gelu_tanh")]
P5 = [(34128256, 641, 12280, 320), (34128256, 65, 16392, 1088), (38256128, 769, 3064, 1088),
      (38256128, 350, 6136, 2048), (38256128, 250, 12280, 2112), (38256128, 150, 10248, 1088),
      # 128 rows by 64 gate columns, three stages in a ring of four, and more
      (38128128, 16600, 64, 192), (38128128, 97, 8200, 256), (38128128, 97, 8200, 576),
      (38128128, 128, 12288, 4096),
      # the wave-split-K kernel's neighbours of these
      (24048096, 150, 6136, 1088), (24064064, 500, 3064, 1024), (24048096, 257, 6136, 2112)]
P5_LARGE = [(44256256, 97, 8200, 64), (44256256, 150, 10248, 576), (44256256, 130, 16392, 1088),
            (48256256, 300, 1000, 1056)]


@pytest.mark.parametrize("kernel,M,N,K,act", LINEAR + LARGE)
def test_linear_vs_fp32(kernel, M, N, K, act):
    print(f"linear {kernel} M={M} N={N} K={K} act={act}", flush=True)
    assert kernel_of(M, N, K, act) == kernel
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
    check_one_ulp(y, bits(ref.to(torch.bfloat16)))


@pytest.mark.parametrize("kernel,M,N,K", P5 + P5_LARGE)
def test_gate_silu_mul_vs_fp32(kernel, M, N, K):
    print(f"P5 {kernel} M={M} N={N} K={K}", flush=True)
    assert kernel_of(M, N, K, p5=True) == kernel
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    wg = (0.02 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    wu = (0.02 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    y = fused_ffn.gate_silu_mul_hip(x, wg.t(), wu.t())
    gate = x.float() @ wg.float().t()
    ref = torch.nn.functional.silu(gate) * (x.float() @ wu.float().t())
    torch.cuda.synchronize()
    check_one_ulp(y, bits(ref.to(torch.bfloat16)))


def test_linear_vs_oracle():
    """128 x 128 tiles, several per CU, at a K the oracle can afford."""
    M, N, K = 4224, 1160, 64
    assert kernel_of(M, N, K, "gelu_tanh") == 34128128
    g = torch.Generator().manual_seed(5)
    x, w = bf16_randn(M, K, gen=g), bf16_randn(N, K, scale=0.1, gen=g)
    b = bf16_randn(N, scale=0.5, gen=g)
    y = linear.linear_hip(x.to(DEV), w.to(DEV), b.to(DEV), act="gelu_tanh")
    torch.cuda.synchronize()
    check_one_ulp(y, oracle.linear(bits(x), bits(w), bits(b), 2, fused=True))


@pytest.mark.parametrize("M,N,K", [(300, 8200, 64), (81, 16392, 64)])
def test_four_wave_tiles_vs_oracle(M, N, K):
    """The 256 x 256 tiles of four waves, ragged in rows and columns."""
    print(f"four-wave tiles M={M} N={N} K={K}", flush=True)
    assert kernel_of(M, N, K) == 44256256
    g = torch.Generator().manual_seed(M)
    x, w = bf16_randn(M, K, gen=g), bf16_randn(N, K, scale=0.1, gen=g)
    b = bf16_randn(N, scale=0.5, gen=g)
    y = linear.linear_hip(x.to(DEV), w.to(DEV), b.to(DEV))
    torch.cuda.synchronize()
    check_one_ulp(y, oracle.linear(bits(x), bits(w), bits(b), 0, fused=True))


@pytest.mark.parametrize("M,N,K", [(97, 8200, 64), (300, 4104, 64)])
def test_four_wave_p5_tiles_vs_oracle(M, N, K):
    """The same for P5: a last tile column that is not whole (N % 128 != 0)."""
    print(f"four-wave P5 tiles M={M} N={N} K={K}", flush=True)
    assert kernel_of(M, N, K, p5=True) == 44256256
    g = torch.Generator().manual_seed(M)
    x = bf16_randn(M, K, gen=g)
    wg, wu = bf16_randn(N, K, scale=0.1, gen=g), bf16_randn(N, K, scale=0.1, gen=g)
    y = fused_ffn.gate_silu_mul_hip(x.to(DEV), wg.to(DEV).t(), wu.to(DEV).t())
    torch.cuda.synchronize()
    check_one_ulp(y, oracle.gate_silu_mul(bits(x), bits(wg), bits(wu), fused=True))

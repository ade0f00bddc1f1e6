// Tiled GEMM with tiles below 256 x 256: the row counts between the
// wave-split-K kernel (gemm_ks.hip) and the four-wave core of gemm.hip, whose
// 256 x 256 tiles need a few thousand rows to give every CU one (N = 4096: 64
// tiles at 1024 rows, 2048 rows half the chip), and the GELU linear at any
// larger size.
//
// Tile.  Four waves own 32 AX x rows by 32 AW weight rows, a quadrant of 16 AX
// by 16 AW each, in v_mfma_f32_16x16x32_bf16 blocks (for P5 half of the weight
// rows are gate rows and half the matching up rows).  K advances 64 at a time
// through LDS, by direct-to-LDS loads of whole 128-byte lines; rows are
// XOR-swizzled by (row >> 1) & 7, so fragment reads are conflict-free.
//
// Two schedules (MI355X, us, N = K = 4096 unless said otherwise; the 256 x 256
// tiles / this kernel):
// * One tile per CU (G = 2): eight waves in two groups of four, in alternation.
//   While one group multiplies a stage from registers the other reads the next one
//   from LDS, and a barrier swaps them; the loads go two or three stages ahead into
//   a ring of three or four that both groups share.  The groups hold the sums of
//   the even and the odd stages and add them at the end.  Before, both groups read
//   and then multiplied together, each with two stages of its own, which left the
//   matrix cores idle through the reads and no LDS for tiles above 128 rows
//   (N = K = 4096: 1500 rows 69 / 49, 2048 75 / 61; K = 12288, 800 rows 142 / 106,
//   2048 219 / 170; N = 1280, K = 5120, 4096 rows 89 / 63; P5 N = 2 x 6144, K =
//   2048, 350 rows 42.5 / 31).  A stage takes what LDS needs to be written once (64
//   bytes a cycle) and read twice (128): 128 rows 420 ns, 192 540, 256 700; at a
//   full chip 570, 690 and 870, 14 TB/s of operands out of L2.
// * More tiles than that (G = 1): four waves, ONE stage of LDS and two or three
//   workgroups to a CU.  A wave reads both K halves of a stage into registers,
//   a barrier frees the stage, the next one's loads go out and the MFMAs run
//   from registers: the other workgroups' MFMAs cover its loads and, at the end,
//   its epilogue.  A second stage costs a third workgroup and is slower (fc1 +
//   GELU, K = 1280, N = 5120, 4096 rows 63.2 against 56.7).  2048 rows 77.8 /
//   60.3; fc1 + GELU at 4096 rows 76.7 / 56.7, at 8192 and 16384 rows with 256 x
//   128 tiles 130 / 113 and 231 / 215 (on another box 241 / 225; a four-wave
//   tile's epilogue, some 8 us of VALU work at one wave per SIMD, runs with its
//   matrix cores idle; without the GELU it is 193 / 198); P5 at 600 rows 177 / 114.
// The K loop's waves raise their priority for the MFMAs, so that a wave with
// operands in registers goes before one that reads LDS (1-2%).
//
// Where the 256 x 256 tiles fill the chip they read LDS and L2 half as often per
// MFMA, and at the power limit that decides (3100 rows: 84 against 93 us).
#include "gelu.hpp"
#include "gemm_mid.hpp"

#include <algorithm>
#include <type_traits>

namespace umic {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) char lds_char;

constexpr int kMidBK = 64;           // K per stage
constexpr int kMidRow = kMidBK * 2;  // staged bytes per row

struct MidArgs {
  const char* x;
  const char* w0;
  const char* w1;
  const uint16_t* bias;  // or NULL
  uint16_t* out;
  int64_t ldo;
  int M, N, stages;     // stages = K / 64
  int ldx, ldw0, ldw1;  // in bytes
  int tiles_m, tiles, gm;
  int act;
};

template <int NB, int AX, int AW, int G>
struct Mid {
  static constexpr int kXRows = 32 * AX, kWRows = 32 * AW;
  static constexpr int kWBytes = kWRows * kMidRow;
  static constexpr int kStage = kXRows * kMidRow + kWBytes;
  // Stages of LDS: one of its own for a four-wave workgroup, a ring of three or
  // four that the two groups of an eight-wave one share.
  static constexpr int S = G == 1 ? 1 : 4 * kStage <= 160 * 1024 ? 4 : 3;
  static constexpr int LW = (AW + G - 1) / G, LX = (AX + G - 1) / G;  // loads of a wave per stage
  static constexpr int kCols = kWRows / NB;       // output columns per tile
  static constexpr int kOutRow = kCols * 2 + 16;  // staged bytes per output row
  static constexpr int kMail = G == 2 ? AX * AW * 4 * 1024 : 0;  // sums handed over
  static constexpr int kLds = std::max(std::max(S * kStage, kXRows * kOutRow), kMail);
  static_assert(AW % (G * NB) == 0 && kLds <= 160 * 1024, "tile");
  static_assert((S - 2) * (LW + LX) < 64, "vmcnt is 6 bits");

  static __device__ __forceinline__ void run(const MidArgs& g, char* smem) {
    // XCD-aware order, as the other tiled kernels: an XCD's tiles are a
    // contiguous run of groups of gm tile rows, rows fastest.
    const int per = (g.tiles + 7) >> 3;
    const int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (t >= g.tiles) return;
    const int tiles_n = g.tiles / g.tiles_m;
    const int tgroup = t / (g.gm * tiles_n), first_m = tgroup * g.gm;
    const int gm = min(g.tiles_m - first_m, g.gm);
    const int in_group = t - tgroup * g.gm * tiles_n;
    const int m0 = (first_m + in_group % gm) * kXRows, n0 = (in_group / gm) * kCols;

    const int lane = threadIdx.x & 63;
    const int w8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = G == 2 ? w8 >> 2 : 0, wave = w8 & 3, wm = wave & 1, wn = wave >> 1;
    const int fr = lane & 15, fc = lane >> 4, lr = lane >> 3, lc = lane & 7;
    lds_char* const ring = (lds_char*)smem;

    // This wave's loads of a stage, 8 rows each: the weight rows (P5: first the
    // gate, then the up rows) and the x rows are dealt out over all the waves,
    // load q of wave w being block q * waves + w.  Rows past M / N re-read the
    // last row; their results are not stored.  Where the x blocks do not divide
    // evenly the last one is loaded by several waves, the same bytes each time.
    constexpr int kWaves = 4 * G;
    int xo[LX], xd[LX], wo[LW];
#pragma unroll
    for (int q = 0; q < LX; ++q) {
      const int blk = min(q * kWaves + w8, 4 * AX - 1), r = blk * 8 + lr;
      xd[q] = kWBytes + blk * 1024;
      xo[q] = min(m0 + r, g.M - 1) * g.ldx + ((lc ^ ((r >> 1) & 7)) * 16);
    }
    auto up = [](int q) { return NB == 2 && q >= LW / 2; };
#pragma unroll
    for (int q = 0; q < LW; ++q) {
      const int r = (q * kWaves + w8) * 8 + lr;
      wo[q] = min(n0 + (up(q) ? r - kWRows / 2 : r), g.N - 1) * (up(q) ? g.ldw1 : g.ldw0) +
              ((lc ^ ((r >> 1) & 7)) * 16);
    }
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc((void*)g.x, 0, g.M * g.ldx, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw0 =
        __builtin_amdgcn_make_buffer_rsrc((void*)g.w0, 0, g.N * g.ldw0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw1 =
        NB == 2 ? __builtin_amdgcn_make_buffer_rsrc((void*)g.w1, 0, g.N * g.ldw1, 0x00020000) : rw0;
    auto load = [&](int slot, int stage) {
      const int k = stage * kMidRow;
      lds_char* const d = ring + slot * kStage;
#pragma unroll
      for (int q = 0; q < LW; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(up(q) ? rw1 : rw0,
                                                 (lds_void*)(d + (q * kWaves + w8) * 1024), 16,
                                                 wo[q], k, 0, 0);
#pragma unroll
      for (int q = 0; q < LX; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)(d + xd[q]), 16, xo[q], k, 0, 0);
    };
    auto arow = [&](int a) {
      return NB == 1 ? wn * 16 * AW + a * 16
                     : (a < AW / 2 ? wn * 8 * AW + a * 16 : 16 * AW + wn * 8 * AW + (a - AW / 2) * 16);
    };
    bf16x8_t wf[2][AW], xf[2][AX];
    auto read = [&](int slot, int h) {
      typedef const __attribute__((address_space(3))) bf16x8_t* frag_p;
      const lds_char* const s =
          ring + slot * kStage + fr * kMidRow + (((h * 4 + fc) ^ ((fr >> 1) & 7)) * 16);
#pragma unroll
      for (int a = 0; a < AW; ++a) wf[h][a] = *(frag_p)(s + arow(a) * kMidRow);
#pragma unroll
      for (int b = 0; b < AX; ++b)
        xf[h][b] = *(frag_p)(s + kWBytes + (wm * 16 * AX + b * 16) * kMidRow);
    };
    f32x4_t acc[AW][AX];
#pragma unroll
    for (int a = 0; a < AW; ++a)
#pragma unroll
      for (int b = 0; b < AX; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto mul = [&] {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int a = 0; a < AW; ++a)
#pragma unroll
          for (int b = 0; b < AX; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][a], xf[h][b], acc[a][b], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
    };
    // s_waitcnt vmcnt(V) (all but V of this wave's loads have landed) or
    // lgkmcnt(0) (its LDS reads are done), then s_barrier; no memory access moves
    // across.
    auto landed = [](auto left) {
      constexpr int V = decltype(left)::value;
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt((V & 15) | (7 << 4) | (15 << 8) | ((V >> 4) << 14));
      asm volatile("" ::: "memory");
    };
    auto reads_done = [] {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
      asm volatile("" ::: "memory");
    };
    auto barrier = [] {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    constexpr std::integral_constant<int, 0> kAll{};
    if constexpr (G == 2) {
      // Phase p: the group of p's parity reads stage p into registers, the other
      // multiplies stage p - 1, and every wave loads its part of stage p + S - 1
      // into the slot that stage p - 1 was read from before the last barrier.  At
      // the end of the phase all but the loads of the last S - 2 phases have
      // landed, so stage p + 1 is in LDS; once nothing is left to load, all have.
      constexpr std::integral_constant<int, (S - 2) * (LW + LX)> kAhead{};
#pragma unroll
      for (int s = 0; s < S - 1; ++s)
        if (s < g.stages) load(s, s);
      if (S - 1 <= g.stages)
        landed(kAhead);
      else
        landed(kAll);
      barrier();
      int slot = 0;  // of stage p
      auto refill = [&](int p) {
        if (p + S - 1 < g.stages) load(slot == 0 ? S - 1 : slot - 1, p + S - 1);
      };
      auto end_phase = [&](int p) {
        if (p + S - 1 < g.stages)
          landed(kAhead);
        else
          landed(kAll);
        barrier();
        slot = slot == S - 1 ? 0 : slot + 1;
      };
      if (grp == 1) {  // phase 0 has nothing to multiply yet
        refill(0);
        end_phase(0);
      }
      int p = grp;
      for (; p < g.stages; p += 2) {
        read(slot, 0);
        read(slot, 1);
        refill(p);
        reads_done();
        end_phase(p);
        refill(p + 1);
        mul();
        end_phase(p + 1);
      }
      if (p == g.stages) barrier();  // the other group's last product
    } else {
      load(0, 0);
      for (int i = 0; i < g.stages; ++i) {
        landed(kAll);
        barrier();
        read(0, 0);
        read(0, 1);
        reads_done();
        barrier();
        if (i + 1 < g.stages) load(0, i + 1);
        mul();
      }
    }
    __syncthreads();  // the LDS is free
    if constexpr (G == 2) {
      // Group 0 finishes x blocks b < H, group 1 the others; each hands the
      // other its sums of them.
      constexpr int H = (AX + 1) / 2;
      f32x4_t* const mail = reinterpret_cast<f32x4_t*>(smem) + wave * AW * AX * 64 + lane;
#pragma unroll
      for (int a = 0; a < AW; ++a)
#pragma unroll
        for (int b = 0; b < AX; ++b)
          if ((b < H) == (grp == 1)) mail[(a * AX + b) * 64] = acc[a][b];
      __syncthreads();
#pragma unroll
      for (int a = 0; a < AW; ++a)
#pragma unroll
        for (int b = 0; b < AX; ++b)
          if ((b < H) == (grp == 0)) acc[a][b] += mail[(a * AX + b) * 64];
      __syncthreads();
      if (grp == 0)
        epilogue<0, H>(g, smem, acc, n0, wm, wn, fr, fc);
      else
        epilogue<H, AX>(g, smem, acc, n0, wm, wn, fr, fc);
    } else {
      epilogue<0, AX>(g, smem, acc, n0, wm, wn, fr, fc);
    }
    __syncthreads();
    // Whole rows out of the staged tile, 16 bytes a lane.
    constexpr int kChunks = kCols / 8;
    for (int c = threadIdx.x; c < kXRows * kChunks; c += 256 * G) {
      const int r = c / kChunks, q = c % kChunks;
      const int row = m0 + r, col = n0 + q * 8;
      if (row < g.M && col < g.N)
        *reinterpret_cast<u32x4*>(g.out + (int64_t)row * g.ldo + col) =
            *reinterpret_cast<const u32x4*>(smem + r * kOutRow + q * 16);
    }
  }

  // x blocks [B0, B1) of this wave into the staged tile: bias, activation or
  // silu(g) * u in fp32, one bf16 rounding, as the other kernels.
  template <int B0, int B1>
  static __device__ __forceinline__ void epilogue(const MidArgs& g, char* smem,
                                                  const f32x4_t (&acc)[AW][AX], int n0, int wm,
                                                  int wn, int fr, int fc) {
    if (NB == 1 && g.act == UMIC_ACT_GELU)
      stage_out<B0, B1, UMIC_ACT_GELU>(g, smem, acc, n0, wm, wn, fr, fc);
    else if (NB == 1 && g.act == UMIC_ACT_GELU_TANH)
      stage_out<B0, B1, UMIC_ACT_GELU_TANH>(g, smem, acc, n0, wm, wn, fr, fc);
    else
      stage_out<B0, B1, UMIC_ACT_NONE>(g, smem, acc, n0, wm, wn, fr, fc);
  }

  template <int B0, int B1, int ACT>
  static __device__ __forceinline__ void stage_out(const MidArgs& g, char* smem,
                                                   const f32x4_t (&acc)[AW][AX], int n0, int wm,
                                                   int wn, int fr, int fc) {
    constexpr int kOut = AW / NB;
#pragma unroll
    for (int a = 0; a < kOut; ++a) {
      const int col = wn * 16 * kOut + a * 16 + fc * 4;
      float bias[4] = {0.f, 0.f, 0.f, 0.f};
      if (NB == 1 && g.bias && n0 + col < g.N)
        unpack4(*reinterpret_cast<const u32x2*>(g.bias + n0 + col), bias);
#pragma unroll
      for (int b = B0; b < B1; ++b) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float y = acc[a][b][e];
          if constexpr (NB == 2) {
            const float den = 1.0f + __builtin_amdgcn_exp2f(y * -1.4426950408889634f);
            y = y * __builtin_amdgcn_rcpf(den) * acc[a + kOut * (NB - 1)][b][e];
          } else {
            y = y + bias[e];
            if constexpr (ACT == UMIC_ACT_GELU) y = gelu_erf(y);
            if constexpr (ACT == UMIC_ACT_GELU_TANH) y = gelu_tanh(y);
          }
          o[e] = y;
        }
        *reinterpret_cast<u32x2*>(smem + (wm * 16 * AX + b * 16 + fr) * kOutRow + col * 2) = pack4(o);
      }
    }
  }
};

template <int NB, int AX, int AW, int G>
__global__ __launch_bounds__(256 * G, 2) void gemm_mid_kernel(MidArgs g) {
  using K = Mid<NB, AX, AW, G>;
  __shared__ __attribute__((aligned(16))) char smem[K::kLds];
  K::run(g, smem);
}

// The kernels, with the time a stage of a tile takes of a CU (MI355X, fitted to
// the sizes above and their neighbours, weights from HBM): stage_ns, plus fill_ns
// times the share of the CUs that have a tile, for at full chip the one-tile
// kernels' 14 TB/s of operands are what L2 gives.  alone: how many tiles a CU with
// one alone is as slow as: the G = 1 kernels need a second workgroup to hide their
// loads.  fixed_ns and gelu_ns: prologue, epilogue and launch, per tile of a CU.
// One-tile kernels qualify only where no CU gets two: beyond that the G = 1
// kernels' overlapped epilogues and shorter last round win (P5 at 1600 rows, 4.9
// tiles a CU, 275 against 288 us).
struct MidKernel {
  int p5, ax, aw, groups;
  double stage_ns, fill_ns, alone, fixed_ns, gelu_ns;
  void (*kern)(MidArgs);
};
const MidKernel kMid[] = {
    {0, 3, 4, 2, 185.0, 265.0, 1.0, 5000.0, 2000.0, gemm_mid_kernel<1, 3, 4, 2>},
    {0, 4, 4, 2, 300.0, 265.0, 1.0, 5000.0, 2500.0, gemm_mid_kernel<1, 4, 4, 2>},
    {0, 6, 4, 2, 440.0, 265.0, 1.0, 5000.0, 3500.0, gemm_mid_kernel<1, 6, 4, 2>},
    {0, 8, 4, 2, 600.0, 265.0, 1.0, 5000.0, 4500.0, gemm_mid_kernel<1, 8, 4, 2>},
    {0, 4, 4, 1, 500.0, 0.0, 1.6, 5000.0, 0.0, gemm_mid_kernel<1, 4, 4, 1>},
    {0, 8, 4, 1, 1000.0, 0.0, 1.05, 5000.0, 0.0, gemm_mid_kernel<1, 8, 4, 1>},
    {1, 4, 4, 2, 300.0, 265.0, 1.0, 5500.0, 0.0, gemm_mid_kernel<2, 4, 4, 2>},
    {1, 8, 4, 2, 500.0, 265.0, 1.0, 8000.0, 0.0, gemm_mid_kernel<2, 8, 4, 2>},
    {1, 4, 8, 1, 870.0, 0.0, 1.2, 5000.0, 0.0, gemm_mid_kernel<2, 4, 8, 1>},
};
// Weights too large to still be in a cache cost more: the G = 1 linears, where the
// wait for a stage is covered by the other workgroups alone, and the one-tile P5,
// whose 100 MB and more are all read in one round (N = 2 x 12288, K = 4096: 64 rows
// 49 us, 250 rows 65).
constexpr int64_t kMidColdBytes = (int64_t)64 << 20;
constexpr double kMidCold1 = 1.15, kMidCold2 = 1.3, kMidMany = 1.05;

int64_t mid_tiles(const MidKernel& k, int64_t M, int64_t N, int64_t* tiles_m) {
  const int64_t cols = k.aw * 32 / (k.p5 ? 2 : 1);
  *tiles_m = (M + k.ax * 32 - 1) / (k.ax * 32);
  return *tiles_m * ((N + cols - 1) / cols);
}

const MidKernel* mid_choose(bool p5, int64_t M, int64_t N, int64_t K, int act, int64_t cus,
                            double* ns) {
  const MidKernel* best = nullptr;
  const bool cold = N * K * (p5 ? 4 : 2) >= kMidColdBytes;
  for (const MidKernel& k : kMid) {
    if (k.p5 != (int)p5) continue;
    int64_t tiles_m;
    const int64_t tiles = mid_tiles(k, M, N, &tiles_m);
    if (tiles > (int64_t)1 << 28 || (k.groups == 2 && tiles > cus)) continue;
    const double cold_by = !cold || p5 != (k.groups == 2) ? 1.0 : p5 ? kMidCold2 : kMidCold1;
    // past four tiles to a CU the 128-row ones' re-reads of x and w show
    const int64_t per_cu = (tiles + cus - 1) / cus;
    const double c = per_cu <= 1 ? k.alone : per_cu > 4 && k.ax == 4 ? kMidMany * per_cu : per_cu;
    const double stage = k.stage_ns + k.fill_ns * std::min(1.0, (double)tiles / (double)cus);
    const double t = k.fixed_ns + (act == UMIC_ACT_NONE ? 0.0 : k.gelu_ns) +
                     c * (double)(K / kMidBK) * stage * cold_by;
    if (!best || t < *ns) {
      best = &k;
      *ns = t;
    }
  }
  return best;
}

}  // namespace

double mid_time_ns(bool p5, int64_t M, int64_t N, int64_t K, int act, int64_t cus,
                   TileShape* tile) {
  double ns = 0.0;
  if (M <= 0 || N <= 0 || K <= 0 || K % kMidBK || cus <= 0) return -1.0;
  const MidKernel* const k = mid_choose(p5, M, N, K, act, cus, &ns);
  if (!k) return -1.0;
  if (tile) *tile = TileShape{k->ax * 32, k->aw * 32, k->groups * 4};
  return ns;
}

int launch_mid(bool p5, const KsCall& c, hipStream_t st) {
  double ns = 0.0;
  const int64_t cus = device_cus();
  const MidKernel* const k = cus > 0 ? mid_choose(p5, c.M, c.seg[0].N, c.K, c.act, cus, &ns) : nullptr;
  if (!k) return UMIC_ERR_UNSUPPORTED;
  const KsSeg& s = c.seg[0];
  MidArgs g{};
  g.x = reinterpret_cast<const char*>(c.x);
  g.w0 = reinterpret_cast<const char*>(s.w0);
  g.w1 = reinterpret_cast<const char*>(s.w1);
  g.bias = s.bias;
  g.out = s.out;
  g.ldo = s.ldo;
  g.M = (int)c.M;
  g.N = (int)s.N;
  g.stages = (int)(c.K / kMidBK);
  g.ldx = (int)(c.ldx * 2);
  g.ldw0 = (int)(s.ldw0 * 2);
  g.ldw1 = (int)(s.ldw1 * 2);
  g.act = c.act;
  int64_t tiles_m;
  g.tiles = (int)mid_tiles(*k, c.M, s.N, &tiles_m);
  g.tiles_m = (int)tiles_m;
  // One-tile launches take up to six tile rows at a time, so that an XCD's 32
  // tiles are about square and read the fewest bytes into its L2 (N = 1280, K =
  // 5120, 4096 rows, 192-row tiles 63 us against 68 with all 22 rows; N = 4096, K =
  // 12288, 2048 rows 173 against 176 with all eight; one row at a time costs 10%).
  // G = 1: launches of about one round keep a column's row tiles together, longer
  // ones take four rows, so that x slabs live through a round too (fc1 at 16384
  // rows 214 against 227 us with 16).
  g.gm = k->groups == 2 ? std::min(g.tiles_m, 6) : g.tiles <= 2 * cus ? g.tiles_m : 4;
  hipLaunchKernelGGL(k->kern, dim3((unsigned)((g.tiles + 7) / 8 * 8)),
                     dim3((unsigned)(256 * k->groups)), 0, st, g);
  return launch_status();
}

}  // namespace umic

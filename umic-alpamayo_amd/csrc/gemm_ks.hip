// Wave-split-K GEMM: linears and P5 over a few up to some hundred rows.
//
//   out = act(x @ w^T + bias)          out = silu(x @ wg^T) * (x @ wu^T)
//
// Between the decode GEMV (1-2 rows) and the 256 x 256 tiles of gemm.hip the
// product is bound by moving the operands into the CUs: at 64 rows, K = 4096
// the weights alone take 5.6 us from memory, the MFMAs 1.5.  A 256-row tile
// leaves most CUs idle there (16 workgroups for N = 4096) and runs K in one
// serial chain.  Here
//
// * a workgroup owns a small tile, 16 FM x rows by 16 FN weight rows, sized
//   so that about one per CU covers the output;
// * its W waves split K, not the tile: wave w takes the 64-deep K units
//   w, w + W, ... and computes the WHOLE tile on them.  Every operand byte
//   then enters the CU once and is read from LDS once (a wave's fragments
//   are used FM or FN times from registers), and no wave waits for another
//   inside the K loop: each has its own ring of P units in LDS, filled by its
//   own direct-to-LDS loads and drained by its own waits.  One barrier at the
//   end, then the W fp32 partial tiles are summed through LDS in wave order
//   (deterministic) and the epilogue runs on the sums.
//
// Staging through LDS is for the loads: a fragment's lanes lie on 16 rows, so
// a load straight into fragment layout touches another row with every lane
// and runs at a quarter of the rate (measured about 62 cycles per 1 KB
// instruction against 16: M = 256, N = K = 4096 took 31.5 us, staged 15.2).
// A direct-to-LDS load moves 8 rows of 128 bytes, whole cache lines; chunks
// are XOR-swizzled by (row >> 1) & 7 so the fragment reads are conflict-free,
// as in gemm.hip.
//
// What bounds it (MI355X): a CU takes in about 95 bytes/ns of operands from L2
// or the Infinity Cache, x rows included and whatever the depth P or W, and
// waits longer for weights that come from HBM.  So the tile is chosen for the
// fewest bytes per CU, (FM + FN) * 16 * K * 2 times the tiles a CU gets: see
// ks_choose.
#include "gelu.hpp"
#include "gemm_ks.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace umic {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) char lds_char;

constexpr int kKsUnit = 64;          // K per unit
constexpr int kKsRow = kKsUnit * 2;  // staged bytes per row
constexpr int kKsFrag = 16 * kKsRow; // staged bytes of a 16-row fragment block

struct KsSegArgs {
  const char* w0;
  const char* w1;
  const uint16_t* bias;
  uint16_t* out;
  int64_t ldo;
  int N, ldw0, ldw1;  // leading dims in bytes
};
struct KsArgs {
  const char* x;
  const uint16_t* resid;
  int64_t ldr;
  KsSegArgs seg[kKsMaxSegs];
  int first[kKsMaxSegs + 1];  // first column tile of each segment
  int count;
  int M, ldx, units;          // ldx in bytes; units = K / 64
  int tiles_m, tiles;
  int act;
};

// Loads of the weights with the non-temporal hint (NT) keep x in L2; chosen
// by the launcher.
template <int NB, int FM, int FN, int W, int P, bool NT>
struct Ks {
  static constexpr int F = FM + FN;
  static constexpr int kSlot = F * kKsFrag;              // LDS of a unit
  static constexpr int kLoads = F * 2;                   // load instructions of a unit
  static constexpr int kRing = W * P * kSlot;
  static constexpr int kTile = FM * FN * 1024;           // one wave's partial tile
  static constexpr int R = W * kTile <= 160 * 1024 ? W : W / 2;  // partials in LDS at a time
  static constexpr int kLds = std::max(kRing, R * kTile);
  // Larger tiles hold one K half's fragments at a time: both halves' and the
  // accumulators would not fit the registers of two waves per SIMD.
  static constexpr int HB = F >= 10 ? 1 : 2;
  static_assert(kLds <= 160 * 1024, "LDS");
  static_assert((P - 1) * kLoads < 64, "vmcnt is 6 bits");
  static_assert(FN % NB == 0, "P5: as many up as gate blocks");

  template <int VM>
  static __device__ __forceinline__ void wait_loads() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | (15 << 8) | ((VM >> 4) << 14));
    asm volatile("" ::: "memory");
  }
  static __device__ __forceinline__ void wait_reads() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
    asm volatile("" ::: "memory");
  }

  static __device__ __forceinline__ void run(const KsArgs& g, char* smem) {
    // XCD-aware order: an XCD works through a contiguous run of tiles, the
    // row tiles of one column tile together, so its L2 reads the weights once.
    const int per = (g.tiles + 7) >> 3;
    const int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (t >= g.tiles) return;
    const int tn = t / g.tiles_m, tm = t - tn * g.tiles_m;
    int si = 0;
#pragma unroll
    for (int i = 1; i < kKsMaxSegs; ++i)
      if (NB == 1 && i < g.count && tn >= g.first[i]) si = i;
    const KsSegArgs& sg = g.seg[si];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = tm * FM * 16, n0 = (tn - g.first[si]) * (FN / NB) * 16;

    // Load i of a fragment block: rows 8i .. 8i + 7, lane l the 16-byte chunk
    // that the swizzle puts at slot l % 8 of row l / 8.  Rows past M / N
    // re-read the last row (their results are not stored).
    const int lr = lane >> 3, lc = lane & 7;
    int xo[FM][2], wo[FN][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = i * 8 + lr, c = (lc ^ ((r >> 1) & 7)) * 16;
#pragma unroll
      for (int b = 0; b < FM; ++b) xo[b][i] = min(m0 + b * 16 + r, g.M - 1) * g.ldx + c;
#pragma unroll
      for (int a = 0; a < FN; ++a) {
        const bool up = NB == 2 && a >= FN / 2;
        wo[a][i] = min(n0 + (up ? a - FN / 2 : a) * 16 + r, sg.N - 1) * (up ? sg.ldw1 : sg.ldw0) + c;
      }
    }
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc((void*)g.x, 0, g.M * g.ldx, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw0 =
        __builtin_amdgcn_make_buffer_rsrc((void*)sg.w0, 0, sg.N * sg.ldw0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw1 =
        NB == 2 ? __builtin_amdgcn_make_buffer_rsrc((void*)sg.w1, 0, sg.N * sg.ldw1, 0x00020000) : rw0;
    lds_char* const ring = (lds_char*)smem + wave * P * kSlot;
    auto load = [&](int p, int u) {
      const int k = u * kKsRow;
      lds_char* const d = ring + p * kSlot;
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(NB == 2 && a >= FN / 2 ? rw1 : rw0,
                                                   (lds_void*)(d + a * kKsFrag + i * 1024), 16,
                                                   wo[a][i], k, 0, NT ? 2 : 0);
#pragma unroll
      for (int b = 0; b < FM; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)(d + (FN + b) * kKsFrag + i * 1024),
                                                   16, xo[b][i], k, 0, 0);
    };

    const int fr = lane & 15, fc = lane >> 4;
    bf16x8_t wf[HB][FN], xf[HB][FM];
    auto read = [&](int p, int h) {
      const lds_char* const s =
          ring + p * kSlot + fr * kKsRow + (((h * 4 + fc) ^ ((fr >> 1) & 7)) * 16);
      typedef const __attribute__((address_space(3))) bf16x8_t* frag_p;
#pragma unroll
      for (int a = 0; a < FN; ++a) wf[h % HB][a] = *(frag_p)(s + a * kKsFrag);
#pragma unroll
      for (int b = 0; b < FM; ++b) xf[h % HB][b] = *(frag_p)(s + (FN + b) * kKsFrag);
    };
    f32x4_t acc[FN][FM];
#pragma unroll
    for (int a = 0; a < FN; ++a)
#pragma unroll
      for (int b = 0; b < FM; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto mul = [&](int h) {
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h % HB][a], xf[h % HB][b],
                                                              acc[a][b], 0, 0, 0);
    };
    // One unit whose loads have landed; refill() runs once its LDS reads are
    // done, so the loads it issues are in flight under the MFMAs.
    auto unit = [&](int p, auto refill) {
      if constexpr (HB == 1) {
        read(p, 0);
        wait_reads();
        __builtin_amdgcn_sched_barrier(0);
        mul(0);
        __builtin_amdgcn_sched_barrier(0);
        read(p, 1);
        wait_reads();
        __builtin_amdgcn_sched_barrier(0);
        refill();
        __builtin_amdgcn_sched_barrier(0);
        mul(1);
      } else {
        read(p, 0);
        read(p, 1);
        wait_reads();
        __builtin_amdgcn_sched_barrier(0);
        refill();
        __builtin_amdgcn_sched_barrier(0);
        mul(0);
        mul(1);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // This wave's n units: wave, wave + W, ...; the last P take no refill and
    // wait for everything.
    const int n = (g.units - wave + W - 1) / W;  // <= 0: no unit
#pragma unroll
    for (int p = 0; p < P; ++p)
      if (p < n) load(p, wave + p * W);
    int i = 0;
    for (; i + P < n; ++i) {
      wait_loads<(P - 1) * kLoads>();
      unit(i % P, [&] { load(i % P, wave + (i + P) * W); });
    }
    wait_loads<0>();
    for (; i < n; ++i) unit(i % P, [] {});

    // Partial tiles through LDS (the rings are idle once every wave is here).
    __syncthreads();
    f32x4_t(*const part)[FN][FM][64] = reinterpret_cast<f32x4_t(*)[FN][FM][64]>(smem);
    auto put = [&](int r, bool add) {
#pragma unroll
      for (int a = 0; a < FN; ++a)
#pragma unroll
        for (int b = 0; b < FM; ++b)
          part[r][a][b][lane] = add ? acc[a][b] + part[r][a][b][lane] : acc[a][b];
    };
    if constexpr (R < W) {
      if (wave >= R) put(wave - R, false);
      __syncthreads();
      if (wave < R) put(wave, true);
    } else {
      put(wave, false);
    }
    __syncthreads();
    // Block (a, b): x row m0 + 16 b + lane % 16, columns n0 + 16 a + 4 (lane
    // / 16) .. + 4 of the sums, 8 bytes of output per lane.
    constexpr int kOut = FN / NB;
    for (int s = wave; s < kOut * FM; s += W) {
      const int a = s % kOut, b = s / kOut;
      const int row = m0 + b * 16 + fr, col = n0 + a * 16 + fc * 4;
      f32x4_t v = part[0][a][b][lane], u = part[0][NB == 2 ? a + kOut : a][b][lane];
#pragma unroll
      for (int r = 1; r < R; ++r) {
        v += part[r][a][b][lane];
        if constexpr (NB == 2) u += part[r][a + kOut][b][lane];
      }
      if (row >= g.M || col >= sg.N) continue;  // N % 8 == 0: four columns together
      float o[4], bias[4] = {0.f, 0.f, 0.f, 0.f}, res[4];
      if (NB == 1 && sg.bias) unpack4(*reinterpret_cast<const u32x2*>(sg.bias + col), bias);
      if (NB == 1 && g.resid)  // rows of 2-byte alignment at least: N % 8 says nothing of ldr
#pragma unroll
        for (int e = 0; e < 4; ++e) res[e] = bf2f(g.resid[(int64_t)row * g.ldr + col + e]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float y = v[e];
        if constexpr (NB == 2) {
          // silu(g) * u as the tiled kernels form it
          const float den = 1.0f + __builtin_amdgcn_exp2f(y * -1.4426950408889634f);
          y = y * __builtin_amdgcn_rcpf(den) * u[e];
        } else {
          y = y + bias[e];
          if (g.act == UMIC_ACT_GELU) y = gelu_erf(y);
          if (g.act == UMIC_ACT_GELU_TANH) y = gelu_tanh(y);
          if (g.resid) y = rbf(y) + res[e];
        }
        o[e] = y;
      }
      *reinterpret_cast<u32x2*>(sg.out + (int64_t)row * sg.ldo + col) = pack4(o);
    }
  }
};

// Two waves per SIMD: 8 waves of one workgroup, or two workgroups of 4 where
// their LDS fits.
template <int NB, int FM, int FN, int W, int P, bool NT>
__global__ __launch_bounds__(W * 64, 2) void gemm_ks_kernel(KsArgs g) {
  using K = Ks<NB, FM, FN, W, P, NT>;
  __shared__ __attribute__((aligned(16))) char smem[K::kLds];
  K::run(g, smem);
}

struct KsKernel {
  int fm, fn, waves;  // fn: weight blocks (P5: gate and up together)
  void (*kern)(KsArgs);
  void (*kern_nt)(KsArgs);
};
#define KS(NB, FM, FN, W, P) \
  {FM, FN, W, gemm_ks_kernel<NB, FM, FN, W, P, false>, gemm_ks_kernel<NB, FM, FN, W, P, true>}
// Eight waves with the LDS of a whole CU for the tiles of which a CU gets one,
// four waves, two workgroups to a CU, for those of which it gets more: at M =
// 400, N = K = 4096 (448 tiles of 64 x 64) 25.6 against 28.5 us, at M = 256,
// K = 12288 (256 tiles) 58.0 against 53.9.  (Ten blocks take the registers of
// eight waves either way.)  Small tiles have room for a second unit in flight.
const KsKernel kKsLinear[] = {
    KS(1, 1, 1, 8, 2), KS(1, 1, 2, 8, 2), KS(1, 2, 1, 8, 2), KS(1, 2, 2, 8, 2), KS(1, 3, 2, 8, 1),
    KS(1, 2, 4, 8, 1), KS(1, 4, 2, 8, 1), KS(1, 3, 4, 8, 1), KS(1, 4, 4, 8, 1), KS(1, 5, 4, 8, 1),
    KS(1, 4, 6, 8, 1), KS(1, 6, 4, 8, 1), KS(1, 3, 4, 4, 1), KS(1, 4, 4, 4, 1), KS(1, 5, 4, 4, 1)};
const KsKernel kKsP5[] = {
    KS(2, 1, 2, 8, 2), KS(2, 1, 6, 8, 1), KS(2, 2, 2, 8, 1), KS(2, 2, 4, 8, 1), KS(2, 2, 6, 8, 1),
    KS(2, 3, 6, 8, 1), KS(2, 4, 6, 8, 1), KS(2, 2, 4, 4, 1), KS(2, 4, 4, 4, 1), KS(2, 3, 6, 4, 1)};
#undef KS

// Weights of a launch that reads them once (one row tile) and that are larger
// than this are loaded non-temporally: they come from HBM whatever was read
// before, and x keeps its place in L2 (P5, N = 2 x 12288, K = 4096 at 64 rows
// 38.1 against 42.5 us, at 32 rows 31.3 against 34.9).  Smaller ones may still
// be in the Infinity Cache from their last use, and the hint costs there (o_proj,
// 33.6 MB read every third call, 32 rows: 8.6 against 8.1 us).
constexpr int64_t kKsStreamBytes = (int64_t)64 << 20;

// The kernel whose busiest CU takes in the fewest operand bytes, c tiles of
// 16 (FM + FN) rows by K each, at the measured rate, plus a fixed cost per tile
// (the reduction and the epilogue) and, for weights that must come from HBM,
// the CU's share of them at the rate they cost beyond that, in nanoseconds.  Up to eight rows
// only eight-wave kernels of one row block qualify, so that every entry point
// (one linear, several, one with a residual) sums K in the same order there.
constexpr double kKsBytesPerNs = 95.0, kKsColdBytesPerNs = 33.0;
constexpr double kKsFixedNs = 2500.0, kKsTileNs = 900.0;
constexpr int kKsFewRows = 8;

const KsKernel* ks_choose(bool p5, int64_t M, int64_t N, int64_t K, int64_t cus, double* ns) {
  const int64_t wbytes = N * K * 2 * (p5 ? 2 : 1);
  const double cold_ns =
      wbytes >= kKsStreamBytes ? (double)wbytes / (double)cus / kKsColdBytesPerNs : 0.0;
  // x past an XCD's 4 MB of L2 is read again for every column tile (N = 1024, K =
  // 4096: 1024 rows, 8 MB, 18.1 us against 14.4 without this term, 2048 rows 40.1
  // against 26.4)
  const double spill = 1.0 + std::min(0.5, std::max(0.0, 0.04 * ((double)(M * K * 2) / 1e6 - 4.2)));
  const KsKernel* best = nullptr;
  const KsKernel* const list = p5 ? kKsP5 : kKsLinear;
  const int count = p5 ? (int)(sizeof(kKsP5) / sizeof(kKsP5[0]))
                       : (int)(sizeof(kKsLinear) / sizeof(kKsLinear[0]));
  for (int i = 0; i < count; ++i) {
    const KsKernel& k = list[i];
    if (M <= kKsFewRows && (k.fm > 1 || k.waves != 8)) continue;
    const int64_t cols = (p5 ? k.fn / 2 : k.fn) * 16;
    const int64_t tiles = ((M + k.fm * 16 - 1) / (k.fm * 16)) * ((N + cols - 1) / cols);
    if (tiles > (int64_t)1 << 28) continue;
    const int64_t c = (tiles + cus - 1) / cus;
    if (k.waves == 4 ? c < 2 : c > 1 && k.fm + k.fn > 6 && k.fm + k.fn < 10) continue;
    const double one = (double)(k.fm + k.fn) * 32.0 * (double)K / kKsBytesPerNs + kKsTileNs;
    // an eight-wave workgroup's next tile waits for the one before; past three
    // tiles of a four-wave one the row tiles' re-reads no longer meet in L2
    const double slow = (c == 1 ? 1.0 : k.waves == 8 ? 1.45 : c > 3 ? 1.3 : 1.0) * spill;
    const double t = kKsFixedNs + cold_ns + (double)c * one * slow;
    if (!best || t < *ns) {
      best = &k;
      *ns = t;
    }
  }
  return best;
}

KsArgs ks_args(const KsCall& c, const KsKernel& k, bool p5) {
  KsArgs g{};
  g.x = reinterpret_cast<const char*>(c.x);
  g.resid = c.resid;
  g.ldr = c.ldr;
  g.count = c.count;
  g.M = (int)c.M;
  g.ldx = (int)(c.ldx * 2);
  g.units = (int)(c.K / kKsUnit);
  g.act = c.act;
  g.tiles_m = (int)((c.M + k.fm * 16 - 1) / (k.fm * 16));
  const int cols = (p5 ? k.fn / 2 : k.fn) * 16;
  int64_t first = 0;
  for (int i = 0; i < c.count; ++i) {
    const KsSeg& s = c.seg[i];
    g.first[i] = (int)first;
    g.seg[i] = KsSegArgs{reinterpret_cast<const char*>(s.w0), reinterpret_cast<const char*>(s.w1),
                         s.bias, s.out, s.ldo, (int)s.N, (int)(s.ldw0 * 2), (int)(s.ldw1 * 2)};
    first += (s.N + cols - 1) / cols;
  }
  for (int i = c.count; i <= kKsMaxSegs; ++i) g.first[i] = (int)first;
  g.tiles = (int)first * g.tiles_m;
  return g;
}

int ks_run(const KsKernel& k, bool nt, const KsArgs& g, hipStream_t st) {
  const unsigned grid = (unsigned)((g.tiles + 7) / 8 * 8);
  hipLaunchKernelGGL(nt ? k.kern_nt : k.kern, dim3(grid), dim3((unsigned)k.waves * 64), 0, st, g);
  return launch_status();
}

}  // namespace

int64_t device_cus() {
  int dev = 0, n = 0;
  static std::atomic<int> cus[64];
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (int c = cus[dev].load(std::memory_order_relaxed)) return c;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  cus[dev].store(n, std::memory_order_relaxed);
  return n;
}

double ks_time_ns(bool p5, int64_t M, int64_t N, int64_t K, int64_t cus, TileShape* tile) {
  double ns = 0.0;
  if (M <= 0 || N <= 0 || K <= 0 || K % kKsUnit || cus <= 0) return -1.0;
  const KsKernel* const k = ks_choose(p5, M, N, K, cus, &ns);
  if (!k) return -1.0;
  if (tile) *tile = TileShape{k->fm * 16, k->fn * 16, k->waves};
  return ns;
}

int launch_ks(bool p5, const KsCall& c, hipStream_t st) {
  int64_t N = 0;
  for (int i = 0; i < c.count; ++i) N += c.seg[i].N;
  const int64_t cus = device_cus();
  double ns = 0.0;
  const KsKernel* const k = cus > 0 ? ks_choose(p5, c.M, N, c.K, cus, &ns) : nullptr;
  if (!k) return UMIC_ERR_UNSUPPORTED;
  const KsArgs g = ks_args(c, *k, p5);
  const bool nt = g.tiles_m == 1 && N * c.K * 2 * (p5 ? 2 : 1) >= kKsStreamBytes;
  return ks_run(*k, nt, g, st);
}

}  // namespace umic

// Projection GEMMs of decode/verify batches for gfx950 (MI355X).
//
// y[rows, n] = x[rows, k] . W[n, k]^T (fp16 in, fp32 sums) for the q/k/v, O
// and down projections of a layer at decode/verify batch sizes (rows <= 128),
// and the FFN's up/gate projection with its SiLU-and-mul.  The weight is the
// whole of the traffic (x is at most 3 MB and stays in L2), so the kernels are
// a stream of W through the compute units:
//
//   - the work is cut into (n-tile of TN columns, k-range) units, one
//     workgroup each, about one per compute unit: TN columns over all of k
//     would give each CU too little of W and make it re-read all of x, so
//     k is split into `splits` ranges and every unit writes fp32 partial
//     sums [split][rows][n]; the consumer of the projection (the next
//     add-RMSNorm, the QK-norm/RoPE/KV-store prologue, or a small sum pass)
//     adds the splits in split order and rounds to fp16 once, which is the
//     GEMM output rounding of F.linear;
//   - a gated unit (the up/gate projection) streams 16 p up rows and the
//     matching gate rows over all of k, applies the SiLU-and-mul to its
//     accumulators and writes fp16 (no partials);
//   - W and x arrive in LDS slots by global_load_lds_dwordx4; rows are
//     XOR-swizzled per 16-byte chunk so the 16 rows an MFMA operand read
//     touches hit distinct banks; v_mfma_f32_16x16x32_f16 with A = weight
//     rows, B = x rows;
//   - stream_gemm_kernel (gated units, and columns tiles of 64 and more):
//     four waves only load, the others only compute, so the stream runs on
//     under the arithmetic; linear_partials_kernel (column tiles of 16 and
//     32, the small models' shapes, where a unit is a few steps long and the
//     launch is most of the time): every wave does both.
//
// Measured on MI355X, us per call with the weights rotated past the MALL,
// before (every wave loading and computing) -> now: Qwen3-8B up/gate 24576 x
// 4096 at 16 / 80 / 128 rows 37.7 / 42.3 / 57.6 -> 34.6 / 36.6 / 42.8 (the W
// stream alone 33.5); q/k/v 4096 -> 6144 10.4 / 14.4 / 18.1 -> 10.3 / 13.6 /
// 16.2; down 12288 -> 4096 17.1 / 22.5 / 34.9 -> 17.2 / 21.5 / 26.1; O 4096 ->
// 4096 7.3 / 9.9 / 13.5 -> 7.2 / 9.4 / 11.1.  Qwen3-0.6B at 64 rows: up/gate
// 9.8 -> 6.0; q/k/v 4.9, O 4.0, down 4.8 stay with the small-tile kernel,
// which the split roles did not beat there.
#include <algorithm>
#include <atomic>

#include "nsd_device.h"

namespace nsd {
namespace {

constexpr int kKStep = 128;                 // k per ring step
constexpr int kStepRowBytes = kKStep * 2;   // one row's chunk of a step
constexpr int kGemmThreads = 256;
constexpr int kGemmLds = 160 * 1024;        // LDS one workgroup may use
constexpr int kMaxSplits = 8;
constexpr int kMaxRowTiles = 8;             // 128 rows

__device__ inline int chunk_swizzle(int row) { return row & 15; }

// NT: non-temporal, for the weight rows: they pass through the caches once a
// forward, and kept out of the replacement they stream faster (the 24576 x
// 4096 weight alone, in 96-row units: 40.8 -> 37.9 us).  The x rows, which
// every workgroup re-reads, keep the default policy.  With x and the
// arithmetic, up/gate + down at 80 rows went from 74.9 to 69.5 us a layer.
// A weight small enough to stay in the MALL from call to call loses by it
// (1024 x 3072 called alone again and again 3.8 -> 4.3 us); a forward's
// weights do not stay.
template <bool NT>
__device__ inline void gemm_dma(uint32_t lds_addr, const void* src) {
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off nt"
                 :
                 : "s"(lds_addr), "v"(src)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(lds_addr), "v"(src)
                 : "memory", "m0");
}
template <int N>
__device__ inline void gemm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ inline void gemm_barrier() { asm volatile("s_barrier" ::: "memory"); }

// ---- small column tiles ----------------------------------------------------
//
// Each of the four waves brings its share of a step (128 k: TN weight rows
// and the x rows) and computes one of its four 32-k sub-steps over every
// output tile; the waves' sums are added in LDS, in wave order, at the end.
template <int MT, int TN>
struct LinearShape {
  static constexpr int kRows = TN + 16 * MT;            // rows of one slot: weight, then x
  static constexpr int kSlot = kRows * kStepRowBytes;
  static constexpr int kRing = 3;                       // two steps in flight
  static constexpr int kLds = kRing * kSlot;
  static constexpr int kDmaPerWave = kRows / 16;        // 4 rows per instruction, 4 waves
  static_assert(kLds <= kGemmLds, "ring");
  static_assert(4 * (TN / 16) * MT * 1024 <= kLds, "reduction buffer");
};

// Unit u = (n-tile u % n_tiles, split u / n_tiles); split s covers steps
// [s T / splits, (s+1) T / splits) of the T = k / 128 steps.
template <int MT, int TN>
__global__ __launch_bounds__(kGemmThreads) void linear_partials_kernel(const f16* __restrict__ x,
                                                                       const f16* __restrict__ w,
                                                                       float* __restrict__ part, int rows,
                                                                       int n, int k, int splits, int n_tiles) {
  using S = LinearShape<MT, TN>;
  constexpr int R = S::kRing;
  constexpr int NI = S::kDmaPerWave;
  constexpr int NJ = TN / 16;
  extern __shared__ __align__(16) char smem_raw[];
  lds_char* ring = (lds_char*)smem_raw;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int nt = blockIdx.x % n_tiles, split = blockIdx.x / n_tiles;
  const int n0 = nt * TN;
  const int T = k / kKStep;
  const int t0 = (int)((int64_t)split * T / splits);
  const int steps = (int)((int64_t)(split + 1) * T / splits) - t0;

  // DMA instruction i of this wave brings rows 4(4i + wave) .. +3 of a slot;
  // lane l the 16-byte chunk (l % 16) ^ swizzle(row) of row l / 16 of them.
  const f16* src[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int row = (4 * i + wave) * 4 + (lane >> 4);
    const int chunk = (lane & 15) ^ chunk_swizzle(row);
    const f16* base = row < TN ? w + (int64_t)(n0 + row) * k
                               : x + (int64_t)(row - TN < rows ? row - TN : rows - 1) * k;  // pad rows: a real row
    src[i] = base + (int64_t)t0 * kKStep + chunk * 8;
  }
  auto issue = [&](int t) {
    const lds_char* slot = ring + (t % R) * S::kSlot;
    static_for<NI>([&](auto u) {
      constexpr int i = decltype(u)::value;  // instructions below TN / 16 bring weight rows, the rest x rows
      gemm_dma<(i < TN / 16)>((uint32_t)(uintptr_t)(slot + (4 * i + wave) * 1024), src[i] + (int64_t)t * kKStep);
    });
  };
  f32x4 acc[NJ][MT];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  int issued = 0;
  for (; issued < R - 1 && issued < steps; ++issued) issue(issued);
  for (int t = 0; t < steps; ++t) {
    // this wave's loads of step t have landed (the ring's later steps may
    // still be in flight), then every wave's; the slot of step t-1 is free
    if (issued - t - 1 >= R - 2) gemm_wait<(R - 2) * NI>();
    else gemm_wait<0>();
    gemm_barrier();
    if (issued < steps) issue(issued++);
    const lds_char* sl = ring + (t % R) * S::kSlot;
    const int ch = 4 * wave + lg;  // lane group's 8 k of the sub-step
    f16x8 a[NJ], b[MT];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int row = 16 * j + lr;
      a[j] = *(const lds_f16x8*)(sl + row * kStepRowBytes + ((ch ^ chunk_swizzle(row)) << 4));
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = TN + 16 * i + lr;
      b[i] = *(const lds_f16x8*)(sl + row * kStepRowBytes + ((ch ^ chunk_swizzle(row)) << 4));
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[j][i] = mfma_k32(a[j], b[i], acc[j][i]);
  }
  // lane (lg, lr) holds columns 4lg .. 4lg+3 of an n-tile for row lr of an
  // m-tile: 16 contiguous bytes of the partial row
  float* out = part + (int64_t)split * rows * n;
  __syncthreads();  // the ring is drained: its LDS holds the waves' sums
  f32x4* red = reinterpret_cast<f32x4*>(smem_raw);  // [wave][tile][lane]
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) red[(wave * NJ * MT + j * MT + i) * 64 + lane] = acc[j][i];
  __syncthreads();
  for (int tile = wave; tile < NJ * MT; tile += 4) {
    f32x4 v = red[tile * 64 + lane];
#pragma unroll
    for (int q = 1; q < 4; ++q) v += red[(q * NJ * MT + tile) * 64 + lane];
    const int j = tile / MT, m = 16 * (tile % MT) + lr;
    if (m < rows) *reinterpret_cast<f32x4*>(out + (int64_t)m * n + n0 + 16 * j + 4 * lg) = v;
  }
}

// ---- large column tiles and the gated projection ---------------------------
//
// kProducers waves bring the unit's W rows and x through LDS and do nothing
// else; NW x MW consumer waves compute.  Work goes in k blocks of KS: an
// x slab (16 MT rows x KS) and SUB = TN / RS steps, each a slot of RS weight
// rows x KS; a block's slab is issued with its first step.  With KS = 256 an
// instruction brings 512-byte runs of two rows: the W stream of the Qwen3-8B
// up/gate alone takes 33.8 us in 512-byte runs, 37.9 in 256-byte runs and
// 34.3 in 1 KB runs, whatever the depth (48 to 144 KB in flight per CU), so
// the ring is three slots and the LDS goes to x.  The x slabs cost the stream
// under 2 us: the same x loaded to registers by the consumers, 64-byte runs of
// 16 rows, cost 12.  Consumer (ng, mg) takes the slot's tiles ng, ng + NW, ...
// and the row tiles mg, mg + MW, ... over all of the block's k, with its x
// operands kept in registers over the block's steps where they fit.  Every sum
// runs over k in order in one accumulator, so a row's bits do not depend on
// the rows beside it.
//
// Step s may be issued once the consumers have passed the barrier of step
// s - R + 1, that is once they are done with step s - R, and with the slab of
// the block XD before when that one's last step is no later: R - 1 <= (XD -
// 1) SUB.
constexpr int kProducers = 4;

template <int MT_, int TN_, int RS_, int KS_, int R_, int XD_, int NW_, int MW_, bool GATED_>
struct StreamShape {
  static constexpr int MT = MT_, TN = TN_, RS = RS_, KS = KS_, R = R_, XD = XD_, NW = NW_, MW = MW_;
  static constexpr bool GATED = GATED_;
  static constexpr int NC = NW * MW, SUB = TN / RS, JS = RS / 16;
  static constexpr int kRowB = KS * 2, kSlot = RS * kRowB, kSlab = 16 * MT * kRowB;
  static constexpr int WI = kSlot / 1024 / kProducers, XI = kSlab / 1024 / kProducers;  // instructions per producer
  static constexpr int RPI = 1024 / kRowB;                                              // rows per instruction
  static constexpr int KW = KS / 32, JW = JS / NW, MI = (MT + MW - 1) / MW;
  static constexpr bool HOIST = SUB > 1 && KW * MI <= 16;  // a block's x operands in at most 64 registers
  static constexpr int kThreads = (kProducers + NC) * kWave;
  static constexpr int kLds = R * kSlot + XD * kSlab;
  static_assert(WI * kProducers * 1024 == kSlot && XI * kProducers * 1024 == kSlab && JW * NW == JS && SUB * RS == TN);
  static_assert(R >= 2 && R - 1 <= (XD - 1) * SUB && kLds <= kGemmLds);
  static_assert(!GATED || (SUB * JW) % 2 == 0);
};

// Unit u as in linear_partials_kernel, in blocks of KS k.
template <class S>
__global__ __launch_bounds__(S::kThreads) void stream_gemm_kernel(const f16* __restrict__ x,
                                                                  const f16* __restrict__ w,
                                                                  float* __restrict__ part, int rows, int n, int k,
                                                                  int splits, int n_tiles, f16* __restrict__ y) {
  constexpr int MT = S::MT, TN = S::TN, RS = S::RS, KS = S::KS, R = S::R, XD = S::XD, P = kProducers;
  constexpr int SUB = S::SUB, WI = S::WI, XI = S::XI, RPI = S::RPI, KW = S::KW, JW = S::JW, MI = S::MI;
  extern __shared__ __align__(16) char smem_raw[];
  lds_char* slabs = (lds_char*)smem_raw;
  lds_char* ring = slabs + XD * S::kSlab;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt = blockIdx.x % n_tiles, split = blockIdx.x / n_tiles;
  const int n0 = nt * (S::GATED ? TN / 2 : TN);
  const int T = k / KS;
  const int t0 = (int)((int64_t)split * T / splits);
  const int blocks = (int)((int64_t)(split + 1) * T / splits) - t0;
  const int steps = blocks * SUB;

  if (wave < P) {
    // instruction i of this wave brings rows RPI (P i + wave) .. of a slot or
    // slab; a lane the 16-byte chunk q ^ (row % 16) of its row
    const int sub_row = lane / (kWave / RPI), q = lane % (kWave / RPI);
    const f16* xsrc[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int r = (i * P + wave) * RPI + sub_row;
      xsrc[i] = x + (int64_t)(r < rows ? r : rows - 1) * k + (int64_t)t0 * KS + (q ^ chunk_swizzle(r)) * 8;
    }
    const f16* wsrc[SUB * WI];
#pragma unroll
    for (int i = 0; i < SUB * WI; ++i) {
      const int r = ((i % WI) * P + wave) * RPI + sub_row;
      const int row = (i / WI) * RS + r;  // the unit's row: gated, its up rows and then the gate rows, n further on
      const int wrow = !S::GATED || row < TN / 2 ? n0 + row : n + n0 + row - TN / 2;
      wsrc[i] = w + (int64_t)wrow * k + (int64_t)t0 * KS + (q ^ chunk_swizzle(r)) * 8;
    }
    int slot_no = 0;
    auto issue = [&](int blk, auto subc) __attribute__((always_inline)) {
      constexpr int sub = decltype(subc)::value;
      if constexpr (sub == 0) {
        const uint32_t slab = (uint32_t)(uintptr_t)(slabs + (blk % XD) * S::kSlab);
#pragma unroll
        for (int i = 0; i < XI; ++i) gemm_dma<false>(slab + (i * P + wave) * 1024, xsrc[i] + (int64_t)blk * KS);
      }
      const uint32_t slot = (uint32_t)(uintptr_t)(ring + slot_no * S::kSlot);
      slot_no = slot_no + 1 == R ? 0 : slot_no + 1;
#pragma unroll
      for (int i = 0; i < WI; ++i)
        gemm_dma<true>(slot + (i * P + wave) * 1024, wsrc[sub * WI + i] + (int64_t)blk * KS);
    };
    auto issue_step = [&](int s) __attribute__((always_inline)) {
      const int blk = s / SUB, sub = s - blk * SUB;
      static_for<SUB>([&](auto u) {
        if (sub == decltype(u)::value) issue(blk, u);
      });
    };
    int issued = 0;
    while (issued < R - 1 && issued < steps) issue_step(issued++);
    for (int s0 = 0; s0 < steps; s0 += SUB) {
      static_for<SUB>([&](auto u) {
        constexpr int sub = decltype(u)::value;
        // this wave's instructions of the R - 2 steps after this one may be
        // outstanding (their slabs among them); then every producer's step
        // has landed and the slot of the step before is free
        constexpr int newer = (R - 2) * WI + (sub + R - 2) / SUB * XI;
        static_assert(newer <= 63, "vmcnt range");
        if (issued - (s0 + sub) - 1 >= R - 2) gemm_wait<newer>();
        else gemm_wait<0>();
        gemm_barrier();
        if (issued < steps) issue_step(issued++);
      });
    }
    return;
  }

  const int c = wave - P;
  const int ng = c % S::NW, mg = c / S::NW;
  int xrow[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int t = i * S::MW + mg;  // past the row tiles: the last one again, not stored
    xrow[i] = (16 * (t < MT ? t : MT - 1) + lr) * S::kRowB;
  }
  f32x4 acc[SUB * JW][MI];
#pragma unroll
  for (int j = 0; j < SUB * JW; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  int slot_no = 0;
  for (int blk = 0; blk < blocks; ++blk) {
    const lds_char* slab = slabs + (blk % XD) * S::kSlab;
    f16x8 kept[S::HOIST ? KW : 1][MI];
#pragma unroll
    for (int sub = 0; sub < SUB; ++sub) {
      // this wave's reads of the step before are done, then the step is in
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      const lds_char* sl = ring + slot_no * S::kSlot;
      slot_no = slot_no + 1 == R ? 0 : slot_no + 1;
#pragma unroll
      for (int s = 0; s < KW; ++s) {
        const int ch = ((s * 4 + lg) ^ lr) << 4;
        f16x8 a[JW], b[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          if (S::HOIST && sub > 0) b[i] = kept[S::HOIST ? s : 0][i];
          else b[i] = *(const lds_f16x8*)(slab + xrow[i] + ch);
          if (S::HOIST && sub == 0) kept[S::HOIST ? s : 0][i] = b[i];
        }
#pragma unroll
        for (int j = 0; j < JW; ++j) a[j] = *(const lds_f16x8*)(sl + (16 * (ng + j * S::NW) + lr) * S::kRowB + ch);
#pragma unroll
        for (int j = 0; j < JW; ++j)
#pragma unroll
          for (int i = 0; i < MI; ++i) acc[sub * JW + j][i] = mfma_k32(a[j], b[i], acc[sub * JW + j][i]);
      }
    }
  }

  // lane (lg, lr) holds columns 4lg .. 4lg+3 of a tile for row lr of a row
  // tile.  Accumulator j is tile ng + (j % JW) NW of step j / JW; gated, the
  // first half are up tiles and the second their gate tiles.
  auto column = [&](int j) { return j / JW * RS + 16 * (ng + j % JW * S::NW) + 4 * lg; };
  auto store = [&](int j, int i, f32x4 v, f32x4 gate) {
    const int t = i * S::MW + mg, m = 16 * t + lr;
    if (t >= MT || m >= rows) return;
    if constexpr (S::GATED) {
      // the SiLU-and-mul of silu_and_mul_kernel on the fp16-rounded sums
      f16x4 h;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f16 up = (f16)v[e];
        const float gf = (float)(f16)gate[e];
        const f16 sg = (f16)(gf / (1.f + expf(-gf)));
        h[e] = (f16)((float)up * (float)sg);
      }
      *reinterpret_cast<f16x4*>(y + (int64_t)m * n + n0 + column(j)) = h;
    } else {
      *reinterpret_cast<f32x4*>(part + ((int64_t)split * rows + m) * n + n0 + column(j)) = v;
    }
  };
  constexpr int NT = SUB * JW, OUT = S::GATED ? NT / 2 : NT;  // accumulator tiles, of which stored
#pragma unroll
  for (int j = 0; j < OUT; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) store(j, i, acc[j][i], acc[S::GATED ? j + OUT : j][i]);
}

// y[i] = fp16(sum over splits of part[s][i]), eight elements per thread.
template <int S>
__global__ __launch_bounds__(256) void sum_partials_kernel(const float* __restrict__ part, int64_t per_split,
                                                           f16* __restrict__ y) {
  for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < per_split / 8; v += (int64_t)gridDim.x * 256) {
    f32x4 lo[S], hi[S];  // the splits' loads go out together
#pragma unroll
    for (int s = 0; s < S; ++s) {
      lo[s] = *reinterpret_cast<const f32x4*>(part + s * per_split + 8 * v);
      hi[s] = *reinterpret_cast<const f32x4*>(part + s * per_split + 8 * v + 4);
    }
#pragma unroll
    for (int s = 1; s < S; ++s) {
      lo[0] += lo[s];
      hi[0] += hi[s];
    }
    f16x8 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = (f16)lo[0][e];
      h[e + 4] = (f16)hi[0][e];
    }
    *reinterpret_cast<f16x8*>(y + 8 * v) = h;
  }
}

struct LinearConfig {
  int tn = 0, splits = 0;
};

// Column tile and k-split for an n x k projection on `cus` compute units:
// the configuration whose units fill the most of whole rounds of one unit
// per CU, with at least four steps per unit where k allows; ties go to the
// 64-column tile (measured fastest where several fill the chip), then 128,
// 32, 16.
LinearConfig choose_linear(int64_t n, int64_t k, int cus) {
  LinearConfig best;
  double best_fill = -1.0;
  const int64_t steps = k / kKStep;
  for (int tn : {64, 128, 32, 16}) {
    if (n % tn) continue;
    const int64_t tiles = n / tn;
    const int64_t cap = std::max<int64_t>(1, std::min<int64_t>(kMaxSplits, steps / 4));
    const int64_t splits = std::max<int64_t>(1, std::min<int64_t>(cap, cus / tiles));
    const int64_t units = tiles * splits;
    const int64_t rounds = (units + cus - 1) / cus;
    const double fill = (double)units / (double)(rounds * cus);
    if (fill > best_fill + 1e-9) {
      best_fill = fill;
      best.tn = tn;
      best.splits = (int)splits;
    }
  }
  return best;
}

int check_linear(int64_t n_rows, int64_t n_out, int64_t n_in, const char* who) {
  if (n_rows < 1 || n_rows > 16 * kMaxRowTiles)
    return fail(NSD_ERR_UNSUPPORTED, "%s: n_rows=%lld outside [1, %d]", who, (long long)n_rows, 16 * kMaxRowTiles);
  if (n_out < 16 || n_out % 16 || n_in < kKStep || n_in % kKStep || n_out > INT32_MAX || n_in > INT32_MAX)
    return fail(NSD_ERR_UNSUPPORTED, "%s: n_out=%lld (a multiple of 16), n_in=%lld (a multiple of 128)", who,
                (long long)n_out, (long long)n_in);
  return NSD_OK;
}

// Raises a kernel's dynamic-LDS limit once per process: a function-local
// static is initialised exactly once even when several threads launch at
// once, and a failure stays reported on every later call.
template <auto Kernel, int kLds>
int allow_lds() {
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  return attr == hipSuccess ? NSD_OK : fail(NSD_ERR_HIP, "linear: LDS attribute: %s", hipGetErrorString(attr));
}

struct GemmArgs {
  const f16* x;
  const f16* w;
  float* part;  // partials, or
  f16* y;       // the gated output
  int rows, n, k, splits;
  hipStream_t st;
};

template <class S>
int launch_stream(const GemmArgs& g) {
  if (int rc = allow_lds<&stream_gemm_kernel<S>, S::kLds>()) return rc;
  const int n_tiles = g.n / (S::GATED ? S::TN / 2 : S::TN);
  hipLaunchKernelGGL(stream_gemm_kernel<S>, dim3(n_tiles * g.splits), dim3(S::kThreads), S::kLds, g.st, g.x, g.w,
                     g.part, g.rows, g.n, g.k, g.splits, n_tiles, g.y);
  return launch_status(S::GATED ? "up_gate_silu_and_mul" : "linear");
}

template <int MT, int TN>
int launch_linear(const GemmArgs& g) {
  constexpr int MW = MT > 1 ? 2 : 1, NW = MT > 1 ? 2 : 4;  // one row tile: the waves split the columns
  if constexpr (TN == 64) {
    return launch_stream<StreamShape<MT, 64, 64, 128, 3, 3, NW, MW, false>>(g);
  } else if constexpr (TN == 128) {
    return launch_stream<StreamShape<MT, 128, 64, 128, 4, 3, NW, MW, false>>(g);
  } else {
    using S = LinearShape<MT, TN>;
    if (int rc = allow_lds<&linear_partials_kernel<MT, TN>, S::kLds>()) return rc;
    const int n_tiles = g.n / TN;
    hipLaunchKernelGGL((linear_partials_kernel<MT, TN>), dim3(n_tiles * g.splits), dim3(kGemmThreads), S::kLds, g.st,
                       g.x, g.w, g.part, g.rows, g.n, g.k, g.splits, n_tiles);
    return launch_status("linear");
  }
}

// A gated unit of PAIRS up tiles and their gate tiles.  k blocks of 256 while
// the x slabs leave room for three slots (up to 80 rows) and k allows, else
// of 128.
template <int MT, int PAIRS>
int launch_gated(const GemmArgs& g) {
  constexpr int TN = 32 * PAIRS;
  constexpr int MW = MT > 1 ? 2 : 1;
  if constexpr (PAIRS == 1) {
    // one slot holds the pair; a wave takes both of its tiles for every W-th row tile
    constexpr int W = MT < 4 ? MT : 4;
    if constexpr (MT <= 4)
      if (g.k % 256 == 0) return launch_stream<StreamShape<MT, TN, 32, 256, 3, 3, 1, W, true>>(g);
    return launch_stream<StreamShape<MT, TN, 32, 128, 4, 4, 1, W, true>>(g);
  } else {
    constexpr int RS = PAIRS == 3 ? 48 : 32, NW = RS / 16;
    if constexpr (MT <= 5)
      if (g.k % 256 == 0) return launch_stream<StreamShape<MT, TN, RS, 256, 3, 2, NW, MW, true>>(g);
    return launch_stream<StreamShape<MT, TN, RS, 128, 4, 3, NW, MW, true>>(g);
  }
}

// Calls f<MT>() for the row tiles' count mt in 1 .. kMaxRowTiles.
template <class F, int... I>
int with_row_tiles(std::integer_sequence<int, I...>, int mt, F&& f) {
  int rc = NSD_ERR_UNSUPPORTED;
  ((mt == I + 1 ? (rc = f(std::integral_constant<int, I + 1>{}), 0) : 0), ...);
  return rc;
}
template <class F>
int with_row_tiles(int rows, F&& f) {
  return with_row_tiles(std::make_integer_sequence<int, kMaxRowTiles>{}, (rows + 15) / 16, f);
}

// Up/gate tile pairs per gated unit, or 0 for a shape the ring kernel takes:
// the most units (the fewest pairs) that one round of the compute units
// holds.  From seven tenths of them busy the gated units are faster at every
// row count measured (ring / gated, us at 1 / 64 / 128 rows; 180 units: 2880
// columns x 1024 5.1 / 9.8 / 15.6 and 4.6 / 6.0 / 8.3, x 4096 13.6 / 23.2 /
// 39.1 and 10.5 / 14.9 / 23.1; 192: 12288 x 2560 22.7 / 27.5 / 37.9 and 21.1 /
// 23.8 / 29.6).  Below, the ring kernel's balanced ranges use every compute
// unit, and it depends on the pairs: 152 units of four pairs (9728 columns) x
// 2560 19.8 / 26.0 / 36.2 and 22.2 / 25.2 / 32.9, but of one (2432) x 2560 9.5
// / 17.2 / 28.2 and 7.4 / 10.7 / 16.4; those stay with the ring kernel.
int gated_pairs(int64_t inter, int cus) {
  for (int pairs = 1; pairs <= 4; ++pairs) {
    if (inter % (16 * pairs)) continue;
    const int64_t units = inter / (16 * pairs);
    if (units <= cus) return units * 10 >= cus * 7 ? pairs : 0;
  }
  return 0;
}

}  // namespace

// Compute units of the current device (queried once per device: the
// decoder stack asks for every projection it enqueues).
int device_cus(int* cus) {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> cached[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess && dev >= 0 && dev < kMaxDevices) {
    const int c = cached[dev].load(std::memory_order_relaxed);
    if (c > 0) {
      *cus = c;
      return NSD_OK;
    }
  }
  if (e == hipSuccess) e = hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return fail(NSD_ERR_HIP, "linear: %s", hipGetErrorString(e));
  if (*cus < 1) return fail(NSD_ERR_HIP, "linear: device %d reports %d compute units", dev, *cus);
  if (dev >= 0 && dev < kMaxDevices) cached[dev].store(*cus, std::memory_order_relaxed);
  return NSD_OK;
}

int up_gate_silu_gated(const void* x, const void* up_gate, void* y, int64_t n_rows, int64_t hidden, int64_t inter,
                       void* stream, bool* served) {
  *served = false;
  int cus = 0;
  if (int rc = device_cus(&cus)) return rc;
  const int pairs = gated_pairs(inter, cus);
  if (pairs == 0 || n_rows > 16 * kMaxRowTiles || hidden % kKStep) return NSD_OK;
  *served = true;
  const GemmArgs g{static_cast<const f16*>(x), static_cast<const f16*>(up_gate), nullptr, static_cast<f16*>(y),
                   (int)n_rows, (int)inter, (int)hidden, 1, as_stream(stream)};
  return with_row_tiles(g.rows, [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    switch (pairs) {
      case 1: return launch_gated<MT, 1>(g);
      case 2: return launch_gated<MT, 2>(g);
      case 3: return launch_gated<MT, 3>(g);
      default: return launch_gated<MT, 4>(g);
    }
  });
}

}  // namespace nsd

using namespace nsd;

extern "C" int nsd_linear_splits(int64_t n_rows, int64_t n_out, int64_t n_in, int* splits) {
  if (splits == nullptr) return fail(NSD_ERR_INVALID, "linear_splits: null output");
  if (int rc = check_linear(n_rows, n_out, n_in, "linear_splits")) return rc;
  int cus = 0;
  if (int rc = device_cus(&cus)) return rc;
  *splits = choose_linear(n_out, n_in, cus).splits;
  return NSD_OK;
}

extern "C" int nsd_linear_partials(const void* x, const void* w, float* partials, int64_t n_rows, int64_t n_out,
                                   int64_t n_in, void* stream) {
  if (int rc = check_linear(n_rows, n_out, n_in, "linear_partials")) return rc;
  if (!x || !w || !partials) return fail(NSD_ERR_INVALID, "linear_partials: null pointer");
  if (!aligned16(x) || !aligned16(w) || !aligned16(partials))
    return fail(NSD_ERR_UNSUPPORTED, "linear_partials: pointers must be 16-byte aligned");
  int cus = 0;
  if (int rc = device_cus(&cus)) return rc;
  const LinearConfig c = choose_linear(n_out, n_in, cus);
  const GemmArgs g{static_cast<const f16*>(x), static_cast<const f16*>(w), partials, nullptr, (int)n_rows, (int)n_out,
                   (int)n_in, c.splits, as_stream(stream)};
  return with_row_tiles(g.rows, [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    switch (c.tn) {
      case 16: return launch_linear<MT, 16>(g);
      case 32: return launch_linear<MT, 32>(g);
      case 64: return launch_linear<MT, 64>(g);
      default: return launch_linear<MT, 128>(g);
    }
  });
}

extern "C" int nsd_sum_partials(const float* partials, int splits, void* y, int64_t n_rows, int64_t n_out,
                                void* stream) {
  if (n_rows < 0 || n_out < 8 || n_out % 8 || splits < 1 || splits > kMaxSplits)
    return fail(NSD_ERR_INVALID, "sum_partials: rows=%lld n_out=%lld splits=%d", (long long)n_rows,
                (long long)n_out, splits);
  if (n_rows == 0) return NSD_OK;
  if (!partials || !y) return fail(NSD_ERR_INVALID, "sum_partials: null pointer");
  if (!aligned16(partials) || !aligned16(y))
    return fail(NSD_ERR_UNSUPPORTED, "sum_partials: pointers must be 16-byte aligned");
  const int64_t per = n_rows * n_out;
  const unsigned grid = (unsigned)std::min<int64_t>((per / 8 + 255) / 256, 1024);
  with_splits(splits, [&](auto count) {
    hipLaunchKernelGGL(sum_partials_kernel<decltype(count)::value>, dim3(grid), dim3(256), 0, as_stream(stream),
                       partials, per, static_cast<f16*>(y));
  });
  return launch_status("sum_partials");
}

// Dense projection GEMM with fused epilogues for the encoder layers, fp16 /
// bf16, gfx950 (CDNA4).
//
//   Y[m, n] = epilogue( sum_k X[m, k] * W[n, k] + bias[n] )
//
// X is the row-major activation [M, K], W the nn.Linear weight [N, K] (both
// K-contiguous), Y row-major [M, N].  Epilogues (applied to the sum rounded to
// the dtype first, as nn.Linear's output is):
//   kEpiBias     : Y = T(acc + bias)                         (QKV projection)
//   kEpiBiasGelu : Y = T(gelu_erf(T(acc + bias)))            (FFN intermediate,
//                  DebertaV2Intermediate = dense then ACT2FN["gelu"], the exact
//                  erf form; _reference.py:470-471)
//   kEpiBiasAdd  : Y = T(T(acc + bias) + R[m, n])            (dense + residual
//                  of DebertaV2SelfOutput / DebertaV2Output before LayerNorm,
//                  _reference.py:108-112, 482-485)
//
// What bounds it.  With tiles of 256 rows and a long K the loop is near the matrix unit:
// at M = 16384, N = K = 3072 (fp16) the 256 x 256 tile takes 232-254 us (two chips), 1.2-1.3
// PFLOP/s, its matrix pipe busy 67-69 % at the clock the power limit leaves
// (1.8 GHz); a loop of 32-deep steps in the compiler's own order took 292 us against 235.  At
// K = 768 the start of a tile and the stores at its end are as long as the loop (16384 rows:
// QKV 62-73 us, pipe busy 42 %; FFN intermediate with GELU 88-93 us, 39 %); with few rows it is
// the latency of the copies.  (profiles/gemm_sq_counters.md)

// Slabs of 64 k.  X and W are copied straight into LDS (buffer loads with the
// LDS bit, 16 bytes a lane: no registers, no address arithmetic in the loop)
// as slabs of 64 k, so that a row of a copy is one whole 128-byte line: with
// 32-deep slabs (64-byte rows) L2 serves twice as many requests for the same
// bytes (256 x 256 tile, N = K = 3072: 250 against 235 us).  A slab row is 128 bytes of LDS whose
// eight 16-byte chunks are permuted by slab_swizzle(row), so that of the 16 rows
// whose chunk 16 lanes read (an MFMA fragment) no two lie in the same banks; the counters still
// show four conflict cycles a read.  STAGES slabs form a ring.
//
// One slab is two 32-deep MFMA steps.  The fragments of a step are read from
// LDS during the MFMAs of the step before (two register sets).  Between the
// two steps of slab t stands the only barrier of the slab: every wavefront has
// then its last fragments of slab t in registers and its own copies of slab
// t + 1 have landed, so that after it slab t + 1 may be read and slab t be
// overwritten by the copies of slab t + STAGES, which are issued during the
// second step.
//
// The order inside a step is written down (sched_barrier between the groups):
// fragment reads and copies are spread over the first three quarters of the
// MFMAs.  Left to the compiler they all come first, and the matrix pipe waits
// for them: 255 against 235 us (N = K = 3072), 82 against 78.5 us at K = 768.
//
// MFMA v_mfma_f32_16x16x32_{f16,bf16} with the weight as the A operand, so a
// lane's accumulators of a 16 x 16 block are four consecutive outputs of one
// row.  The rows of W are assigned to the blocks so that the blocks 2i and
// 2i + 1 of a lane hold eight consecutive outputs (w_row): the epilogue writes
// 16 bytes a lane straight from the registers, with no pass through LDS.
//
// Launch order: workgroup p runs on XCD p % 8.  The tiles are split over the XCDs
// in a grid of xcds_m x 8 / xcds_m ranges, so that the rows of X and of W that one
// XCD reads, which its L2 keeps, are few (launch_gemm; 2048 x 4608 x 1536 on
// 128 x 192 tiles 40 -> 33 us against ranges of whole rows).
//
// k order: every XCD starts at a slab of its own and wraps around.  All tiles walk
// k together, and rows are K * 2 bytes apart, so with K = 3072 or 6144 the rows of
// one slab lie in a few of the memory channels only; eight starting points reach
// eight times as many (4096 x 768 x 3072 30.4 -> 25.4 us, 2048 x 1536 x 6144 57 -> 53).
// So the order of a row's fp32 sums depends on the tile that it lies in: equal rows can differ
// in the last bits.  A start that depends on the columns alone would make them equal within
// a call; it costs 2 % on average (2048 x 1536 x 6144 50.6 -> 60.1 us).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

#include "device_common.h"
#include "dflash.h"
#include "gemm_tile.h"
#include "layernorm.h"

namespace dflash {

namespace {

constexpr int kEpiBias = 0;
constexpr int kEpiBiasGelu = 1;
constexpr int kEpiBiasAdd = 2;
constexpr int kEpiPartial = 3;  // fp32 sums of one of `splits` ranges of K, no bias

// GELU in its erf form, x Phi(x), with Phi(-a) = 2^P(a) for a = |x|: P is a polynomial
// fitted to log2 Phi(-a) where the type's results are not 0: degree 8 on [0, 6] for fp16,
// 10 on [0, 13.3] for bf16, whose range keeps the tail.  Minimax of the relative error of
// Phi(-a), weighted to at most that of formula 7.1.26 of Abramowitz & Stegun everywhere;
// P(0) = -1 exactly, and the leading coefficient is negative, so P falls without bound past
// the range and 2^P goes to 0.  Over all inputs, evaluated in fp32, against that formula
// (which needs a reciprocal besides the exponential):
//                                  fp16: here / formula      bf16: here / formula
//   results not the rounded exact       36 / 256                  77 / 169
//   largest error                  3.7e-7 / 3.9e-7           3.1e-7 / 3.7e-7
//   relative, -5 < x < 0           6e-4 / 1.6e-3             7e-4 / 1.6e-3
//   relative, -6 < x < -5        1.5e-3 / 3.6e-3           2.0e-3 / 3.6e-3
//   relative, -12.9 < x < -6        (0 in fp16)            3.5e-3 / 3.8e-2
// Below x = -12.9, where Phi leaves the normal numbers of fp32, the result is -0.
// Degree 8 on [0, 6] in both types left bf16 with 65 % at x = -8; its two more steps
// cost 95.6 -> 97.4 us (16384 x 3072 x 768).  Degree 9 has 5.9e-7 as its largest error.
template <typename T>
__device__ inline float gelu_erf(float x) {
  constexpr bool kTail = std::is_same_v<T, __bf16>;
  constexpr float kP16[9] = {-1.0f,
                             -1.151114583015442f,
                             -0.4591211974620819f,
                             -0.052764665335416794f,
                             0.007448446471244097f,
                             -0.0004256263200659305f,
                             -7.005319639574736e-05f,
                             1.575876012793742e-05f,
                             -9.36769765758072e-07f};
  constexpr float kPb16[11] = {-1.0f,
                               -1.1511175632476807f,
                               -0.45909154415130615f,
                               -0.05285187065601349f,
                               0.00755681749433279f,
                               -0.00048680207692086697f,
                               -5.7015706261154264e-05f,
                               1.6698662875569426e-05f,
                               -1.668640265961585e-06f,
                               7.945903490735873e-08f,
                               -1.4974058659689149e-09f};
  constexpr int kDegree = kTail ? 10 : 8;
  auto coefficient = [&](int k) { return kTail ? kPb16[k] : kP16[k < 9 ? k : 8]; };
  const float a = fabsf(x);
  float p = coefficient(kDegree);
#pragma unroll
  for (int k = kDegree - 1; k >= 0; --k) p = fmaf(p, a, coefficient(k));
  const float tail = __builtin_amdgcn_exp2f(p);  // Phi(-|x|)
  return x * (x >= 0.0f ? 1.0f - tail : tail);
}

// One buffer_load_dwordx4 with the LDS bit: 16 bytes per lane from `off` + `scalar`
// (`scalar` uniform; zeros where `off` is past the resource's size) to LDS at `lds` + 16 *
// lane (`lds` uniform, in M0, which nothing else in these kernels uses and clang does not take
// as a clobber; one wait state between the write of M0 and the load).  Inline assembly, so
// that the compiler does not wait for copies in flight before fragment reads; they are
// awaited by wait_vmem and the slab's barrier.
__device__ inline void copy16_to_lds(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t scalar,
                                     uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds"
      :
      : "s"(lds), "v"(off), "s"(r), "s"(scalar)
      : "memory");
}

// The same from a 64-bit address per lane, for operands whose tile does not fit
// the 32-bit offsets of a buffer resource.
__device__ inline void copy16_to_lds_far(const void* src, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off"
      :
      : "s"(lds), "v"(src)
      : "memory");
}

// 16-byte store at byte `off` of a buffer, written through the L2 (scope bit sc1).
// For outputs that only a later kernel reads: as dirty lines they push out what this
// kernel still reads and wait to be written back at its end.
__device__ inline void store_through(__amdgpu_buffer_rsrc_t r, uint32_t off, u32x4_t v) {
  constexpr int kSc1 = 16;
  __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, kSc1);
}
// Widest Y whose tile of up to 256 rows 32-bit byte offsets reach.
constexpr int kMaxThroughN = 1 << 20;

// Wait until at most N of this thread's vector-memory operations are pending.
template <int N>
__device__ inline void wait_vmem() {
  static_assert(N >= 0 && N <= 63, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace

struct GemmArgs {
  const void* x;
  const void* w;
  const void* bias;
  const void* residual;
  void* y;
  int M, N, K;
  int m_blocks, n_blocks;
  int through;  // write Y through the L2 (store_through)
  int splits;   // ranges of K (kEpiPartial; y is fp32 [splits, M, N]), else 1
  int xcds_m;  // XCDs along the rows (1, 2, 4, 8); 8 / xcds_m along the columns
};

template <typename T, int EPI, typename CF, Copies COPIES>
__global__ __launch_bounds__(CF::THREADS, CF::WGS) void gemm_kernel(GemmArgs a) {
  using M = Mma<T>;
  using F = typename M::frag;
  constexpr int MB = CF::MB;
  constexpr int NB = CF::NB;
  constexpr int S = CF::STAGES;
  constexpr int kMfmas = MB * NB;   // of one step
  constexpr int kReads = MB + NB;   // fragment reads of one step
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15;
  const int g = lane >> 4;
  const int wm = wave % CF::WAVES_M;  // wavefront row block
  const int wn = wave / CF::WAVES_M;  // wavefront column block

  // Tile of this workgroup (see the file comment): the tile ranges of XCD p % 8,
  // columns fastest.
  const int p = blockIdx.x;
  const int split = EPI == kEpiPartial ? (p >> 3) % a.splits : 0;
  const int index = EPI == kEpiPartial ? (p >> 3) / a.splits : p >> 3;
  const int xm = (p & 7) % a.xcds_m;
  const int xn = (p & 7) / a.xcds_m;
  const int m_lo = a.m_blocks * xm / a.xcds_m;
  const int n_lo = a.n_blocks * xn * a.xcds_m / 8;
  const int cols = a.n_blocks * (xn + 1) * a.xcds_m / 8 - n_lo;
  const int mt = index / max(cols, 1);
  const int mb = m_lo + mt;
  const int nb = n_lo + index - mt * cols;
  if (cols == 0 || mb >= a.m_blocks * (xm + 1) / a.xcds_m) return;  // ranges differ in size
  const int m_base = mb * CF::BM;
  const int n_base = nb * CF::BN;
  const int ld = a.K;  // row stride of X and W
  const KRange range = k_range(a.K, split, EPI == kEpiPartial ? a.splits : 1);
  const int KT = range.slabs;
  const int K = range.k;  // of this workgroup
  const uint32_t row_bytes = static_cast<uint32_t>(ld) * 2u;
  const int rows = min(CF::BM, a.M - m_base);
  const T* X = reinterpret_cast<const T*>(a.x) + static_cast<int64_t>(m_base) * ld + range.first * kSlabK;
  const T* W = reinterpret_cast<const T*>(a.w) + static_cast<int64_t>(n_base) * ld + range.first * kSlabK;
  const uint32_t x_bytes = tile_bytes(rows, row_bytes, range);
  const uint32_t w_bytes = tile_bytes(CF::BN, row_bytes, range);

  // Byte offset of this lane's 16 bytes of copy j from the tile's first row.
  uint32_t xoff[CF::A_LOADS], woff[CF::B_LOADS];
#pragma unroll
  for (int j = 0; j < CF::A_LOADS; ++j) {
    const int r = copy_row<CF>(j, wave, lane);
    xoff[j] = static_cast<uint32_t>(r) * row_bytes + copy_chunk(r, lane) * 16;
  }
#pragma unroll
  for (int j = 0; j < CF::B_LOADS; ++j) {
    const int r = copy_row<CF>(j, wave, lane);
    woff[j] = static_cast<uint32_t>(w_row(r)) * row_bytes + copy_chunk(r, lane) * 16;
  }
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  // The k order starts at a slab of its own on each XCD and wraps around.
  const int k0 = K % kSlabK == 0 ? ((p & 7) * KT) >> 3 : 0;
  // Copy j of slab `kt` into ring stage `stage`.  Past the last slab it fetches
  // nothing (zeros into a stage that is not read again), so that every slab issues
  // the same number of copies and the waits are compile-time.
  auto copy = [&](int j, int kt, uint32_t stage) {
    const bool is_x = j < CF::A_LOADS;
    const int jj = is_x ? j : j - CF::A_LOADS;
    const uint32_t dst = __builtin_amdgcn_readfirstlane(
        lds0 + stage * CF::SLAB + (is_x ? 0 : CF::A_BYTES) + (jj * CF::WAVES + wave) * 1024);
    if constexpr (COPIES == Copies::kFar) {
      // Rows past M repeat row M - 1.
      const int row = copy_row<CF>(jj, wave, lane);
      const int r = is_x ? min(row, rows - 1) : w_row(row);
      copy16_to_lds_far((is_x ? X : W) + static_cast<int64_t>(r) * ld +
                            far_k(kt, k0, range, copy_chunk(row, lane)),
                        dst);
    } else {
      const SlabCopy s = slab_copy<COPIES>(kt, k0, KT, is_x ? x_bytes : w_bytes,
                                           is_x ? xoff[is_x ? jj : 0] : woff[is_x ? 0 : jj]);
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<T*>(is_x ? X : W), static_cast<short>(0), static_cast<int>(s.bytes), 0x00020000);
      copy16_to_lds(rsrc, s.lane, __builtin_amdgcn_readfirstlane(s.scalar), dst);
    }
  };

  // Fragments of step u (0, 1) of a slab at LDS byte `base`: X rows wm*WM + 16i + c,
  // W rows wn*WN + 16i + c, chunk 4u + g.  Every address is a multiple of 16 bytes;
  // saying so keeps the reads single ds_read_b128 (the library is built with
  // unaligned LDS access off, where an unproven alignment becomes byte reads).
  const int swz = slab_swizzle(c);
  const int chunk[2] = {(g ^ swz) * 16, ((4 + g) ^ swz) * 16};
  const int xrow = (wm * CF::WM + c) * (kSlabK * 2);
  const int wrow = CF::A_BYTES + (wn * CF::WN + c) * (kSlabK * 2);
  auto x_frag = [&](uint32_t base, int u, int i) {
    return *static_cast<const F*>(
        __builtin_assume_aligned(smem + base + xrow + chunk[u] + i * 16 * kSlabK * 2, 16));
  };
  auto w_frag = [&](uint32_t base, int u, int i) {
    return *static_cast<const F*>(
        __builtin_assume_aligned(smem + base + wrow + chunk[u] + i * 16 * kSlabK * 2, 16));
  };

  f32x4_t acc[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  F xf[2][MB], wf[2][NB];

#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int j = 0; j < CF::LOADS; ++j) copy(j, s, s);
  wait_vmem<(S - 1) * CF::LOADS>();  // slab 0
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int i = 0; i < NB; ++i) wf[0][i] = w_frag(0, 0, i);
#pragma unroll
  for (int i = 0; i < MB; ++i) xf[0][i] = x_frag(0, 0, i);

  // MFMAs of register set P, meanwhile the fragments of the next step (set P ^ 1,
  // step P ^ 1 of the slab at `base`) and, with COPY, the copies of slab `kt`.
  auto step = [&](auto parity, auto with_copies, uint32_t base, int kt, uint32_t stage) {
    constexpr int P = decltype(parity)::value;
    constexpr bool COPY = decltype(with_copies)::value;
#pragma unroll
    for (int q = 0; q < kMfmas; ++q) {
      __builtin_amdgcn_sched_barrier(0);
      acc[q % NB][q / NB] = M::run(wf[P][q % NB], xf[P][q / NB], acc[q % NB][q / NB]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int z = 0; z < kReads; ++z)
        if (z * kMfmas * 3 / 4 / kReads == q) {
          if (z < NB) {
            wf[P ^ 1][z] = w_frag(base, P ^ 1, z);
          } else {
            xf[P ^ 1][z - NB] = x_frag(base, P ^ 1, z - NB);
          }
        }
      if constexpr (COPY) {
#pragma unroll
        for (int z = 0; z < CF::LOADS; ++z)
          if (z * kMfmas * 3 / 4 / CF::LOADS == q) copy(z, kt, stage);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  uint32_t stage = 0;  // of slab kt
  for (int kt = 0; kt < KT; ++kt) {
    const uint32_t next = stage + 1 == S ? 0 : stage + 1;
    step(std::integral_constant<int, 0>{}, std::false_type{}, stage * CF::SLAB, 0, 0);
    wait_vmem<(S - 2) * CF::LOADS>();  // this wavefront's copies of slab kt + 1
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // (A last half slab has no second step.)
    if (kt * kSlabK + kStepK < K)
      step(std::integral_constant<int, 1>{}, std::true_type{}, next * CF::SLAB, kt + S, stage);
    stage = next;
  }

  if constexpr (EPI == kEpiPartial) {
    float* part = reinterpret_cast<float*>(a.y) + static_cast<int64_t>(split) * a.M * a.N;
#pragma unroll
    for (int j = 0; j < MB; ++j) {
      const int m = m_base + wm * CF::WM + 16 * j + c;
      if (m >= a.M) continue;
      float* row = part + static_cast<int64_t>(m) * a.N + n_base + wn * CF::WN + 8 * g;
#pragma unroll
      for (int i = 0; i < NB; ++i)
        *reinterpret_cast<f32x4_t*>(row + 16 * (i & ~1) + 4 * (i & 1)) = acc[i][j];
    }
    wait_vmem<0>();
    return;
  }
  // ---- epilogue: bias, rounding to T (nn.Linear's output), GELU or residual;
  // eight consecutive outputs of a row per lane and block pair ----
  typedef T Oct __attribute__((ext_vector_type(8)));
  const T* bias = reinterpret_cast<const T*>(a.bias);
  const T* res = reinterpret_cast<const T*>(a.residual);
  T* Y = reinterpret_cast<T*>(a.y);
  Quad<T> bq[NB];  // bias of the four outputs of block i
#pragma unroll
  for (int i = 0; i < NB; ++i)
    bq[i] = *reinterpret_cast<const Quad<T>*>(bias + n_base + wn * CF::WN + 16 * (i & ~1) + 8 * g +
                                              4 * (i & 1));
  const int64_t y_base = static_cast<int64_t>(m_base) * a.N;
  const auto yr = __builtin_amdgcn_make_buffer_rsrc(Y + y_base, static_cast<short>(0), 0x7fffffff,
                                                    0x00020000);
  // Row block by row block, so that the stores to the two halves of a 128-byte
  // line follow each other.
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    const int m = m_base + wm * CF::WM + 16 * j + c;
    const int64_t row = static_cast<int64_t>(m) * a.N + n_base + wn * CF::WN + 8 * g;
#pragma unroll
    for (int i = 0; i < NB; i += 2) {
      Oct out;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const T lin = static_cast<T>(acc[i + (e >> 2)][j][e & 3] +
                                     static_cast<float>(bq[i + (e >> 2)][e & 3]));
        if constexpr (EPI == kEpiBiasGelu) {
          out[e] = static_cast<T>(gelu_erf<T>(static_cast<float>(lin)));
        } else {
          out[e] = lin;
        }
      }
      if (m >= a.M) continue;
      if constexpr (EPI == kEpiBiasAdd) {
        const Oct rv = *reinterpret_cast<const Oct*>(res + row + 16 * i);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          out[e] = static_cast<T>(static_cast<float>(out[e]) + static_cast<float>(rv[e]));
      }
      if (a.through) {
        store_through(yr, static_cast<uint32_t>(row + 16 * i - y_base) * 2u,
                      __builtin_bit_cast(u32x4_t, out));
      } else {
        *reinterpret_cast<Oct*>(Y + row + 16 * i) = out;
      }
    }
  }
  wait_vmem<0>();  // no copy may land in LDS after the workgroup has ended
}

namespace {

// CUs of the current device (cached per device; 256 if it cannot be read).
int gemm_device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 256;
  if (dev < 64) {
    const int known = cache[dev].load(std::memory_order_relaxed);
    if (known > 0) return known;
  }
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    cus = 256;
  if (dev < 64) cache[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

template <typename T, int EPI, typename CF, Copies COPIES>
int launch_copies(GemmArgs args, hipStream_t stream) {
  constexpr auto* kernel = &gemm_kernel<T, EPI, CF, COPIES>;
  // The dynamic LDS limit is raised once per device (the attribute persists).
  static std::atomic<uint64_t> raised{0};
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return static_cast<int>(err);
  const uint64_t bit = dev < 64 ? (uint64_t{1} << dev) : 0;
  if (bit == 0 || (raised.load(std::memory_order_acquire) & bit) == 0) {
    err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, CF::LDS);
    if (err == hipSuccess && bit != 0) raised.fetch_or(bit, std::memory_order_release);
  }
  if (err != hipSuccess) return static_cast<int>(err);
  args.m_blocks = (args.M + CF::BM - 1) / CF::BM;
  args.n_blocks = args.N / CF::BN;
  // Y through the L2 (against left in it: 12 layers of 4096 rows, 768 wide, Y of 6 to 24 MiB,
  // 1416 us against 1462, non-temporal 1508), except a plain output of 64 MiB and more: the
  // QKV output of one ragged 768-wide layer at 12288 rows (54 MiB) even, at 16384 (72
  // MiB) 2.3 % slower through it, as the attention reads it at once.  The FFN intermediate
  // gains at every size, us, left / through: 8192 rows (48 MiB) 214.1 / 207.5, 12288 (72
  // MiB) 316.0 / 305.1, 16384 (96 MiB) 380.2 / 370.5.
  args.through = args.N <= kMaxThroughN &&
                 (EPI == kEpiBiasGelu ||
                  static_cast<int64_t>(args.M) * args.N * 2 < (int64_t{64} << 20));
  // XCDs along the rows and the columns: the split with the fewest rows of X and W
  // for an XCD to read, among those whose largest range needs no more tiles than an
  // even share rounded up to whole rounds of its CUs.
  const int64_t tiles = static_cast<int64_t>(args.m_blocks) * args.n_blocks;
  const int64_t round = (gemm_device_cus() + 7) / 8 * CF::WGS;
  const int64_t rounds = ((tiles + 7) / 8 + round - 1) / round;
  int64_t best = 0;
  int64_t per_xcd = 0;
  for (int gm = 1; gm <= 8; gm *= 2) {
    const int gn = 8 / gm;
    const int64_t mt = (args.m_blocks + gm - 1) / gm;
    const int64_t nt = (args.n_blocks + gn - 1) / gn;
    const int64_t read = mt * CF::BM + nt * CF::BN;
    const bool even = (mt * nt + round - 1) / round <= rounds;
    const int64_t score = read + (even ? 0 : (int64_t{1} << 40) + mt * nt);
    if (best == 0 || score < best) {
      best = score;
      per_xcd = mt * nt;
      args.xcds_m = gm;
    }
  }
  const int64_t grid = 8 * per_xcd * args.splits;
  if (grid > 0x7fffffff) return DFLASH_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(CF::THREADS), CF::LDS,
                     stream, args);
  return static_cast<int>(hipGetLastError());
}

template <typename T, int EPI, typename CF>
int launch_gemm(const GemmArgs& args, hipStream_t stream) {
  return args.K % kSlabK == 0 ? launch_copies<T, EPI, CF, Copies::kWhole>(args, stream)
                              : launch_copies<T, EPI, CF, Copies::kHalf>(args, stream);
}

// Time of a launch in microseconds on a tile configuration, from its tiles and
// its K:
//   rounds of CUs * WGS tiles, each fixed + slabs * slab time; the slab time of a
//   round with n tiles is slab1 + slab1_load * n / CUs while every CU has at most
//   one tile, and reaches slab_full with WGS tiles on a CU; gelu: the GELU epilogue.
// The constants are a least-squares fit (in the logarithm) to timings of every
// configuration at K and N of 768- and 1536-wide layers (all four projections) and M = 16 ..
// 16384 (HIP graphs of back-to-back calls over weights and activations that change from call
// to call, fp16).  bench.py --gemm-table times such a set: taking the configuration with the
// smallest modelled time was 0.6-0.9 % slower on average than taking the fastest one of
// each shape, and at most 12-14 % (80 shapes, two chips;
// profiles/gemm_projection_device_times.md).  The CUs are those of the device; the
// constants are an MI355X's.
struct GemmCost {
  float fixed, slab1, slab1_load, slab_full, gelu;
};

template <typename CF>
float gemm_cost(const GemmArgs& a, bool gelu, const GemmCost& c, int cus) {
  const int64_t tiles =
      static_cast<int64_t>((a.M + CF::BM - 1) / CF::BM) * (a.N / CF::BN) * a.splits;
  const int64_t cap = static_cast<int64_t>(cus) * CF::WGS;
  const int all_slabs = (a.K + kSlabK - 1) / kSlabK;
  const float slabs = static_cast<float>((all_slabs + a.splits - 1) / a.splits);
  auto round = [&](int64_t n) {
    const int64_t per_cu = (n + cus - 1) / cus;
    float slab = c.slab1 + c.slab1_load * static_cast<float>(n < cus ? n : cus) / cus;
    if constexpr (CF::WGS > 1)
      slab += (c.slab_full - slab) * static_cast<float>(per_cu - 1) / (CF::WGS - 1);
    return c.fixed + slabs * slab + (gelu ? c.gelu * per_cu / CF::WGS : 0.0f);
  };
  const int64_t full = tiles / cap;
  const int64_t rest = tiles - full * cap;
  return (full > 0 ? static_cast<float>(full) * round(cap) : 0.0f) + (rest > 0 ? round(rest) : 0.0f);
}

// The configuration with the smallest modelled time; with splits > 1 among the ones
// built for partial sums.
int best_config(const GemmArgs& args, bool gelu, float* us) {
  const int cus = gemm_device_cus();
  int config = 0;
  auto consider = [&](int number, auto cf, const GemmCost& cost) {
    if (args.N % decltype(cf)::BN != 0) return;
    const float t = gemm_cost<decltype(cf)>(args, gelu, cost, cus);
    if (config == 0 || t < *us) {
      config = number;
      *us = t;
    }
  };
  if (args.splits == 1) {
    consider(1, Cfg128x192{}, {3.72f, 0.684f, 0.175f, 1.339f, 3.54f});
    consider(2, Cfg128x128{}, {3.15f, 0.580f, 0.193f, 0.879f, 2.41f});
    consider(3, Cfg256x192{}, {5.39f, 0.832f, 0.390f, 0.0f, 2.99f});
    consider(4, Cfg64x128{}, {3.27f, 0.298f, 0.028f, 0.571f, 1.07f});
    consider(5, Cfg64x64{}, {3.89f, 0.386f, 0.0f, 0.619f, 0.98f});
    consider(6, Cfg256x256{}, {6.84f, 0.994f, 0.505f, 0.0f, 3.69f});
    consider(7, Cfg128x192Deep{}, {4.76f, 0.485f, 0.201f, 0.0f, 1.77f});
    consider(8, Cfg128x128Deep{}, {4.10f, 0.382f, 0.110f, 0.0f, 1.11f});
  }
  consider(9, Cfg128x64{}, {3.22f, 0.282f, 0.052f, 0.563f, 0.88f});
  consider(10, Cfg64x64Deep{}, {2.65f, 0.233f, 0.004f, 0.361f, 0.37f});
  consider(11, Cfg32x64{}, {2.12f, 0.212f, 0.0f, 0.266f, 0.22f});
  return config;
}

// config: 0 = automatic, else the number of a configuration.
template <typename T, int EPI>
int pick_config(const GemmArgs& args, int config, hipStream_t stream) {
  // A tile's rows must lie within 32-bit byte offsets of its first one (256 rows
  // of 2 K bytes); past that, 64 x 64 tiles with 64-bit copy addresses.
  const bool far = args.K >= (1 << 23);
  if (config == 0 && far) config = 5;
  if (config == 0) {
    float us = 0.0f;
    config = best_config(args, EPI == kEpiBiasGelu, &us);
  }
  auto fits = [&](auto cf) { return args.N % decltype(cf)::BN == 0; };
#define DFLASH_GEMM_CASE(NUM, CF)                                                \
  case NUM:                                                                      \
    if (!fits(CF{})) return DFLASH_ERR_SHAPE;                                    \
    if (far) return launch_copies<T, EPI, Cfg64x64, Copies::kFar>(args, stream); \
    return launch_gemm<T, EPI, CF>(args, stream);
  switch (config) {
    DFLASH_GEMM_CASE(1, Cfg128x192)
    DFLASH_GEMM_CASE(2, Cfg128x128)
    DFLASH_GEMM_CASE(3, Cfg256x192)
    DFLASH_GEMM_CASE(4, Cfg64x128)
    DFLASH_GEMM_CASE(5, Cfg64x64)
    DFLASH_GEMM_CASE(6, Cfg256x256)
    DFLASH_GEMM_CASE(7, Cfg128x192Deep)
    DFLASH_GEMM_CASE(8, Cfg128x128Deep)
    DFLASH_GEMM_CASE(9, Cfg128x64)
    DFLASH_GEMM_CASE(10, Cfg64x64Deep)
    DFLASH_GEMM_CASE(11, Cfg32x64)
    default:
      return DFLASH_ERR_SHAPE;
  }
#undef DFLASH_GEMM_CASE
}

template <typename T>
int dispatch_epilogue(const GemmArgs& args, int epilogue, int config, hipStream_t stream) {
  switch (epilogue) {
    case DFLASH_GEMM_BIAS:
      return pick_config<T, kEpiBias>(args, config, stream);
    case DFLASH_GEMM_BIAS_GELU:
      return pick_config<T, kEpiBiasGelu>(args, config, stream);
    case DFLASH_GEMM_BIAS_ADD:
      return pick_config<T, kEpiBiasAdd>(args, config, stream);
    default:
      return DFLASH_ERR_SHAPE;
  }
}

template <typename T>
int launch_partial(const GemmArgs& args, int config, hipStream_t stream) {
  switch (config) {
    case 9:
      return launch_gemm<T, kEpiPartial, Cfg128x64>(args, stream);
    case 10:
      return launch_gemm<T, kEpiPartial, Cfg64x64Deep>(args, stream);
    case 11:
      return launch_gemm<T, kEpiPartial, Cfg32x64>(args, stream);
    default:
      return DFLASH_ERR_SHAPE;
  }
}

constexpr int kMaxSplits = 8;

// Ranges of K (1, 2, 4 or 8) of an output block's projection, and the
// configuration for more than one.  With few rows the tiles leave most CUs idle and
// walk all of K one after the other; the LayerNorm reads every row anyway and adds
// the ranges' sums on the way.  Split where the modelled time, with the partial sums
// written and read at 4 MB a microsecond, is at least a microsecond less.  Projection and
// LayerNorm together, unsplit / split, us: 64 x 768 x 3072 15.5 / 8.9 (8 ranges),
// 512 x 768 x 3072 15.8 / 13.6 (2), 64 x 1536 x 6144 24.6 / 14.6 (8), 64 x 768 x 768 8.5 / 7.2
// (2); from 1024 rows none is split.
int output_splits(int M, int N, int K, int* config) {
  *config = 0;
  GemmArgs args{};
  args.M = M;
  args.N = N;
  args.K = K;
  args.splits = 1;
  float best = 0.0f;
  if (K >= (1 << 23) || best_config(args, false, &best) == 0) return 1;
  best -= 1.0f;
  int splits = 1;
  for (int s = 2; s <= kMaxSplits && K / s >= 4 * kSlabK; s *= 2) {
    args.splits = s;
    float us = 0.0f;
    const int number = best_config(args, false, &us);
    us += 8.0f * s * static_cast<float>(M) * static_cast<float>(N) / 4e6f;
    if (number != 0 && us < best) {
      best = us;
      splits = s;
      *config = number;
    }
  }
  return splits;
}

}  // namespace

}  // namespace dflash

using namespace dflash;

extern "C" int dflash_linear_fwd(const void* x, const void* weight, const void* bias,
                                 const void* residual, void* y, int M, int N, int K,
                                 int epilogue, int dtype, void* stream) {
  if (M < 0 || N < 1 || K < 1) return DFLASH_ERR_SHAPE;
  if (M == 0) return DFLASH_OK;
  if (!x || !weight || !bias || !y) return DFLASH_ERR_NULL;
  if ((epilogue & 0xff) == DFLASH_GEMM_BIAS_ADD && !residual) return DFLASH_ERR_NULL;
  if (N % 64 != 0 || K % kStepK != 0) return DFLASH_ERR_SHAPE;
  if (static_cast<int64_t>(M) * K >= (int64_t{1} << 31) ||
      static_cast<int64_t>(M) * N >= (int64_t{1} << 31))
    return DFLASH_ERR_TOO_LARGE;
  const uintptr_t addr_or = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) |
                            reinterpret_cast<uintptr_t>(y) |
                            reinterpret_cast<uintptr_t>(residual);
  if (addr_or % 16 != 0 || reinterpret_cast<uintptr_t>(bias) % 8 != 0) return DFLASH_ERR_ALIGN;
  // Bits 8.. of `epilogue` select a tile configuration (0 = automatic).
  const int config = epilogue >> 8;
  epilogue &= 0xff;
  GemmArgs args{x, weight, bias, residual, y, M, N, K, 0, 0, 0, 1, 1};
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == DFLASH_DTYPE_FP16) return dispatch_epilogue<_Float16>(args, epilogue, config, s);
  if (dtype == DFLASH_DTYPE_BF16) return dispatch_epilogue<__bf16>(args, epilogue, config, s);
  return DFLASH_ERR_DTYPE;
}

extern "C" size_t dflash_output_block_workspace_bytes(int M, int N, int K) {
  if (M < 1 || N < 1 || K < 1) return 0;
  int config = 0;
  const int splits = output_splits(M, N, K, &config);
  return static_cast<size_t>(M) * N * (splits > 1 ? sizeof(float) * splits : 2);
}

extern "C" int dflash_output_block_fwd(const void* x, const void* weight, const void* bias,
                                       const void* residual, const void* gamma, const void* beta,
                                       void* out, int M, int N, int K, float eps, int dtype,
                                       void* workspace, size_t workspace_bytes, void* stream) {
  if (M < 0 || N < 1 || K < 1) return DFLASH_ERR_SHAPE;
  if (M == 0) return DFLASH_OK;
  if (!residual || !workspace) return DFLASH_ERR_NULL;
  if (workspace_bytes < dflash_output_block_workspace_bytes(M, N, K)) return DFLASH_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return DFLASH_ERR_ALIGN;
  int config = 0;
  const int splits = output_splits(M, N, K, &config);
  if (splits == 1) {
    const int rc = dflash_linear_fwd(x, weight, bias, nullptr, workspace, M, N, K,
                                     DFLASH_GEMM_BIAS, dtype, stream);
    if (rc != DFLASH_OK) return rc;
    return dflash_add_layernorm_fwd(workspace, residual, gamma, beta, out, M, N, eps, dtype,
                                    stream);
  }
  if (!x || !weight || !bias || !gamma || !beta || !out) return DFLASH_ERR_NULL;
  if (N % 64 != 0 || K % kStepK != 0 || N > 4096) return DFLASH_ERR_SHAPE;
  if (dtype != DFLASH_DTYPE_FP16 && dtype != DFLASH_DTYPE_BF16) return DFLASH_ERR_DTYPE;
  if (static_cast<int64_t>(M) * K >= (int64_t{1} << 31)) return DFLASH_ERR_TOO_LARGE;
  const uintptr_t wide = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight);
  const uintptr_t quad = reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(residual) |
                         reinterpret_cast<uintptr_t>(gamma) | reinterpret_cast<uintptr_t>(beta) |
                         reinterpret_cast<uintptr_t>(out);
  if (wide % 16 != 0 || quad % 8 != 0) return DFLASH_ERR_ALIGN;
  GemmArgs args{x, weight, nullptr, nullptr, workspace, M, N, K, 0, 0, 0, splits, 1};
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int rc = dtype == DFLASH_DTYPE_FP16 ? launch_partial<_Float16>(args, config, s)
                                            : launch_partial<__bf16>(args, config, s);
  if (rc != DFLASH_OK) return rc;
  return launch_partials_layernorm(static_cast<const float*>(workspace), splits, bias, residual,
                                   gamma, beta, out, M, N, eps, dtype, s);
}

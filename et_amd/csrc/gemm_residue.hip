// FP64 products on the int8 matrix cores, exact modulo 16 coprime moduli
// (residue.hpp has the arithmetic and its error).
//
// The FP64 matrix cores reach 78 TFLOP/s on this chip and the FP64 kernels 62
// of them; the int8 products here run at 2.4-2.6 POP/s (the kernel's 2548 TOP/s
// on random bytes; 3491 on zeros, where the power limit does not bind), so 17 of them
// per FP64 product are worth up to 150 TFLOP/s (with the product of 8-bit floats, whose
// instruction has half the k, 2.2 POP/s and 130 in a residual).  A product runs as
//   1. row norms of op(A) and op(B)^T            (reads each operand once)
//   2. residue packs: 17 bytes per element, in the order the matrix cores read
//      (a byte per modulus, and the magnitude)
//   3. 16 int8 products, each sum reduced to one byte per output, and before
//      them the product of the magnitudes, which flags the 64 x 64 blocks that
//      need the FP64 kernel
//   4. reconstruction of C from its 16 bytes     (writes C once)
//   5. the flagged blocks on the FP64 kernel
// on panels of A and B whose packs fit a bounded workspace.
#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>

#include "gemm.hpp"
#include "kernels.hpp"
#include "residue.hpp"
#include "tile_map.hpp"

namespace etg {
namespace {

using residue::kC;
using residue::kModuli;

typedef int i4 __attribute__((ext_vector_type(4)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kDepth = 64;                    // k per step (one MFMA step)
constexpr int kPlanes = kModuli + 1;          // of a pack: the residues and the magnitudes

// ---------------------------------------------------------------------------
// 1. Scale exponents.  Element (r, k) of the rows x K operand is X[k + r ld]
// (kcontig) or X[r + k ld].  Bound by HBM: each operand is read once.
// ---------------------------------------------------------------------------

// One workgroup per row.
__global__ __launch_bounds__(256) void row_exponents_kcontig_kernel(const double* __restrict__ X, int64_t ld,
                                                                    int64_t strideX, int64_t K,
                                                                    int64_t exp_stride, int* __restrict__ e,
                                                                    float* __restrict__ nrm) {
  __shared__ double ss[4];
  __shared__ unsigned long long mm[4];
  const int64_t r = blockIdx.x, bz = blockIdx.y;
  const double* x = X + bz * strideX + r * ld;
  double s = 0.0;
  unsigned long long mx = 0;
#pragma unroll 4
  for (int64_t k = threadIdx.x; k < K; k += 256) {
    const double v = x[k];
    s += v * v;
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v) & 0x7fffffffffffffffull;
    mx = b > mx ? b : mx;
  }
  for (int off = 32; off > 0; off >>= 1) {
    s += __shfl_xor(s, off, 64);
    const unsigned long long o = __shfl_xor(mx, off, 64);
    mx = o > mx ? o : mx;
  }
  if ((threadIdx.x & 63) == 0) {
    ss[threadIdx.x >> 6] = s;
    mm[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < 4; ++q) {
      s += ss[q];
      mx = mm[q] > mx ? mm[q] : mx;
    }
    e[bz * exp_stride + r] = residue::scale_exponent(s, mx, K);
    nrm[bz * exp_stride + r] = residue::scaled_norm(s, mx);
  }
}

// 64 rows per workgroup (lanes along the contiguous rows), four k at a time, over
// one of gridDim.y ranges of k; partial sums per range.
__global__ __launch_bounds__(256) void row_norms_partial_kernel(const double* __restrict__ X, int64_t ld,
                                                                int64_t strideX, int64_t rows, int64_t K,
                                                                int64_t k_per, double* __restrict__ ps,
                                                                unsigned long long* __restrict__ pm) {
  __shared__ double ss[4][64];
  __shared__ unsigned long long mm[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t r = int64_t(blockIdx.x) * 64 + lane, bz = blockIdx.z;
  const int64_t k0 = int64_t(blockIdx.y) * k_per, k1 = min(K, k0 + k_per);
  const double* x = X + bz * strideX + r;
  double s = 0.0;
  unsigned long long mx = 0;
  if (r < rows) {
#pragma unroll 4
    for (int64_t k = k0 + w; k < k1; k += 4) {
      const double v = x[k * ld];
      s += v * v;
      const unsigned long long b = __builtin_bit_cast(unsigned long long, v) & 0x7fffffffffffffffull;
      mx = b > mx ? b : mx;
    }
  }
  ss[w][lane] = s;
  mm[w][lane] = mx;
  __syncthreads();
  if (w == 0 && r < rows) {
    for (int q = 1; q < 4; ++q) {
      s += ss[q][lane];
      mx = mm[q][lane] > mx ? mm[q][lane] : mx;
    }
    const int64_t at = (bz * gridDim.y + blockIdx.y) * rows + r;
    ps[at] = s;
    pm[at] = mx;
  }
}

__global__ __launch_bounds__(256) void row_exponents_finish_kernel(const double* __restrict__ ps,
                                                                   const unsigned long long* __restrict__ pm,
                                                                   int64_t rows, int parts, int64_t K,
                                                                   int64_t exp_stride, int* __restrict__ e,
                                                                    float* __restrict__ nrm) {
  const int64_t r = int64_t(blockIdx.x) * 256 + threadIdx.x, bz = blockIdx.y;
  if (r >= rows) return;
  double s = 0.0;
  unsigned long long mx = 0;
  for (int q = 0; q < parts; ++q) {
    const int64_t at = (bz * parts + q) * rows + r;
    s += ps[at];
    mx = pm[at] > mx ? pm[at] : mx;
  }
  e[bz * exp_stride + r] = residue::scale_exponent(s, mx, K);
  nrm[bz * exp_stride + r] = residue::scaled_norm(s, mx);
}

// ---------------------------------------------------------------------------
// 2. Residue packs.  Per modulus one plane of 1 KB chunks (16 rows x 64 k: lane
// l holds 16 consecutive k of row l % 16 from 16 (l / 16) on), row blocks
// outermost, k steps contiguous.  One wave forms the 17 chunks of a (row block,
// k step).  Some 90 VALU operations per element (four per modulus, and the bytes'
// packing) against 8 bytes read and 17 written: bound by HBM, 37 M elements in
// 154 us (6.0 TB/s).
// ---------------------------------------------------------------------------
// The 16 values are formed here, in the order of the source, not where they are used.
__device__ inline void pin(uint32_t (&x)[16]) {
#pragma unroll
  for (int j = 0; j < 16; ++j) asm volatile("" : "+v"(x[j]));
  __builtin_amdgcn_sched_barrier(0);
}

// The low bytes of 16 words.
__device__ inline u4 pack_bytes(const uint32_t (&x)[16]) {
  u4 w;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t p01 = __builtin_amdgcn_perm(x[4 * q + 1], x[4 * q], 0x0c0c0400u);
    const uint32_t p23 = __builtin_amdgcn_perm(x[4 * q + 3], x[4 * q + 2], 0x0c0c0400u);
    w[q] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
  }
  return w;
}

constexpr int kPackLd = kDepth + 2;           // LDS row of a staged chunk (doubles)

__global__ __launch_bounds__(256) void residue_pack_kernel(const double* __restrict__ X, int64_t ld, int64_t strideX,
                                                           int kcontig, int64_t rows, int64_t K, int64_t KS,
                                                           int64_t plane, const int* __restrict__ e,
                                                           int64_t exp_stride, u4* __restrict__ P,
                                                           int* __restrict__ flags, int64_t n_flags) {
  __shared__ __attribute__((aligned(16))) double stage[4][16 * kPackLd];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t ks = int64_t(blockIdx.x) * 4 + wave;
  const int64_t rb = blockIdx.y, bz = blockIdx.z;
  const int64_t r = rb * 16 + (lane & 15), k0 = ks * kDepth + 16 * (lane >> 4);
  const int ex = r < rows ? e[bz * exp_stride + r] : 0;
  // the products' flags, cleared on the way
  for (int64_t f = ((bz * gridDim.y + rb) * gridDim.x + blockIdx.x) * 256 + threadIdx.x; f < n_flags;
       f += int64_t(gridDim.x) * gridDim.y * gridDim.z * 256)
    flags[f] = 0;
  uint32_t lo[16], hi[16];
  if (kcontig) {
    // whole rows of the chunk (512 contiguous bytes per load) through LDS: read by
    // each lane from global memory, 64 rows' lines per load, the pack took 2.7 times
    // as long (6912 x 14400: 1150 us)
    const double* x = X + bz * strideX + rb * 16 * ld;
    const int64_t kl = ks * kDepth + lane;
    double* t = stage[wave];
    // (loads at clamped indices: under a condition each would wait for the one before it;
    // with those the products of 17020 x 820 x 17020 took 4.89 -> 4.55 ms)
    const int64_t last = rows - 1 - rb * 16, kc = min(kl, K - 1);
    double v[16];
#pragma unroll
    for (int rr = 0; rr < 16; ++rr) v[rr] = x[min(int64_t(rr), last) * ld + kc];
#pragma unroll
    for (int rr = 0; rr < 16; ++rr) t[rr * kPackLd + lane] = (rr <= last && kl < K) ? v[rr] : 0.0;
    __syncthreads();
    const double2* src = reinterpret_cast<const double2*>(&t[(lane & 15) * kPackLd + 16 * (lane >> 4)]);
    const bool ok = ex != residue::kNotFinite;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const double2 v = src[j];
      residue::to_integer(ok ? v.x : 0.0, ex, lo[2 * j], hi[2 * j]);
      residue::to_integer(ok ? v.y : 0.0, ex, lo[2 * j + 1], hi[2 * j + 1]);
    }
  } else {
    const double* x = X + bz * strideX + min(r, rows - 1) + min(k0, K - 1) * ld;
    const int n = (r < rows && ex != residue::kNotFinite && k0 < K) ? int(min<int64_t>(16, K - k0)) : 0;
    const int64_t last = max(int64_t(0), K - 1 - k0);
    double v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = x[min(int64_t(j), last) * ld];
#pragma unroll
    for (int j = 0; j < 16; ++j) residue::to_integer(j < n ? v[j] : 0.0, ex, lo[j], hi[j]);
  }
  if (ks >= KS) return;
  u4* dst = P + bz * kPlanes * plane + (rb * KS + ks) * 64 + lane;
#pragma unroll
  for (int i = 0; i < kModuli; ++i) {
    // residue_byte of the 16 elements side by side: a byte dot product's result can
    // be read three operations later, and the compiler would wait that out each time
    uint32_t x[16];
    if (residue::kMod[i] == 256) {
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = lo[j];
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = residue::byte_dot(lo[j], kC.low[i], kC.offset[i]);
      pin(x);
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = residue::byte_dot(hi[j], kC.high[i], x[j]);
      pin(x);
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = residue::low_byte(x[j], kC.invf[i], kC.c[i]);
    }
    dst[i * plane] = pack_bytes(x);
  }
  uint32_t q[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) q[j] = residue::magnitude_byte(hi[j]);
  dst[kModuli * plane] = pack_bytes(q);
}

// ---------------------------------------------------------------------------
// 3. The int8 products.  Waves in 2 x WN, each 128 x 64 of the output (8 x 4
// blocks, 128 int32 accumulators per lane): tiles of 256 x 128 (WN = 2, two
// workgroups per CU, three LDS stages) or 256 x 256 (WN = 4, one, four stages).
// Steps of 64 k (1 KB chunks) go from global memory straight into an LDS stage,
// kStages - 1 steps ahead of their use; a wave waits for its own copies of the
// step by count, then one barrier makes everyone's visible and frees the stage
// read in the step before.  A step is 32 MFMAs (512 cycles) per wave against 12
// KB of LDS reads.  Two workgroups per CU hide barriers, the first copies and the
// byte epilogue under each other's products, but drift apart along k until their
// tiles no longer meet in the L2: TOP/s with 15 planes of random bytes for
//   m = n = 6912, k =    1600    3200    14400   28800      m = n = k = 1536
//   256 x 128            2360    2400     1780    1990                  1790
//   256 x 256            2170    2440     2560    2480                  1470
// so depths up to kShortDepth take the small tile.  Four waves of 128 x 128
// reached 1890-2240 (one wave per SIMD), 128 x 128 tiles 2200 (LDS reads).
// blockIdx.y is the modulus, blockIdx.z the batch entry.
// ---------------------------------------------------------------------------
constexpr int64_t kShortDepth = 3200;

constexpr int kWaveM = 8, kWaveN = 4;         // 16 x 16 blocks of a wave
constexpr int kBlocksM = kTileM / 16;

struct Params {
  const u4 *A, *B;                 // packs (planes of the first modulus)
  uint32_t* R;                     // one byte per output and modulus: tiles of 16 x 16 blocks in fragment order
  int64_t KS;
  int64_t planeA, planeB, planeR;  // from one modulus to the next (u4, u4, u32 units)
  int64_t strideA, strideB, strideR;   // from one batch entry to the next
  TileMap tiles;
  // per tile the 64 x 64 blocks that are left to the FP64 kernel (bit: row block + 4 column
  // block): zero before the launch, set by the product of the magnitudes
  int* flags;
  int64_t strideF;
  // of the guard product
  int64_t m, n;
  const float *na, *nb;            // norms of the rows
  int64_t na_stride, nb_stride;
};

// Waits until at most N of this wave's vector-memory operations are outstanding.
template <int N>
__device__ inline void wait_copies() {
  __builtin_amdgcn_s_waitcnt((N & 0xf) | 0x70 | 0xf00 | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// 16 x 16 sums of products of 8-bit floats (5 exponent bits), half h of a chunk's k.
__device__ inline i4 mfma_magnitudes(i4 a, i4 b, int h, i4 c) {
  typedef int i2 __attribute__((ext_vector_type(2)));
  const i2 ah = h ? i2{a[2], a[3]} : i2{a[0], a[1]}, bh = h ? i2{b[2], b[3]} : i2{b[0], b[1]};
  return __builtin_bit_cast(i4, __builtin_amdgcn_mfma_f32_16x16x32_bf8_bf8(__builtin_bit_cast(long, ah), __builtin_bit_cast(long, bh),
                                                                          __builtin_bit_cast(f4, c), 0, 0, 0));
}

// blockIdx.y = 0: the product of the magnitudes, which flags the blocks with an output
// below the threshold or with a row that is not finite.  It comes first, and a product
// that finds its blocks flagged already has nothing to do; one that started before gives
// residues that nobody reads.  (A launch of its own left CUs idle: 820 x 17020 x 17020
// 6.19 ms with 15 moduli, 5.43 in one.)
template <int WN, int kStages>
__global__ __launch_bounds__(128 * WN, WN == 2 ? 2 : 1) void residue_product_kernel(Params p) {
  constexpr int kBlocksN = WN * kWaveN;
  constexpr int kCopiesA = kBlocksM / (2 * WN), kCopiesB = kBlocksN / (2 * WN);   // chunks a wave copies per step
  __shared__ u4 lds[kStages][(kBlocksM + kBlocksN) * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int slot = slot_of(blockIdx.x, gridDim.x);
  int tile_m, tile_n;
  if (!tile_of(p.tiles, slot, tile_m, tile_n)) return;
  const bool guard = blockIdx.y == 0;
  const int z = guard ? kModuli : int(blockIdx.y) - 1;
  const int64_t bz = blockIdx.z;
  int* flags = p.flags + bz * p.strideF + slot;
  constexpr int kAllBlocks = (1 << (4 * WN)) - 1;
  if (!guard && __builtin_amdgcn_readfirstlane(__hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == kAllBlocks)
    return;
  const u4* sa = p.A + bz * p.strideA + z * p.planeA + int64_t(tile_m) * kBlocksM * p.KS * 64;
  const u4* sb = p.B + bz * p.strideB + z * p.planeB + int64_t(tile_n) * kBlocksN * p.KS * 64;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<u4*>(sa), (short)0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<u4*>(sb), (short)0, 0x7fffffff, 0x00020000);
  const uint32_t row_bytes = uint32_t(p.KS) * 1024u;     // one row block of a plane (at most 2 MB)
  auto load = [&](int stage, int64_t s) {
    const uint32_t voff = uint32_t(s) * 1024u + uint32_t(lane) * 16u;
#pragma unroll
    for (int q = 0; q < kCopiesA; ++q) {
      const int c = wave * kCopiesA + q;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void*)(&lds[stage][c * 64]), 16, voff,
                                               uint32_t(c) * row_bytes, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < kCopiesB; ++q) {
      const int c = wave * kCopiesB + q;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void*)(&lds[stage][(kBlocksM + c) * 64]), 16, voff,
                                               uint32_t(c) * row_bytes, 0, 0);
    }
  };
  i4 acc[kWaveM][kWaveN];
#pragma unroll
  for (int i = 0; i < kWaveM; ++i)
#pragma unroll
    for (int j = 0; j < kWaveN; ++j) acc[i][j] = i4{0, 0, 0, 0};
  // the four B fragments, then each row block's products with the next block's A
  // fragment read ahead of them (order pinned by the scheduling groups); the magnitudes'
  // 64 k are two products of 32 k, sums in FP32
  auto compute = [&](int stage, auto magnitudes) {
    const u4* As = &lds[stage][wm * kWaveM * 64];
    const u4* Bs = &lds[stage][(kBlocksM + wn * kWaveN) * 64];
    i4 a[2], b[kWaveN];
    a[0] = __builtin_bit_cast(i4, As[lane]);
#pragma unroll
    for (int j = 0; j < kWaveN; ++j) b[j] = __builtin_bit_cast(i4, Bs[j * 64 + lane]);
#pragma unroll
    for (int i = 0; i < kWaveM; ++i) {
      if (i + 1 < kWaveM) a[(i + 1) & 1] = __builtin_bit_cast(i4, As[(i + 1) * 64 + lane]);
      if constexpr (magnitudes) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < kWaveN; ++j) acc[i][j] = mfma_magnitudes(a[i & 1], b[j], h, acc[i][j]);
      } else {
#pragma unroll
        for (int j = 0; j < kWaveN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i & 1], b[j], acc[i][j], 0, 0, 0);
      }
      if (i == 0) __builtin_amdgcn_sched_group_barrier(0x100, kWaveN + 2, 0);
      else if (i + 1 < kWaveM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, magnitudes ? 2 * kWaveN : kWaveN, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  const int64_t ns = p.KS;
#pragma unroll
  for (int s = 0; s < kStages - 1; ++s)
    if (s < ns) load(s, s);
  auto steps = [&](auto magnitudes) {
    int stage = 0;
    int64_t s = 0;
    for (; s + kStages - 1 < ns; ++s) {
      wait_copies<(kStages - 2) * (kCopiesA + kCopiesB)>();
      load(stage == 0 ? kStages - 1 : stage - 1, s + kStages - 1);
      compute(stage, magnitudes);
      stage = stage + 1 == kStages ? 0 : stage + 1;
    }
    for (; s < ns; ++s) {
      wait_copies<0>();
      compute(stage, magnitudes);
      stage = stage + 1 == kStages ? 0 : stage + 1;
    }
  };
  if (!guard) steps(std::false_type{});
  if (guard) {
    steps(std::true_type{});
    // (in the copies' LDS: beside a second array the compiler waits for every copy in
    // flight before each read of a stage, 1.7 times the kernel's time)
    int* found = reinterpret_cast<int*>(&lds[0][0]);
    __syncthreads();
    const int64_t row0 = int64_t(tile_m) * kTileM + wm * (kWaveM * 16) + 4 * (lane >> 4);
    const int64_t col0 = (int64_t(tile_n) * kBlocksN + wn * kWaveN) * 16 + (lane & 15);
    // (norms of rows past the edge: inside the padded array, not used)
    const f4* na = reinterpret_cast<const f4*>(p.na + bz * p.na_stride + row0);
    const float* nb = p.nb + bz * p.nb_stride + col0;
    f4 nr[kWaveM];
#pragma unroll
    for (int i = 0; i < kWaveM; ++i) nr[i] = na[i * 4];
    bool lost[2] = {false, false};             // the wave's two blocks
#pragma unroll
    for (int j = 0; j < kWaveN; ++j) {
      const float nc = col0 + j * 16 < p.n ? nb[j * 16] : residue::kZeroNorm;
#pragma unroll
      for (int i = 0; i < kWaveM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int bits = acc[i][j][r];       // (bit_cast of the element itself takes the first one)
          lost[i / 4] |= row0 + i * 16 + r < p.m && nr[i][r] > 0.0f && nc > 0.0f &&
                         !(__builtin_bit_cast(float, bits) >= residue::kThreshold * fmaxf(nr[i][r], nc));
        }
    }
    static_assert(kWaveM == 8 && kWaveN == 4, "two 64 x 64 blocks of a wave");
    int mine = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {              // blocks past the edge have nothing to do
      const bool past = int64_t(tile_m) * kTileM + (wm * 2 + h) * 64 >= p.m || (int64_t(tile_n) * WN + wn) * 64 >= p.n;
      if (past || __ballot(lost[h]) != 0) mine |= 1 << (wm * 2 + h + 4 * wn);
    }
    if (lane == 0) found[wave] = mine;
    __syncthreads();
    if (tid == 0) {
      int all = 0;
#pragma unroll
      for (int w = 0; w < 2 * WN; ++w) all |= found[w];
      __hip_atomic_store(flags, all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return;
  }
  const double m = kC.md[z], inv = kC.invd[z];
  uint32_t* R = p.R + bz * p.strideR + z * p.planeR +
                int64_t(slot) * (kBlocksM * kBlocksN * 64);
#pragma unroll
  for (int i = 0; i < kWaveM; ++i)
#pragma unroll
    for (int j = 0; j < kWaveN; ++j) {
      uint32_t b[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = residue::residue_byte_of_sum(acc[i][j][r], m, inv);
      const uint32_t p01 = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);
      const uint32_t p23 = __builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u);
      R[((wn * kWaveN + j) * kBlocksM + wm * kWaveM + i) * 64 + lane] =
          __builtin_amdgcn_perm(p23, p01, 0x05040100u);
    }
}

// ---------------------------------------------------------------------------
// 4. Reconstruction: C = alpha op(A) op(B) + beta C from the 16 bytes of each
// output.  A lane takes the four rows of one column that its word of each plane
// holds.  Bound by HBM (16 bytes read, 8 written, 8 more read with beta).
// Flagged blocks are the FP64 kernel's (gemm_flagged_blocks).
// ---------------------------------------------------------------------------
struct Output {
  const uint32_t* R;
  int64_t planeR, strideR;
  TileMap tiles;
  int64_t m, n, K;                        // of this panel
  const int *ea, *eb;
  int64_t ea_stride, eb_stride;
  double alpha, beta;
  double* C;
  int64_t ldc, strideC;
  int vec_rows;                           // rows written four at a time (alignment checked on the host)
  const int* flags;                       // as in Params
  int64_t strideF;
};

__global__ __launch_bounds__(256) void residue_reconstruct_kernel(Output p) {
  const int lane = threadIdx.x & 63;
  const int blocks_n = p.tiles.tile_n / 16;
  const int per_tile = kBlocksM * blocks_n / 4;
  const int slot = int(blockIdx.x / unsigned(per_tile));
  const int blk = int(blockIdx.x % unsigned(per_tile)) * 4 + int(threadIdx.x >> 6);
  int tile_m, tile_n;
  if (!tile_of(p.tiles, slot, tile_m, tile_n)) return;
  const int64_t bz = blockIdx.y;
  if (p.flags[bz * p.strideF + slot] >> ((blk % kBlocksM) / 4 + blk / kBlocksM / 4 * 4) & 1) return;
  const int64_t row = int64_t(tile_m) * kTileM + (blk % kBlocksM) * 16 + 4 * (lane >> 4);
  const int64_t col = (int64_t(tile_n) * blocks_n + blk / kBlocksM) * 16 + (lane & 15);
  if (row >= p.m || col >= p.n) return;
  const uint32_t* R = p.R + bz * p.strideR + (int64_t(slot) * (kBlocksM * blocks_n) + blk) * 64 + lane;
  uint32_t w[kModuli];
#pragma unroll
  for (int i = 0; i < kModuli; ++i) w[i] = R[i * p.planeR];
  const int eb = p.eb[bz * p.eb_stride + col];
  const int* ea = p.ea + bz * p.ea_stride + row;
  const int rows = int(min<int64_t>(4, p.m - row));
  double v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    double hi = 0.0, lo = 0.0;
#pragma unroll
    for (int i = 0; i < kModuli; ++i) {
      const double b = double(int(w[i] << (24 - 8 * r)) >> 24);
      hi = fma(b, kC.fhi[i], hi);
      lo = fma(b, kC.flo[i], lo);
    }
    v[r] = r < rows ? residue::reconstruct(hi, lo, ea[r], eb) : 0.0;
  }
  double* c = p.C + bz * p.strideC + row + col * p.ldc;
  if (p.vec_rows) {
    double2* c2 = reinterpret_cast<double2*>(c);
    double2 x = {p.alpha * v[0], p.alpha * v[1]}, y = {p.alpha * v[2], p.alpha * v[3]};
    if (p.beta != 0.0) {
      const double2 o0 = c2[0], o1 = c2[1];
      x.x += p.beta * o0.x; x.y += p.beta * o0.y;
      y.x += p.beta * o1.x; y.y += p.beta * o1.y;
    }
    c2[0] = x;
    c2[1] = y;
    return;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (r < rows) c[r] = p.beta == 0.0 ? p.alpha * v[r] : p.alpha * v[r] + p.beta * c[r];
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct Panels {
  int64_t KS, rows_m, rows_n, batch;          // panel rows of op(A) and op(B)^T, batch entries per group
  int64_t out_m, out_n;                       // outputs of a panel taken at once (their residues)
  int tile_n;                                 // columns of a tile
  bool same;                                  // op(A)^T and op(B) are one array, packed once
  int64_t a_entries, b_entries;               // batch entries packed per group (1 for a shared operand)
  int64_t rm_p, rn_p;                         // panel rows padded to whole tiles
  int64_t parts;                              // k ranges of the row norms
  size_t bytes_a, bytes_b, bytes_r, bytes_e, bytes_n, bytes_f;
  size_t total() const { return bytes_a + bytes_b + bytes_r + bytes_e + bytes_n + bytes_f; }
};

size_t align256(size_t x) { return (x + 255) / 256 * 256; }
int64_t round_up(int64_t x, int64_t to) { return ceil_div(x, to) * to; }

// op(A)^T and op(B) are one array.
bool one_operand(const Gemm& g) {
  return g.A == g.B && g.ta != g.tb && g.lda == g.ldb && g.m == g.n && g.batch == 1;
}

// Buffer sizes of the panels; what the packs leave is the room for the residues,
// which go by columns (at least 512, or all), then rows.  False when that does not fit.
bool size_panels(const Gemm& g, size_t capacity, Panels& p) {
  p.rm_p = round_up(p.rows_m, kTileM);
  p.rn_p = round_up(p.rows_n, p.tile_n);
  p.a_entries = g.strideA == 0 ? 1 : p.batch;
  p.b_entries = g.strideB == 0 ? 1 : p.batch;
  if (p.same) p.rm_p = p.rn_p = std::max(p.rm_p, p.rn_p);
  p.bytes_a = align256(size_t(p.a_entries * kPlanes) * size_t(p.rm_p * p.KS * kDepth));
  p.bytes_b = p.same ? 0 : align256(size_t(p.b_entries * kPlanes) * size_t(p.rn_p * p.KS * kDepth));
  p.bytes_e = align256((sizeof(int) + sizeof(float)) * size_t(p.a_entries * p.rm_p + p.b_entries * p.rn_p));
  p.bytes_n = align256(16 * size_t(std::max(p.a_entries * p.rm_p, p.b_entries * p.rn_p) * p.parts));
  p.bytes_r = p.bytes_f = 0;
  if (p.total() >= capacity) return false;
  // outputs: a byte per modulus, and the flags of a tile
  const int64_t room = int64_t(double(capacity - p.total()) / (double(p.batch) * (kModuli + 0.001))) - 512;
  auto residues_of = [&](int64_t outputs) {
    p.bytes_r = align256(size_t(p.batch * kModuli) * size_t(outputs));
    p.bytes_f = align256(sizeof(int) * size_t(p.batch) * size_t(outputs / (int64_t(kTileM) * p.tile_n)));
    return p.total() <= capacity;
  };
  p.out_m = p.rm_p;
  p.out_n = p.rn_p;
  // a quarter of the capacity (or all) for the residues: thinner pieces leave CUs idle
  if (room < std::min(p.rm_p * p.rn_p, int64_t(capacity / 4) / (p.batch * kModuli))) return false;
  // of a lower block triangle as many columns as have room: the first ones are the
  // longest, and only tiles of the triangle are kept
  const int64_t tile = int64_t(kTileM) * p.tile_n;
  if (g.lower > 0 && p.rows_m == g.m && p.rows_n == g.n) {
    auto outputs = [&](int64_t cols) { return map_tiles(p.rm_p, cols, p.tile_n, g.lower, 0, 0).count * tile; };
    int64_t fit = 0, over = p.rn_p / p.tile_n + 1;                       // column tiles
    while (over - fit > 1) {
      const int64_t mid = (fit + over) / 2;
      (outputs(mid * p.tile_n) <= room ? fit : over) = mid;
    }
    if (fit * p.tile_n >= std::min<int64_t>(p.rn_p, 512)) {
      p.out_n = fit * p.tile_n;
      return residues_of(outputs(p.out_n));
    }
  }
  const int64_t least = std::min<int64_t>(p.out_n, 512);
  if (p.out_m * p.out_n > room) p.out_n = std::max(least, room / p.out_m / p.tile_n * p.tile_n);
  if (p.out_m * p.out_n > room) p.out_m = room / p.out_n / kTileM * kTileM;
  if (p.out_m < std::min<int64_t>(p.rm_p, 1024)) return false;
  return residues_of(p.out_m * p.out_n);
}

// The whole product where its packs fit the capacity, else equal groups of the
// batch, else (one entry at a time) equal panels of rows, the longer panel split
// first.  A panel more of one operand packs the other once more: 7.3 ps per element
// against the 13.3 fs of products that each of its elements has with every row
// of the panel, so panels of 2560 rows cost a fifth, of 6912 rows a twelfth.
bool plan_panels(const Gemm& g, size_t capacity, Panels& p) {
  p.KS = ceil_div(g.k, kDepth);
  p.tile_n = g.k <= kShortDepth ? 128 : 256;
  p.parts = std::max<int64_t>(1, std::min<int64_t>(64, g.k / 256));
  p.rows_m = g.m;
  p.rows_n = g.n;
  p.batch = g.batch;
  p.same = one_operand(g);
  int64_t groups = 1, pm = 1, pn = 1;
  while (!size_panels(g, capacity, p)) {
    if (p.same) {
      p.same = false;
    } else if (p.batch > 1) {
      p.batch = ceil_div(g.batch, ++groups);
    } else if (p.rows_m >= p.rows_n) {
      if (p.rows_m <= kTileM) return false;
      p.rows_m = std::min(g.m, round_up(ceil_div(g.m, ++pm), kTileM));
    } else {
      if (p.rows_n <= kTileM) return false;
      p.rows_n = std::min(g.n, round_up(ceil_div(g.n, ++pn), kTileM));
    }
  }
  return true;
}

// One operand panel: exponents, then the pack.
void pack_operand(hipStream_t s, const double* X, int64_t ld, int64_t strideX, bool kcontig, int64_t rows, int64_t K,
                  int64_t KS, int64_t rows_p, int64_t entries, int64_t parts, void* norms, int* e, float* nrm, u4* P, int* flags,
                  int64_t n_flags) {
  if (kcontig) {
    row_exponents_kcontig_kernel<<<dim3(unsigned(rows), unsigned(entries)), 256, 0, s>>>(X, ld, strideX, K, rows_p, e, nrm);
    ETG_LAUNCH("row_exponents");
  } else {
    const int64_t k_per = ceil_div(K, parts);
    double* ps = static_cast<double*>(norms);
    unsigned long long* pm = reinterpret_cast<unsigned long long*>(ps + entries * rows * parts);
    row_norms_partial_kernel<<<dim3(unsigned(ceil_div(rows, 64)), unsigned(parts), unsigned(entries)), 256, 0, s>>>(
        X, ld, strideX, rows, K, k_per, ps, pm);
    ETG_LAUNCH("row_norms");
    row_exponents_finish_kernel<<<dim3(unsigned(ceil_div(rows, 256)), unsigned(entries)), 256, 0, s>>>(
        ps, pm, rows, int(parts), K, rows_p, e, nrm);
    ETG_LAUNCH("row_exponents");
  }
  residue_pack_kernel<<<dim3(unsigned(ceil_div(KS, 4)), unsigned(ceil_div(rows, 16)), unsigned(entries)), 256, 0, s>>>(
      X, ld, strideX, kcontig ? 1 : 0, rows, K, KS, rows_p * KS * (kDepth / 16), e, rows_p, P,
      flags, n_flags);
  ETG_LAUNCH("residue_pack");
}

}  // namespace

// Estimated microseconds of the int8 path against those of the FP64 kernels
// (`fp64_seconds`, at least the 50 TFLOP/s that products of a few hundred rows reach).
// Products: rounds of 512 or 256 workgroups, each 0.69 or 0.74 us per step of 64 k and 2.1
// to begin and end; the last of a few rounds counts half as a whole one (its workgroups
// run faster alone).  Packs 7.3 ps per operand element with the norms, an operand shared
// by both sides once; 7.6 ps per output; 35 us of launches.  Fitted to 260 products of
// m, n = 128 .. 19000, k = 128 .. 32768 (0.6 .. 400 GFLOP): 9 % rms.  Of these the rule sends
// none to the slower path by more than 5 %, and leaves two that would gain as much on the
// FP64 kernels; without the rounds and with the constants of 15 moduli it sent twelve
// (5559 x 3230 x 313 1.31 times slower, 424 x 2101 x 26993 912 against 1050 us).
bool residue_pays(const Gemm& g, double fp64_seconds) {
  if (g.k > residue::kMaxDepth || std::min(g.m, g.n) < 128 || g.k < 128) return false;
  const double b = double(g.batch), m = double(g.m), n = double(g.n), k = double(g.k);
  const bool small = g.k <= kShortDepth;
  const double tiles = double(ceil_div(g.m, kTileM)) * double(ceil_div(g.n, small ? 128 : 256)) * b;
  const double q = tiles * kPlanes / (small ? 512.0 : 256.0);
  const double rounds = q > 8.0 ? q : 0.5 * std::ceil(q) + 0.5 * std::max(1.0, q);
  const double products = rounds * ((small ? 0.69 : 0.74) * double(ceil_div(g.k, kDepth)) + 2.1);
  const double elements = (g.strideA == 0 ? 1.0 : b) * m * k + (one_operand(g) ? 0.0 : (g.strideB == 0 ? 1.0 : b) * n * k);
  const double us = 35.0 + products + 7.3e-6 * elements + 7.6e-6 * m * n * b;
  return us < 1e6 * std::min(fp64_seconds, 2.0 * m * n * k * b / 50e12);
}

bool residue_fits(const Gemm& g, const GemmWorkspace* ws) {
  Panels p{};
  return ws->residue && !ws->residue->refused && plan_panels(g, ws->residue->capacity, p);
}

bool gemm_residue(hipStream_t stream, const Gemm& g, GemmWorkspace* ws, bool may_allocate, GemmLaunch* info) {
  ResidueWorkspace* rw = ws->residue.get();
  Panels p{};
  if (rw == nullptr || rw->refused || !plan_panels(g, rw->capacity, p)) return false;
  if (rw->buf.bytes() == 0) {
    if (!may_allocate) return false;
    try {
      rw->buf.resize(rw->capacity);
    } catch (const Error&) {
      (void)hipGetLastError();
      rw->refused = true;
      return false;
    }
  }
  char* base = rw->buf.as<char>();
  u4* PA = reinterpret_cast<u4*>(base);
  u4* PB = p.same ? PA : reinterpret_cast<u4*>(base + p.bytes_a);
  uint32_t* R = reinterpret_cast<uint32_t*>(base + p.bytes_a + p.bytes_b);
  int* ea = reinterpret_cast<int*>(base + p.bytes_a + p.bytes_b + p.bytes_r);
  int* eb = p.same ? ea : ea + p.a_entries * p.rm_p;
  float* na = reinterpret_cast<float*>(ea + p.a_entries * p.rm_p + p.b_entries * p.rn_p);
  float* nrm_b = p.same ? na : na + p.a_entries * p.rm_p;
  void* norms = base + p.bytes_a + p.bytes_b + p.bytes_r + p.bytes_e;
  int* flags = reinterpret_cast<int*>(base + p.bytes_a + p.bytes_b + p.bytes_r + p.bytes_e + p.bytes_n);
  const bool a_kcontig = g.ta, b_kcontig = !g.tb;
  const int64_t pm = ceil_div(g.m, p.rows_m), pn = ceil_div(g.n, p.rows_n);
  // one panel of op(A), group of batch entries and panel of op(B); an operand is
  // packed again only where the last pack was another one
  int64_t a_is = -1, b_is = -1;
  auto panel = [&](int64_t mi, int64_t bi, int64_t ni) {
    const int64_t m0 = mi * p.rows_m, b0 = bi * p.batch, n0 = ni * p.rows_n;
    const int64_t m = std::min(p.rows_m, g.m - m0), n = std::min(p.rows_n, g.n - n0), nb = std::min(p.batch, g.batch - b0);
    const double* A = g.A + b0 * g.strideA + (a_kcontig ? m0 * g.lda : m0);
    const double* B = g.B + b0 * g.strideB + (b_kcontig ? n0 * g.ldb : n0);
    const int64_t a_want = mi + (g.strideA == 0 ? 0 : pm * bi), b_want = ni + (g.strideB == 0 ? 0 : pn * bi);
    const int64_t n_flags = int64_t(p.bytes_f / sizeof(int));
    bool clear = false;                  // the flags of the next launch
    if (a_want != a_is) {
      pack_operand(stream, A, g.lda, g.strideA, a_kcontig, m, g.k, p.KS, p.rm_p, g.strideA == 0 ? 1 : nb, p.parts, norms,
                   ea, na, PA, flags, n_flags);
      clear = true;
    }
    if (b_want != b_is && !p.same) {
      pack_operand(stream, B, g.ldb, g.strideB, b_kcontig, n, g.k, p.KS, p.rn_p, g.strideB == 0 ? 1 : nb, p.parts, norms,
                   eb, nrm_b, PB, flags, clear ? 0 : n_flags);
      clear = true;
    }
    a_is = a_want;
    b_is = b_want;
    for (int64_t c0 = 0; c0 < n; c0 += p.out_n) {
      // first row of the panel that these columns need, down to a whole tile
      const int64_t first = g.lower > 0 ? (n0 + c0) / g.lower * g.lower - m0 : 0;
      for (int64_t r0 = first > 0 ? first / kTileM * kTileM : 0; r0 < m; r0 += p.out_m) {
        const int64_t mo = std::min(p.out_m, m - r0), no = std::min(p.out_n, n - c0);
        Params q{};
        q.A = PA + r0 * p.KS * (kDepth / 16);
        q.B = PB + c0 * p.KS * (kDepth / 16);
        q.R = R;
        q.KS = p.KS;
        q.tiles = map_tiles(mo, no, p.tile_n, g.lower, m0 + r0, n0 + c0);
        q.planeA = p.rm_p * p.KS * (kDepth / 16);
        q.planeB = p.rn_p * p.KS * (kDepth / 16);
        q.planeR = int64_t(q.tiles.count) * kTileM * p.tile_n / 4;
        q.strideA = g.strideA == 0 ? 0 : kPlanes * q.planeA;
        q.strideB = g.strideB == 0 ? 0 : kPlanes * q.planeB;
        q.strideR = kModuli * q.planeR;
        q.flags = flags;
        q.strideF = q.tiles.count;
        q.m = mo; q.n = no;
        q.na = na + r0; q.nb = nrm_b + c0;
        q.na_stride = g.strideA == 0 ? 0 : p.rm_p;
        q.nb_stride = g.strideB == 0 ? 0 : p.rn_p;
        const unsigned tiles = unsigned(q.tiles.count);
        const dim3 grid(tiles, kPlanes, unsigned(nb));
        if (!clear) fill(stream, reinterpret_cast<double*>(flags), ceil_div(nb * q.strideF, 2), 0.0);
        clear = false;
        if (p.tile_n == 128)
          residue_product_kernel<2, 3><<<grid, 256, 0, stream>>>(q);
        else
          residue_product_kernel<4, 4><<<grid, 512, 0, stream>>>(q);
        ETG_LAUNCH("residue_product");
        Output o{};
        o.R = R;
        o.planeR = q.planeR;
        o.strideR = q.strideR;
        o.tiles = q.tiles;
        o.m = mo; o.n = no; o.K = g.k;
        o.ea = ea + r0; o.eb = eb + c0;
        o.ea_stride = q.na_stride;
        o.eb_stride = q.nb_stride;
        o.alpha = g.alpha; o.beta = g.beta;
        o.C = g.C + b0 * g.strideC + m0 + r0 + (n0 + c0) * g.ldc;
        o.ldc = g.ldc; o.strideC = g.strideC;
        o.vec_rows = mo % 4 == 0 && g.ldc % 2 == 0 && (g.batch == 1 || g.strideC % 2 == 0) &&
                     reinterpret_cast<uintptr_t>(o.C) % 16 == 0;
        o.flags = flags;
        o.strideF = q.strideF;
        residue_reconstruct_kernel<<<dim3(tiles * unsigned(kBlocksM * p.tile_n / 64), unsigned(nb)), 256, 0, stream>>>(o);
        ETG_LAUNCH("residue_reconstruct");
        Gemm f = g;
        f.m = mo; f.n = no;
        f.A = A + (a_kcontig ? r0 * g.lda : r0);
        f.B = B + (b_kcontig ? c0 * g.ldb : c0);
        f.C = o.C;
        f.batch = nb;
        gemm_flagged_blocks(stream, f, q.tiles, flags, q.strideF);
      }
    }
  };
  // the outer operand's panels are packed once, the inner one's once per outer panel
  // (and both once per group of the batch unless shared)
  const int64_t ng = ceil_div(g.batch, p.batch);
  const bool a_outer = g.batch > 1 ? g.strideA == 0 || g.strideB != 0
                                   : (pn > 1 ? g.m + pm * g.n : g.m + g.n) <= (pm > 1 ? g.n + pn * g.m : g.n + g.m);
  for (int64_t x = 0; x < (a_outer ? pm : pn); ++x)
    for (int64_t bi = 0; bi < ng; ++bi)
      for (int64_t y = 0; y < (a_outer ? pn : pm); ++y) panel(a_outer ? x : y, bi, a_outer ? y : x);
  *info = GemmLaunch{p.tile_n == 128 ? "gemm_residue<256x128>" : "gemm_residue<256x256>", 1};
  return true;
}

}  // namespace etg

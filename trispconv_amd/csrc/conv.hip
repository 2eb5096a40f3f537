// Fused sparse convolution: gather -> GEMM -> scatter over all kernel slots in
// one launch, plus the weight packer that feeds it.
//
// Reference semantics (trispconv/pytorch/functional.py:27-51, GPU branch):
// out = 0; for k ascending: out[pairs_out[k]] += feat[pairs_in[k]] @ W[k] in
// fp32 (fp16/bf16 inputs upcast, :34-36); then + bias; then one rounding to the
// input dtype (:51).  The reference launches one Triton kernel per slot with an
// atomic-add scatter (triton_kernels.py:31-92).
//
// MI355X design: output-stationary implicit GEMM.  A workgroup owns a tile of
// output rows (in the order the plan chose) and one column tile; it keeps the
// fp32 accumulators in registers across all slots, gathers each slot's input
// rows straight into MFMA operand registers, stages the slot's weight slice in
// LDS (double-buffered), and writes each output row exactly once.  No atomics:
// every output element is a fixed sequence of fp32 operations, so results are
// bitwise reproducible and independent of the tile order.
//
// Two code shapes share that structure:
//   * mfma: f32/f16/bf16 with C_in a multiple of 16, C_out of 32 and K <= 64
//     — v_mfma_f32_32x32x16_{f16,bf16} (f32 as three bf16 values), 4 waves x
//     (64 rows x BN cols) per tile.
//   * narrow: every other layer (a LiDAR encoder's 4 -> 16 or 5 -> 16 first
//     layer, 16-wide outputs, 20 class scores, K > 64) —
//     v_mfma_f32_16x16x32_{f16,bf16} or v_mfma_f32_16x16x4_f32 over (slot,
//     channel) pairs, 16 rows per wave.
//
// The epilogue adds the bias and, when asked, an eval-mode batch norm and a
// ReLU (a BatchNorm1d and ReLU following the convolution in a
// SparseSequential), all in fp32 before the one rounding.  The batch norm is
// read from its running statistics and affine parameters on every launch, so
// no folded copy of them can go stale.
#include "common.hpp"

#include <algorithm>
#include <type_traits>

namespace tsc {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

enum Path { kMfma = 1, kNarrow = 2 };

// Input-channel chunk of one stage: 64 bytes of every gathered row per lane
// half (64 channels of f16/bf16, 32 of f32), or half that when the channels
// do not divide.  With C_in an odd multiple of 16 the last chunk's upper half
// is padding: those lanes read the zero row and the packed weight holds zeros.
int pick_ck(int dtype, int c_in) {
  if (dtype == TSC_F32) return 32;
  return c_in % 64 == 0 ? 64 : 32;
}
int pick_bn(int c_out) { return c_out % 128 == 0 ? 128 : (c_out % 64 == 0 ? 64 : 32); }
int64_t mfma_chunks(int c_in, int ck) { return ceil_div(c_in, ck); }

// The 32x32 tile for every dtype when C_in is a multiple of 16 and C_out of 32
// (the slot table of K <= 64 slots fits LDS); the narrow MFMA kernel for every
// other width.
Path pick_path(int dtype, int c_in, int c_out, int K) {
  if (c_in % 16 == 0 && c_out % 32 == 0 && K <= 64) return kMfma;
  return kNarrow;
}

// Channels of a slot in the narrow kernel's reduction: C_in rounded up to
// whole 4-channel pieces (the padding has zero weights), so that a piece never
// straddles two slots.
int narrow_cp(int c_in) { return (c_in + 3) / 4 * 4; }

// Steps of the narrow kernel: 16 bytes of reduction values (slot, channel)
// per lane quad, i.e. 32 values for f16/bf16 and 16 for f32; the last step is
// padded with zero weights.
int64_t narrow_steps(int dtype, int K, int c_in) {
  return ceil_div((int64_t)K * narrow_cp(c_in), 4 * (16 / dtype_bytes(dtype)));
}

// ----------------------------------------------------------- weight pack --
__device__ __forceinline__ float load_any(const void* p, int dt, int64_t i) {
  if (dt == TSC_F32) return static_cast<const float*>(p)[i];
  if (dt == TSC_F16) return __half2float(static_cast<const __half*>(p)[i]);
  return __bfloat162float(static_cast<const __hip_bfloat16*>(p)[i]);
}

// Entry i of a per-channel parameter (bias, batch-norm statistics) as fp32
// without a branch on the dtype: two 16-bit reads that are in bounds for every
// dtype (the halves of an fp32, or the same 16-bit entry twice), then selects.
// A three-way branch here, in the epilogue, once led the compiler to leave the
// output address undefined on the bf16 arm.
__device__ __forceinline__ float load_param(const void* p, int dt, int64_t i) {
  const uint16_t* q = static_cast<const uint16_t*>(p);
  const bool wide = dt == TSC_F32;
  const uint32_t lo = q[wide ? 2 * i : i];
  const uint32_t hi = q[wide ? 2 * i + 1 : i];
  const uint32_t bits = wide ? (lo | (hi << 16)) : (dt == TSC_BF16 ? lo << 16 : 0u);
  const float h = __half2float(__ushort_as_half(static_cast<unsigned short>(lo)));
  return dt == TSC_F16 ? h : __uint_as_float(bits);
}

// What happens to an output element after the slot sum: v = acc + bias[c];
// with a batch norm v = (v - mean[c]) / sqrt(var[c] + eps) * gamma[c] +
// beta[c]; with relu v = max(v, 0) (NaN stays NaN); then one rounding.
struct Epilogue {
  const void* bias;     // per output channel, bias_dt, or null
  int bias_dt;
  const void* mean;     // batch-norm running mean and variance, or null for none
  const void* var;
  const void* gamma;    // its affine weight and bias, each null for 1 and 0
  const void* beta;
  int bn_dt;            // dtype of mean, var, gamma and beta
  float eps;
  int relu;
};

// The batch norm of channel c as v * sc + sh: sc = gamma / sqrt(var + eps),
// sh = beta - mean * sc (the linear-plus-constant form torch's CPU batch norm
// evaluates).  1 and 0 without a batch norm.
__device__ __forceinline__ void channel_affine(const Epilogue& ep, int64_t c, float& sc,
                                               float& sh) {
  sc = 1.f;
  sh = 0.f;
  if (!ep.mean) return;
  float s = 1.f / sqrtf(load_param(ep.var, ep.bn_dt, c) + ep.eps);
  if (ep.gamma) s *= load_param(ep.gamma, ep.bn_dt, c);
  const float b = ep.beta ? load_param(ep.beta, ep.bn_dt, c) : 0.f;
  sc = s;
  sh = b - load_param(ep.mean, ep.bn_dt, c) * s;
}

__device__ __forceinline__ float finish(float v, float scale, float shift, bool affine, bool relu) {
  if (affine) v = fmaf(v, scale, shift);
  if (relu) v = v < 0.f ? 0.f : v;
  return v;
}

__device__ __forceinline__ float src_weight(const void* w, int dt, int layout, int K, int c_in,
                                            int c_out, int k, int ci, int co) {
  const int64_t idx = layout == 0 ? ((int64_t)co * K + k) * c_in + ci
                                  : ((int64_t)k * c_in + ci) * c_out + co;
  return load_any(w, dt, idx);
}

// f32 layers of the 32x32 tile hold two things about their weights besides them,
// where the last chunk is half padding (C_in % 32 == 16) in that padding, which
// only ever multiplies zero rows, else behind the layout:
//   * the range word, the buffer's last: the bits of their largest magnitude, or
//     kNoSplit where a weight is not finite or so small that three bf16 values
//     do not hold it (a finite number, so its products with zeros are zeros);
//   * a float per column, 1 where the column has a weight other than 0, else 0.
constexpr uint32_t kNoSplit = 0xff7fffffu;        // -FLT_MAX, above every magnitude's bits
constexpr uint32_t kSplitHolds = (127 - 110) << 23;  // 2^-110: larger values split without a rest
__host__ __device__ __forceinline__ int range_tail(int c_in, int c_out) {
  return c_in % 32 ? 0 : c_out + 4;
}
__host__ __device__ __forceinline__ uint32_t* range_word(const float* packed, int64_t layout, int c_in,
                                                         int c_out) {
  return reinterpret_cast<uint32_t*>(const_cast<float*>(packed)) + layout + range_tail(c_in, c_out) - 1;
}
// Padding: lane 32 + column % 32 of the column's block, the last stage's last
// vector, one float before the range word's place in it.
__device__ __forceinline__ float* column_flag(const float* packed, int64_t layout, int c_in, int c_out,
                                              int column) {
  return const_cast<float*>(packed) + layout +
         (c_in % 32 ? -32 * c_out + column / 32 * 1024 + 3 * 256 + (32 + column % 32) * 4 + 2 : column);
}

// MFMA layout: [k][chunk][c_out/32][u][lane][16/sizeof(T)].  Lane l of a
// 32-column block n supplies column n*32 + l%32, and for lane half h = l/32
// the channels c*CK + h*CK/2 + u*(16/sizeof(T)) + 0.. of chunk c: the same
// channel split the A operand uses, so that each lane's A data is a
// contiguous CK/2-channel (64-byte) run of a row.  An f16/bf16 MFMA step
// (32x32x16) takes one 16-byte vector per lane, an f32 one two of them (split
// into three bf16 operands), a step of the f32 unit (32x32x2) one element.
template <typename T>
__global__ void pack_mfma_kernel(const void* w, int w_dt, int layout, int K, int c_in, int c_out,
                                 int ck, T* packed) {
  constexpr int VPL = 16 / sizeof(T);  // values per 16-byte vector
  const int ub = (ck / 2) / VPL;      // vectors per lane per chunk
  const int nbt = c_out / 32;
  const int nch = (c_in + ck - 1) / ck;  // the last chunk may be half padding
  const int64_t total = (int64_t)K * nch * ck * c_out;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int i = e % VPL;
    const int lane = (e / VPL) & 63;
    int64_t r = e / (VPL * 64);
    const int u = r % ub;
    r /= ub;
    const int nb = r % nbt;
    r /= nbt;
    const int c = r % nch;
    const int k = r / nch;
    const int ci = c * ck + (lane >> 5) * (ck / 2) + u * VPL + i;
    const int co = nb * 32 + (lane & 31);
    packed[e] = from_f32<T>(ci < c_in ? src_weight(w, w_dt, layout, K, c_in, c_out, k, ci, co)
                                      : 0.f);
  }
  if constexpr (std::is_same<T, float>::value)  // no column marked, no magnitude seen (padding is 0 too)
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < range_tail(c_in, c_out);
         e += gridDim.x * blockDim.x)
      packed[total + e] = 0.f;
}

// The range word and the column marks.  KRSC weights are [column][slot and
// channel]: a block takes one column; flat ones end in the columns: a block takes
// 32 of them.  One atomic per block, as they all meet in one word: packing 27 x 64
// -> 64 takes 6.0 us with it, 24.6 with one per wave, 4.1 without the range.
template <bool KRSC>
__global__ void __launch_bounds__(1024) weight_range_kernel(const void* w, int w_dt, int64_t rows, int c_in,
                                                            int c_out, float* packed, int64_t layout) {
  constexpr int CB = KRSC ? 1 : 32, RL = 1024 / CB;
  const int col = blockIdx.x * CB + threadIdx.x % CB;
  uint32_t most = 0;
#pragma unroll 4
  for (int64_t r = (int64_t)blockIdx.y * RL + threadIdx.x / CB; r < rows; r += (int64_t)gridDim.y * RL) {
    const uint32_t v = __float_as_uint(load_any(w, w_dt, KRSC ? col * rows + r : r * c_out + col)) & 0x7fffffffu;
    const bool held = v < 0x7f800000u && (v == 0 || v >= kSplitHolds);
    most = max(most, held ? v : kNoSplit);
  }
  if (most) *column_flag(packed, layout, c_in, c_out, col) = 1.f;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(most, off, kWave)));
  __shared__ uint32_t s_most[1024 / kWave];
  if (threadIdx.x % kWave == 0) s_most[threadIdx.x / kWave] = most;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (const uint32_t m : s_most) most = max(most, m);
    atomicMax(range_word(packed, layout, c_in, c_out), most);
  }
}

// The direct-to-LDS kernel's output rows are written once and not read
// again by the launch: when a row is whole 128-byte lines (nt), non-temporal
// stores keep them from displacing the gathered input rows in the caches.
// Measured: headline 128->128 layer 310-312 -> 306-308 us, two such layers
// in sequence (the second gathering the first's output) no slower, the
// encoder's 64->64 layers 28.5 -> 28.0 us, the LiDAR 64->64 fp32 layer 137
// -> 135 us.  Not for the register-gather kernel: the 674k-row 32->64 bf16
// strided layer's output (86 MB) is the next inverse layer's input, which
// then misses the Infinity Cache (that layer 56 -> 61 us).
__device__ __forceinline__ void store_out(void* dst, uint4 v, bool nt) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  if (nt) {
    const u32x4 w = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(w, static_cast<u32x4*>(dst));
  } else {
    *static_cast<uint4*>(dst) = v;
  }
}

// Operand source for absent neighbours: lanes whose output row has no input
// through the current slot read zeros from here instead of branching around
// their loads (64 bytes per lane are read at most).
__device__ __attribute__((aligned(256))) uint4 g_zero_row[16];

// Weights of widths that do not fill the narrow kernel's pieces and tiles keep
// their own type: packed for 16-bit features they come in one of two forms, told
// apart by the buffer's last word.
//   * Weights of the features' type: the narrow layout, and kNarrowForm (a NaN
//     with bits of its own).
//   * Others: f32, [slot][channel][column].  The last word is then the last
//     weight, with a NaN's bits made plain, or 0 in a longer buffer.
constexpr uint32_t kNarrowForm = 0x7fc5a51eu;
bool has_forms(int dtype, int c_in, int c_out) {
  return dtype != TSC_F32 && (c_in % 4 != 0 || c_out % 16 != 0);
}
int64_t narrow_bytes(int dtype, int K, int c_in, int c_out) {
  return narrow_steps(dtype, K, c_in) * ceil_div(c_out, 16) * 64 * 16;
}

__global__ void __launch_bounds__(256) pack_wide_kernel(const void* w, int w_dt, int layout, int K,
                                                        int c_in, int c_out, float* packed,
                                                        uint32_t* form) {
  const int64_t total = (int64_t)K * c_in * c_out;
  for (int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
    const int co = e % c_out;
    const int ci = (e / c_out) % c_in;
    const int k = e / ((int64_t)c_in * c_out);
    const float v = src_weight(w, w_dt, layout, K, c_in, c_out, k, ci, co);
    packed[e] = v == v ? v : __uint_as_float(0x7fc00000u);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0 && form >= reinterpret_cast<uint32_t*>(packed) + total)
    *form = 0u;
}

// Narrow layout: [step i][ceil(c_out/16)][lane][LV], LV = 16 / sizeof(T)
// values.  Lane l of 16-column tile n supplies column n*16 + l%16 and the
// reduction values r = 4*LV*i + LV*(l/16) + 0..LV-1, r = k * cp + c for slot k
// and channel c, cp = C_in rounded up to a multiple of 4: the values the A
// operand's lane l gathers for its row.  Zero past the last slot, the last
// channel and the last column.
template <typename T>
__global__ void pack_narrow_kernel(const void* w, int w_dt, int layout, int K, int c_in,
                                   int c_out, int64_t nsteps, T* packed, uint32_t* form) {
  if (form && blockIdx.x == 0 && threadIdx.x == 0) *form = kNarrowForm;
  constexpr int LV = 16 / (int)sizeof(T);
  const int nt_all = (c_out + 15) / 16;
  const int cp = (c_in + 3) / 4 * 4;
  const int64_t total = nsteps * nt_all * 64 * LV;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int v = e % LV;
    const int lane = (e / LV) % 64;
    const int nt = (e / (64 * LV)) % nt_all;
    const int64_t i = e / (64 * LV * (int64_t)nt_all);
    const int64_t r = 4 * LV * i + LV * (lane / 16) + v;
    const int k = static_cast<int>(r / cp);
    const int ci = static_cast<int>(r % cp);
    const int co = nt * 16 + lane % 16;
    const bool in = k < K && ci < c_in && co < c_out;
    packed[e] = from_f32<T>(in ? src_weight(w, w_dt, layout, K, c_in, c_out, k, ci, co) : 0.f);
  }
}

// ---------------------------------------------------------------- MFMA --
template <typename T> struct MfmaOp;
template <> struct MfmaOp<__half> {
  using V = f16x8;
  static __device__ __forceinline__ f32x16 run(V a, V b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct MfmaOp<__hip_bfloat16> {
  using V = bf16x8;
  static __device__ __forceinline__ f32x16 run(V a, V b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct MfmaOp<float> {
  using V = float;
  static __device__ __forceinline__ f32x16 run(V a, V b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
};

// ------------------------------------------------- f32 on the bf16 cores --
// f32 operands as sums of three bf16 values each, x = hi + mid + lo: hi is x
// rounded to bf16, mid the rest rounded to bf16, lo what is left, which has at
// most 8 significant bits and is exact.  A product is then six bf16 products,
//   x * y = lo*hi' + hi*lo' + mid*mid' + mid*hi' + hi*mid' + hi*hi'
// (exact each, summed in the f32 accumulator); the three left out are below
// 2^-24 of it.  A 32x32x16 bf16 MFMA takes 32 cycles, eight 32x32x2 f32 ones
// take 512, so a stage's matrix work falls to 6 * 32 / 512 = 0.375 of the f32
// unit's; the splits are vector work (11 instructions for two values).
// Relative 2-norm error against 64 bits, the f32 unit's and this one's:
// 27 x 64 -> 64 SubM, 100k rows, 5.3e-7 and 4.5e-7; 64 -> 64 stride 2 on
// LiDAR voxels 4.4e-7 and 3.7e-7.  Their times (the first's launch, the
// second's whole frame with its build and plan): 179 -> 133 us, 301 -> 251 us.
// What three bf16 values cannot hold is computed once more on the f32 unit
// (Redo below), element by element, so that neither the tile nor the order
// decides which sums those are:
//   * A value that is not finite or rounds to infinity in bf16 makes its
//     products NaN: accumulators that end up not finite.
//   * Below 2^-110 lo is short of bf16's exponents (subnormals, which both units
//     keep, end at 2^-133): an error of up to 2^-134, times the other operand.
//     For features that is at most max|w| 2^-134 for each of up to 2^18
//     products, so sums of at least max|w| 2^-88 have it below 2^-28 of them,
//     and smaller ones are computed again (max|w| from the range word of the
//     packed weights).  A sum of exactly zero is, where its column has weights
//     and its row gathers a value so small that all three parts may vanish.
//   * Layers with such weights run on the f32 unit throughout: nothing bounds
//     the features that would multiply their errors.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void split_pair(float x, float y, uint32_t& hi, uint32_t& mid,
                                           uint32_t& lo) {
  auto pack = [](float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
  };
  auto low = [](uint32_t v) { return __uint_as_float(v << 16); };
  auto high = [](uint32_t v) { return __uint_as_float(v & 0xffff0000u); };
  hi = pack(x, y);
  const float rx = x - low(hi), ry = y - high(hi);
  mid = pack(rx, ry);
  lo = pack(rx - low(mid), ry - high(mid));
}

struct Split8 {  // eight f32 values of one operand
  bf16x8 hi, mid, lo;
};
__device__ __forceinline__ Split8 split8(const uint4& a, const uint4& b) {
  const float4 x = __builtin_bit_cast(float4, a), y = __builtin_bit_cast(float4, b);
  uint4 h, m, l;
  split_pair(x.x, x.y, h.x, m.x, l.x);
  split_pair(x.z, x.w, h.y, m.y, l.y);
  split_pair(y.x, y.y, h.z, m.z, l.z);
  split_pair(y.z, y.w, h.w, m.w, l.w);
  return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m),
          __builtin_bit_cast(bf16x8, l)};
}
__device__ __forceinline__ f32x16 mfma_split(const Split8& a, const Split8& b, f32x16 c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.lo, b.hi, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.hi, b.lo, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.mid, b.mid, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.mid, b.hi, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.hi, b.mid, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.hi, b.hi, c, 0, 0, 0);
}

// A split weight slab in LDS: [plane hi/mid/lo][column block nb][half t of the
// 32-channel chunk][lane][16 bytes].  Vector u of block nb (four f32 values of
// each lane, as packed) goes to half u / 2, eight bytes at (u % 2) * 8: an
// operand of half t is then one 16-byte read per plane.
template <int NB>
__device__ __forceinline__ void store_split(uint4* slab, int nb, int u, int lane, const uint4& v) {
  const float4 x = __builtin_bit_cast(float4, v);
  uint2 pl[3];
  split_pair(x.x, x.y, pl[0].x, pl[1].x, pl[2].x);
  split_pair(x.z, x.w, pl[0].y, pl[1].y, pl[2].y);
#pragma unroll
  for (int p = 0; p < 3; ++p)
    reinterpret_cast<uint2*>(slab)[(((p * NB + nb) * 2 + (u >> 1)) * 64 + lane) * 2 + (u & 1)] = pl[p];
}
template <int NB>
__device__ __forceinline__ Split8 load_split(const uint4* slab, int nb, int t, int lane) {
  auto plane = [&](int p) {
    return __builtin_bit_cast(bf16x8, slab[((p * NB + nb) * 2 + t) * 64 + lane]);
  };
  return {plane(0), plane(1), plane(2)};
}

// The smallest sum that the split settles, from the packed weights' range word;
// infinity: none (the layer runs on the f32 unit).
__device__ __forceinline__ float split_limit(uint32_t range) {
  const float limit = fmaxf(0x1p-80f, __uint_as_float(range) * 0x1p-88f);
  return __uint_as_float(__builtin_amdgcn_readfirstlane(
      range == kNoSplit ? 0x7f800000u : __float_as_uint(limit)));
}

// Bit r set: row r of a 32-row block is in `rows` and gathers a value other than
// zero below 2^-132, which the split may turn into nothing.  s_orow: the block's
// output rows; first: its first processing position.  Sixteen lanes read a row,
// four rows of a wave and four slots at a time.
__device__ uint32_t vanishing_rows(const float* __restrict__ feat, int c_in,
                                   const int32_t* __restrict__ nbr, int nbr_ordered, int64_t n_out,
                                   int K, const int32_t* s_orow, int64_t first, uint32_t rows) {
  constexpr uint32_t kVanishing = (1u << 17) << 1;  // 2^-132's bits, shifted left
  constexpr int G = 4;
  const int lane = threadIdx.x & 63, group = lane >> 4, piece = lane & 15;
  uint32_t found = 0;
  for (int i = 0; i < 32; i += 4) {
    if (((rows >> i) & 15u) == 0) continue;
    const int r = i + group;
    const int32_t o = s_orow[r];
    const bool look = o >= 0 && ((rows >> r) & 1);
    bool any = false;
    for (int k0 = 0; k0 < K; k0 += G) {
      int32_t j[G];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        j[u] = -1;
        if (look && k0 + u < K)
          j[u] = nbr ? nbr[(int64_t)(k0 + u) * n_out + (nbr_ordered ? first + r : (int64_t)o)] : o;
      }
      for (int c = piece; c < c_in / 4; c += 16) {
        uint4 v[G];
#pragma unroll
        for (int u = 0; u < G; ++u)
          v[u] = j[u] >= 0 ? reinterpret_cast<const uint4*>(feat + (int64_t)j[u] * c_in)[c]
                           : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int u = 0; u < G; ++u)
          any |= (v[u].x << 1) - 1u < kVanishing - 1u || (v[u].y << 1) - 1u < kVanishing - 1u ||
                 (v[u].z << 1) - 1u < kVanishing - 1u || (v[u].w << 1) - 1u < kVanishing - 1u;
      }
    }
    const uint64_t b = __ballot(any);
#pragma unroll
    for (int g = 0; g < 4; ++g) found |= ((b >> (16 * g)) & 0xffffu) ? 1u << (i + g) : 0u;
  }
  return found;
}

// The elements of this lane's accumulators that the f32 unit computes again (see
// above), one bit each.
template <int RB, int NB>
struct Redo {
  uint32_t bits[(RB * NB + 1) / 2];
  // whether there may be any: 0 * x is 0 for every finite x, else NaN
  static __device__ __forceinline__ bool any(const f32x16 (&acc)[RB][NB], float limit) {
    float z = 0.f, least = 3.4028235e38f;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          z = fmaf(acc[rb][nb][i], 0.f, z);
          least = fminf(least, fabsf(acc[rb][nb][i]));
        }
    return !(z == 0.f) || least < limit;
  }
  // a wave's rows past the layer's last (it has `left` rows) sum to 1, not 0: a
  // layer's partial tile would otherwise always look for vanished sums, at the
  // end of the launch (64->64, 100k rows 132 -> 137 us)
  static __device__ __forceinline__ void pad(f32x16 (&acc)[RB][NB], int64_t left) {
    if (left >= 32 * RB) return;
    const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (rb * 32 + (i >> 2) * 8 + h * 4 + (i & 3) >= left) acc[rb][nb][i] = 1.f;
  }
  // rows of one block with an element of exactly zero in a column that has
  // weights, as row bits.  flag: this lane's column of the first block's mark.
  static __device__ __forceinline__ uint32_t zero_rows(const f32x16 (&acc)[NB], const float* flag,
                                                       int flag_stride) {
    bool live[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) live[nb] = flag[nb * flag_stride] != 0.f;
    uint32_t rows = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      bool zero = false;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) zero |= acc[nb][i] == 0.f && live[nb];
      const uint64_t b = __ballot(zero);
      const int r = (i >> 2) * 8 + (i & 3);
      rows |= (static_cast<uint32_t>(b) ? 1u << r : 0u) | (static_cast<uint32_t>(b >> 32) ? 16u << r : 0u);
    }
    return rows;
  }
  // vanish: per block, the rows whose zeros may be sums that vanished
  __device__ __forceinline__ void find(const f32x16 (&acc)[RB][NB], float limit,
                                       const uint32_t (&vanish)[RB]) {
    const int h = (threadIdx.x & 63) >> 5;
    for (uint32_t& b : bits) b = 0;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float v = fabsf(acc[rb][nb][i]);
          const int r = (i >> 2) * 8 + h * 4 + (i & 3);
          const bool bad = !(v <= 3.4028235e38f) ||
                           (v < limit && (v != 0.f || ((vanish[rb] >> r) & 1)));
          const int e = (rb * NB + nb) * 16 + i;
          bits[e / 32] |= (bad ? 1u : 0u) << (e % 32);
        }
  }
  __device__ __forceinline__ void all() {
    for (uint32_t& b : bits) b = 0xffffffffu;
  }
  __device__ __forceinline__ bool some() const {
    uint32_t m = 0;
    for (const uint32_t b : bits) m |= b;
    return m != 0;
  }
  __device__ __forceinline__ bool has(int rb, int nb, int i) const {
    const int e = (rb * NB + nb) * 16 + i;
    return (bits[e / 32] >> (e % 32)) & 1u;
  }
};

constexpr int kTileRows = kConvTileRows;  // 4 waves x 64 rows
constexpr int kSplitRows = 64;            // rows of a small-layer tile (its 4 waves split the slots)


template <int N> using Slot = std::integral_constant<int, N>;

// XCD placement: workgroups are dispatched round-robin over the 8 XCDs, in
// grid order.  Row tiles are dealt round-robin too (the execution order puts
// the tiles with the most slots first, so every XCD gets an even share of the
// heavy ones), and all column tiles of a row tile run one after another on the
// same XCD, sharing its L2 for the gathered rows.  Returns the work item
// (row tile * ncol + column tile) of workgroup lin.
__device__ __forceinline__ uint32_t dealt_item(uint32_t lin, uint32_t grid, uint32_t ncol) {
  const uint32_t dealt = (grid / (8 * ncol)) * (8 * ncol);  // whole rounds of 8 row tiles
  const uint32_t x = lin % 8, j = lin / 8;
  return lin < dealt ? ((j / ncol) * 8 + x) * ncol + j % ncol : lin;
}

// Output rows each wave stages per epilogue pass: 32 rows of up to 256 bytes,
// else 16, so the staging area stays within 35 KB for two workgroups per CU.
constexpr int mfma_stage_rows(int row_bytes) { return row_bytes <= 256 ? 32 : 16; }

// One workgroup (4 waves, one per SIMD) per CU; each wave owns 64 rows x BN
// columns of a 256-row tile.  The work of a tile is a sequence of stages
// (slot k present in the tile, 64- or 32-channel input chunk c).  Gathered
// input rows are loaded straight into MFMA operand registers RING-1 stages
// ahead (a ring of RING register buffers, so RING-1 stages of gathers are in
// flight while one computes); the stage's weight slab is loaded into registers
// one stage ahead and written to an LDS double buffer after the MFMAs, so all
// four waves share one copy.  fp32 accumulators live in AGPRs.
template <typename T, int BN, int CK>
__global__ void __launch_bounds__(256, 2) conv_mfma_kernel(
    const T* __restrict__ feat, int c_in, const T* __restrict__ W, Epilogue ep,
    const int32_t* __restrict__ nbr, const int32_t* __restrict__ order, int nbr_ordered,
    int64_t n_out, int K, int c_out, T* __restrict__ out) {
  using Op = MfmaOp<T>;
  using V = typename Op::V;
  constexpr int RING = 2;                        // operand buffers: this stage and the next
  constexpr bool F32 = std::is_same<T, float>::value;
  constexpr int VPL = 16 / (int)sizeof(T);       // values per 16-byte vector
  constexpr int UB = (CK / 2) / VPL;             // vectors per lane per row and stage
  static_assert(UB * VPL * 2 == CK && UB >= 1, "chunk must split into 16-byte runs");
  constexpr int NB = BN / 32;                    // 32-wide column blocks
  constexpr int SLAB_VECS = BN * CK * (int)sizeof(T) / 16;  // 16-byte vectors of one weight stage
  constexpr int WV = SLAB_VECS >= 256 ? SLAB_VECS / 256 : 1;
  constexpr bool FULL = SLAB_VECS % 256 == 0;
  static_assert(WV <= 4, "weight slab too large for the register stage");

  static_assert(!F32 || (UB == 4 && SLAB_VECS == 256 * NB), "a wave's share is one vector per block");
  __shared__ __attribute__((aligned(16))) uint4 s_w[2][F32 ? SLAB_VECS * 3 / 2 : SLAB_VECS];
  __shared__ __attribute__((aligned(16))) int32_t s_orow[kTileRows];
  __shared__ float s_bias[BN];        // this column tile's bias in fp32 (0 without one)
  __shared__ float s_scale[BN];       // its affine epilogue (1 and 0 without one)
  __shared__ float s_shift[BN];
  __shared__ uint64_t s_mask[4];      // per wave: slots its rows use (K <= 64)
  extern __shared__ int32_t s_nbr[];  // [K][kTileRows]; output staging at the end

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int h = lane >> 5;
  const uint32_t ncol = static_cast<uint32_t>(c_out / BN);
  // the launch keeps the grid below 2^31 workgroups
  const uint32_t item = dealt_item(blockIdx.x, gridDim.x, ncol);
  const int64_t tile0 = static_cast<int64_t>(item / ncol) * kTileRows;
  const int nbt = static_cast<int>(item % ncol);
  const int nch = (c_in + CK - 1) / CK;  // C_in % 16 == 0: the last chunk may be half padding
  uint32_t range = 0;  // f32: asked for here, used after the set-up
  if constexpr (F32) range = *range_word(W, (int64_t)K * nch * CK * c_out, c_in, c_out);

  // ---- tile set-up: output rows, their slot lists and slot masks.  The map
  // entries are read 32 slots at a time, all in flight before any is used
  // (rows past the end read column 0 and are then discarded).  A map permuted
  // into the execution order is indexed by processing position, so its first
  // batch goes out before the order lookup: one memory round trip, not two.
  {
    const int64_t tr = tile0 + t;
    const bool in = tr < n_out;
    uint64_t m = 0;
    int32_t jv[32];
    auto issue = [&](int k0, int64_t src_row, int32_t self) {
      if (nbr) {
        const int32_t* col = nbr + src_row;
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          const int k = k0 + i < K ? k0 + i : K - 1;
          jv[i] = col[(int64_t)k * n_out];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) jv[i] = self;
      }
    };
    auto consume = [&](int k0, int32_t orow) {
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int k = k0 + i;
        const int32_t j = orow >= 0 ? jv[i] : -1;
        if (k < K) {
          s_nbr[k * kTileRows + t] = j;
          m |= (j >= 0 ? uint64_t(1) : uint64_t(0)) << k;
        }
      }
    };
    // column of the map holding this row: its processing position when the map
    // was permuted into the execution order (contiguous reads), else the row
    int32_t orow;
    if (nbr && nbr_ordered) {
      issue(0, in ? tr : 0, 0);
      orow = in ? (order ? order[tr] : static_cast<int32_t>(tr)) : -1;
    } else {
      orow = in ? (order ? order[tr] : static_cast<int32_t>(tr)) : -1;
      issue(0, orow >= 0 ? orow : 0, orow >= 0 ? orow : 0);
    }
    s_orow[t] = orow;
    if (t < BN) {
      const int64_t col = (int64_t)nbt * BN + t;
      s_bias[t] = ep.bias ? load_param(ep.bias, ep.bias_dt, col) : 0.f;
      channel_affine(ep, col, s_scale[t], s_shift[t]);
    }
    consume(0, orow);
    for (int k0 = 32; k0 < K; k0 += 32) {
      issue(k0, nbr_ordered ? (in ? tr : 0) : (orow >= 0 ? orow : 0), orow >= 0 ? orow : 0);
      consume(k0, orow);
    }
    // OR over the wave (two 32-bit halves)
    uint32_t lo = static_cast<uint32_t>(m), hi = static_cast<uint32_t>(m >> 32);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      lo |= __shfl_xor(lo, off, kWave);
      hi |= __shfl_xor(hi, off, kWave);
    }
    if (lane == 0) s_mask[wave] = (static_cast<uint64_t>(hi) << 32) | lo;
  }
  __syncthreads();
  // the tile's slots, wave-uniform (scalar registers)
  const uint64_t umask_v = s_mask[0] | s_mask[1] | s_mask[2] | s_mask[3];
  const uint64_t umask =
      (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(umask_v >> 32))) << 32) |
      __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(umask_v));
  // the slots this wave's own rows use
  const uint64_t wmask_v = s_mask[wave];
  const uint64_t wmask =
      (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(wmask_v >> 32))) << 32) |
      __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(wmask_v));
  const int r0 = wave * 64 + (lane & 31);  // tile rows of this lane's A operands
  const int r1 = r0 + 32;

  // stage (k, c) -> the next stage: the next chunk of slot k, else chunk 0
  // of the tile's next slot; k == K marks the end.  Branch-free (bit scan),
  // so a loop body is one scheduling region.  k may start at -1.
  auto advance = [&](int& k, int& c) {
    const bool done = k >= K;
    const bool more_c = c + 1 < nch;
    const uint64_t above = k + 1 < 64 ? umask >> (k + 1) : 0;
    const int nk = above ? k + 1 + __builtin_ctzll(above) : K;
    const int k2 = done ? K : (more_c ? k : nk);
    c = done ? c : (more_c ? c + 1 : 0);
    k = k2;
  };

  const uint4* Wv = reinterpret_cast<const uint4*>(W);
  const int nbt_all = c_out / 32;
  // the zero row's address, held in scalar registers for the whole kernel
  // (otherwise it is reloaded from the GOT, with a wait, in every stage)
  uint64_t zero_addr = reinterpret_cast<uint64_t>(g_zero_row);
  asm volatile("" : "+s"(zero_addr));
  const uint64_t feat_addr = reinterpret_cast<uint64_t>(feat);
  const uint32_t row_bytes = static_cast<uint32_t>(c_in) * static_cast<uint32_t>(sizeof(T));

  f32x16 acc[2][NB];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[rb][nb][i] = 0.f;
  if constexpr (F32) Redo<2, NB>::pad(acc, n_out - tile0 - wave * 64);

  uint4 ring[RING][2][UB];  // gathered operands: this stage and the next
  uint4 w0, w1, w2, w3;        // this thread's share of the next weight slab

  // Loads are issued whether or not the stage exists (past the last stage they
  // re-read stage 0 or the zero row), keeping the loop body straight-line.
  auto load_w = [&](int k, int c) {
    if (k >= K) k = c = 0;
    const uint4* src = Wv + (((int64_t)k * nch + c) * nbt_all + (int64_t)nbt * NB) * UB * 64 + t;
    if (FULL || t < SLAB_VECS) w0 = src[0];
    if constexpr (WV > 1) w1 = src[256];
    if constexpr (WV > 2) w2 = src[512];
    if constexpr (WV > 3) w3 = src[768];
  };
  auto store_w = [&](uint4* dst, auto split) {
    if constexpr (decltype(split)::value) {  // vector m*256 + t: block m, vector `wave` of it
      store_split<NB>(dst, 0, wave, lane, w0);
      if constexpr (WV > 1) store_split<NB>(dst, 1, wave, lane, w1);
      if constexpr (WV > 2) store_split<NB>(dst, 2, wave, lane, w2);
      if constexpr (WV > 3) store_split<NB>(dst, 3, wave, lane, w3);
      return;
    }
    if (FULL || t < SLAB_VECS) dst[t] = w0;
    if constexpr (WV > 1) dst[256 + t] = w1;
    if constexpr (WV > 2) dst[512 + t] = w2;
    if constexpr (WV > 3) dst[768 + t] = w3;
  };
  auto load_a = [&](auto slot, int k, int c) {
    constexpr int S = decltype(slot)::value;
    const bool live = k < K;
    const int kk = live ? k : K - 1;  // reads stay in the table; dead stages use -1
    const int32_t e0 = s_nbr[kk * kTileRows + r0];
    const int32_t e1 = s_nbr[kk * kTileRows + r1];
    const int32_t j0 = live ? e0 : -1;
    const int32_t j1 = live ? e1 : -1;
    const int coff = c * CK + h * (CK / 2);
    const bool pad = coff >= c_in;  // the upper half of a half-filled last chunk
    // one 64-bit multiply-add per row, the zero row by a lane-mask select
    const uint64_t base = feat_addr + static_cast<uint64_t>(coff) * sizeof(T);
    const uint64_t a0 = static_cast<uint64_t>(static_cast<uint32_t>(j0)) * static_cast<uint64_t>(row_bytes) + base;
    const uint64_t a1 = static_cast<uint64_t>(static_cast<uint32_t>(j1)) * static_cast<uint64_t>(row_bytes) + base;
    const uint4* p0 = global_ptr<uint4>(select_lanes64(__ballot(j0 >= 0 && !pad), a0, zero_addr));
    const uint4* p1 = global_ptr<uint4>(select_lanes64(__ballot(j1 >= 0 && !pad), a1, zero_addr));
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      ring[S][0][u] = p0[u];
      ring[S][1][u] = p1[u];
    }
  };
  // Every wave takes part in every stage of its tile (the waves share the
  // weight slab through LDS), but it issues the stage's MFMAs only when one of
  // its own rows has an input through the stage's slot: the matrix core then
  // serves the other workgroup's wave on the same SIMD.  Inside a computed
  // stage, rows without input through the slot multiply the zero row and add
  // exact zeros, so skipping a stage leaves every finite result unchanged.
  auto compute = [&](auto slot, const uint4* sw, int k, auto split) {
    constexpr int S = decltype(slot)::value;
    if (k >= K || !((wmask >> k) & 1)) return;
    if constexpr (decltype(split)::value) {
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const Split8 a0 = split8(ring[S][0][2 * t2], ring[S][0][2 * t2 + 1]);
        const Split8 a1 = split8(ring[S][1][2 * t2], ring[S][1][2 * t2 + 1]);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const Split8 b = load_split<NB>(sw, nb, t2, lane);
          acc[0][nb] = mfma_split(a0, b, acc[0][nb]);
          acc[1][nb] = mfma_split(a1, b, acc[1][nb]);
        }
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const uint4 bv = sw[(nb * UB + u) * 64 + lane];
        if constexpr (F32) {
          // four 32x32x2 steps per vector: step i uses element i of A and B
          const float4 a0 = __builtin_bit_cast(float4, ring[S][0][u]);
          const float4 a1 = __builtin_bit_cast(float4, ring[S][1][u]);
          const float4 b4 = __builtin_bit_cast(float4, bv);
          acc[0][nb] = Op::run(a0.x, b4.x, acc[0][nb]);
          acc[1][nb] = Op::run(a1.x, b4.x, acc[1][nb]);
          acc[0][nb] = Op::run(a0.y, b4.y, acc[0][nb]);
          acc[1][nb] = Op::run(a1.y, b4.y, acc[1][nb]);
          acc[0][nb] = Op::run(a0.z, b4.z, acc[0][nb]);
          acc[1][nb] = Op::run(a1.z, b4.z, acc[1][nb]);
          acc[0][nb] = Op::run(a0.w, b4.w, acc[0][nb]);
          acc[1][nb] = Op::run(a1.w, b4.w, acc[1][nb]);
        } else {
          const V b = __builtin_bit_cast(V, bv);
          acc[0][nb] = Op::run(__builtin_bit_cast(V, ring[S][0][u]), b, acc[0][nb]);
          acc[1][nb] = Op::run(__builtin_bit_cast(V, ring[S][1][u]), b, acc[1][nb]);
        }
      }
    }
  };

  const float limit = F32 ? split_limit(range) : 0.f;
  const bool no_split = F32 && limit > 3.4028235e38f;  // the f32 unit computes the whole tile, below

  // Two waves per SIMD (two workgroups per CU): while one wave waits for its
  // gathers or at the barrier, the other's MFMAs keep the matrix core busy.
  // The next stage's loads are issued before this stage's MFMAs, the weights
  // first (they are waited for before the barrier, the gathered operands only
  // in the next stage); the scheduling barrier keeps the compiler from sinking
  // the loads below the MFMAs.
  auto run = [&](auto split) {
    // current stage (kc, cc) and the next one (kn, cn)
    int kc = -1, cc = nch - 1;
    advance(kc, cc);  // the tile's first slot
    int kn = kc, cn = cc;
    advance(kn, cn);
    load_w(kc, cc);
    load_a(Slot<0>{}, kc, cc);
    if (decltype(split)::value && no_split) kc = K;  // here, so that the first loads do not wait for it
    store_w(s_w[0], split);
    __syncthreads();
    auto body = [&](auto slot) {
      constexpr int S = decltype(slot)::value;
      load_w(kn, cn);                           // next stage's weights
      load_a(Slot<(S + 1) % RING>{}, kn, cn);   // next stage's operands
      __builtin_amdgcn_sched_barrier(0);
      compute(Slot<S>{}, s_w[S], kc, split);
      store_w(s_w[(S + 1) % RING], split);
      __syncthreads();
      kc = kn;
      cc = cn;
      advance(kn, cn);
    };
    while (kc < K) {
      body(Slot<0>{});
      body(Slot<1>{});
    }
  };
  run(std::bool_constant<F32>{});
  bool rerun = false;
  if constexpr (F32) rerun = __syncthreads_or(Redo<2, NB>::any(acc, limit));

  // ---- epilogue: + bias (and the affine map and ReLU when asked), round
  // once, store each output element once.
  const bool affine = ep.mean != nullptr;
  const bool relu = ep.relu != 0;
  // Each wave transposes its accumulators through LDS, PR rows at a time, so
  // that lanes write 16-byte pieces of output rows instead of single
  // elements.  32x32 accumulator layout: register i of lane l holds row
  // (i/4)*8 + (l/32)*4 + i%4 and column l%32 of the block.
  constexpr int ROW_BYTES = BN * (int)sizeof(T);
  constexpr int STRIDE = ROW_BYTES + 16;            // padded LDS row
  constexpr int CHUNKS = ROW_BYTES / 16;            // 16-byte pieces per row
  constexpr int PR = mfma_stage_rows(ROW_BYTES);    // rows staged per wave and pass
  char* stage = reinterpret_cast<char*>(s_nbr) + wave * PR * STRIDE;
  // this lane's columns' bias and batch norm, read once: the staging stores
  // go through a pointer the compiler cannot tell apart from these arrays, so
  // read in the loop they would be loaded again after every store
  float cbias[NB], cscale[NB], cshift[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int cl = nb * 32 + (lane & 31);
    cbias[nb] = s_bias[cl];
    cscale[nb] = s_scale[cl];
    cshift[nb] = s_shift[cl];
  }
#pragma unroll
  for (int pass = 0; pass < 64 / PR; ++pass) {
    if (no_split) break;
    __syncthreads();                                // the staging area is free
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int rblk = rb * 32 + (i >> 2) * 8;    // + h*4 + i%4 stays within 8 rows
        if (rblk / PR != pass) continue;
        const int row = rblk % PR + h * 4 + (i & 3);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int cl = nb * 32 + (lane & 31);
          *reinterpret_cast<T*>(stage + row * STRIDE + cl * (int)sizeof(T)) =
              from_f32<T>(finish(acc[rb][nb][i] + cbias[nb], cscale[nb], cshift[nb], affine,
                                 relu));
        }
      }
    __syncthreads();
    // every LDS read of the pass is issued before the first store waits
    constexpr int NQ = PR * CHUNKS / 64;
    int32_t orows[NQ];
    uint4 vals[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int piece = q * 64 + lane;
      const int row = piece / CHUNKS, ch = piece % CHUNKS;
      orows[q] = s_orow[wave * 64 + pass * PR + row];
      vals[q] = *reinterpret_cast<const uint4*>(stage + row * STRIDE + ch * 16);
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int ch = (q * 64 + lane) % CHUNKS;
      if (orows[q] >= 0)
        *reinterpret_cast<uint4*>(out + (int64_t)orows[q] * c_out + nbt * BN + ch * (16 / (int)sizeof(T))) = vals[q];
    }
  }
  if constexpr (F32) {
    if (rerun) {  // workgroup-uniform, and rare
      Redo<2, NB> bad;
      if (no_split) {
        bad.all();
      } else {
        const float* const flag = column_flag(W, (int64_t)K * nch * CK * c_out, c_in, c_out, nbt * BN + (lane & 31));
        const int flag_stride = c_in % 32 ? 1024 : 32;
        uint32_t vanish[2];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          const uint32_t zeros = Redo<2, NB>::zero_rows(acc[rb], flag, flag_stride);
          vanish[rb] = zeros ? vanishing_rows(feat, c_in, nbr, nbr_ordered, n_out, K,
                                              s_orow + wave * 64 + rb * 32, tile0 + wave * 64 + rb * 32,
                                              zeros)
                             : 0u;
        }
        bad.find(acc, limit, vanish);
      }
      if (!__syncthreads_or(bad.some())) return;
      // the stores above are done, and the staged slot lists are read again
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      for (int k = 0; k < K; ++k) {
        const int32_t o = s_orow[t];
        const int64_t col = nbr_ordered ? tile0 + t : (int64_t)o;
        s_nbr[k * kTileRows + t] = o < 0 ? -1 : nbr ? nbr[(int64_t)k * n_out + col] : o;
      }
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[rb][nb] = f32x16{};
      __syncthreads();
      run(std::false_type{});
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int32_t o = s_orow[wave * 64 + rb * 32 + (i >> 2) * 8 + h * 4 + (i & 3)];
            if (bad.has(rb, nb, i) && o >= 0)
              out[(int64_t)o * c_out + nbt * BN + nb * 32 + (lane & 31)] = from_f32<T>(
                  finish(acc[rb][nb][i] + cbias[nb], cscale[nb], cshift[nb], affine, relu));
          }
    }
  }
}

// ------------------------------------------------------ LDS DMA variant --
// The same tile schedule as conv_mfma_kernel, for layers whose stages are
// 128 bytes of every row (64 channels of f16/bf16 with C_in a multiple of 64,
// 32 of f32 with C_in a multiple of 32) and with a neighbour map (K > 1).
// A wave computes RB blocks of 32 rows: 64 rows (256-row tiles) on large
// layers, 32 (128-row tiles) on layers whose time is one heavy tile's chain
// of stages rather than the sum of all tiles' work.  Its operands reach LDS through direct-to-LDS loads
// (global_load_lds_dwordx4: each lane names a global address, the 16 bytes
// land at M0 + 16 * lane), which changes how the gathered rows pass the
// vector L1:
//   - each quad of lanes reads one row's 64 contiguous bytes, which the L1
//     serves as one access (an MFMA operand layout, 32 rows in 32 lanes,
//     costs one access per lane);
//   - the data skips the registers, so no transpose is needed to reach the
//     operand layout: the MFMA reads its operands from LDS in that layout.
// The weight slab and the map entries of each stage come the same way, so no
// load the compiler can see remains in the main loop.  The DMA instructions
// are issued from inline assembly: the compiler does not know they write LDS
// and adds no waits for them (given the builtin, it waits for every
// outstanding DMA before any LDS read).  The kernel waits with explicit
// s_waitcnt at three points (below).  Nothing else in these kernels reads M0.
__device__ __attribute__((aligned(16))) int32_t g_no_row[4] = {-1, -1, -1, -1};

__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p));  // low 32 bits of a shared pointer
}
__device__ __forceinline__ void dma_b128(const void* g, uint32_t m0) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(m0) : "memory");
}
__device__ __forceinline__ void dma_b32(const void* g, uint32_t m0) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" : : "v"(g), "s"(m0) : "memory");
}

// Dynamic LDS of conv_dma_kernel: two weight slabs, each wave's operand rows
// of one stage (32 * RB rows x 128 bytes) and two stages of its map entries.
// f32: one weight slab as loaded and two split ones.
template <typename T, int BN, int RB>
constexpr size_t dma_pool_bytes() {
  return (size_t)(sizeof(T) == 4 ? 4 : 2) * BN * 128 + (size_t)4 * 32 * RB * 128 + (size_t)4 * 2 * 256;
}

template <typename T, int BN, int RB>
__global__ void __launch_bounds__(256, 2) conv_dma_kernel(
    const T* __restrict__ feat, int c_in, const T* __restrict__ W, Epilogue ep,
    const int32_t* __restrict__ nbr, const int32_t* __restrict__ order, int nbr_ordered,
    int64_t n_out, int K, int c_out, T* __restrict__ out) {
  using Op = MfmaOp<T>;
  using V = typename Op::V;
  constexpr bool F32 = std::is_same<T, float>::value;
  constexpr int CK = 128 / (int)sizeof(T);   // channels of a stage: 128 bytes of each row
  constexpr int UB = 4;                      // 16-byte vectors per lane per row and stage
  constexpr int NB = BN / 32;
  constexpr int SLAB_VECS = BN * CK * (int)sizeof(T) / 16;
  constexpr int WD = SLAB_VECS / 256;        // slab DMA instructions per wave
  static_assert(SLAB_VECS % 256 == 0, "a slab splits into 1 KB pieces per wave");
  constexpr int SLAB_BYTES = SLAB_VECS * 16;
  constexpr int WR = 32 * RB;                // rows of a wave: RB blocks of 32
  constexpr int TR = 4 * WR;                 // rows of a tile
  constexpr int A_BYTES = WR * CK * (int)sizeof(T);  // one wave's rows of one stage (4 or 8 KB)
  static_assert(RB == 1 || RB == 2, "one or two 32-row blocks per wave");
  // f32 slabs are loaded into one buffer, of which each wave loads and then
  // reads only its own vectors, and split into two others that all waves read
  constexpr int SPLIT_BYTES = SLAB_BYTES * 3 / 2;
  constexpr int W_BYTES = F32 ? SLAB_BYTES + 2 * SPLIT_BYTES : 2 * SLAB_BYTES;
  static_assert(!F32 || WD == NB, "a wave's share of an f32 slab is one vector per column block");
  static_assert(A_BYTES == 4096 * RB && (size_t)W_BYTES + 4 * A_BYTES + 2048 == dma_pool_bytes<T, BN, RB>(),
                "pool layout");
  // pool: slabs [W_BYTES] (f16/bf16 two; f32 one, then two split) | operand
  // rows [4 waves][A_BYTES] | map entries [4 waves][2][64]; the output staging
  // at the end
  extern __shared__ __attribute__((aligned(16))) char pool[];
  __shared__ __attribute__((aligned(16))) int32_t s_orow[TR];
  __shared__ float s_bias[BN];
  __shared__ float s_scale[BN];
  __shared__ float s_shift[BN];
  __shared__ uint64_t s_bmask[TR / 32];  // slots used by each 32-row block

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int h = lane >> 5;
  const uint32_t wave_u = __builtin_amdgcn_readfirstlane(wave);
  const uint32_t ncol = static_cast<uint32_t>(c_out / BN);
  const uint32_t item = dealt_item(blockIdx.x, gridDim.x, ncol);
  const int64_t tile0 = static_cast<int64_t>(item / ncol) * TR;
  const int nbt = static_cast<int>(item % ncol);
  const int nch = c_in / CK;
  uint32_t range = 0;
  if constexpr (F32) range = *range_word(W, (int64_t)K * nch * CK * c_out, c_in, c_out);

  // ---- tile set-up: output rows and slot masks (the entries themselves are
  // loaded again stage by stage), as in conv_mfma_kernel; thread t < TR
  // takes tile row t, which wave t / WR computes
  {
    const int64_t tr = tile0 + t;
    const bool in = t < TR && tr < n_out;
    uint64_t m = 0;
    int32_t jv[32];
    auto issue = [&](int k0, int64_t src_row) {
      const int32_t* col = nbr + src_row;
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int k = k0 + i < K ? k0 + i : K - 1;
        jv[i] = col[(int64_t)k * n_out];
      }
    };
    auto consume = [&](int k0, int32_t orow) {
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int k = k0 + i;
        if (k < K && orow >= 0 && jv[i] >= 0) m |= uint64_t(1) << k;
      }
    };
    int32_t orow;
    if (nbr_ordered == 2) {
      // the plan's slot mask of each position follows the map as its row K
      // (K <= 32): one word per row instead of all of its entries
      const uint32_t pm = reinterpret_cast<const uint32_t*>(nbr)[(int64_t)K * n_out + (in ? tr : 0)];
      orow = in ? order[tr] : -1;
      m = orow >= 0 ? pm : 0u;
    } else if (nbr_ordered) {
      issue(0, in ? tr : 0);
      orow = in ? (order ? order[tr] : static_cast<int32_t>(tr)) : -1;
    } else {
      orow = in ? (order ? order[tr] : static_cast<int32_t>(tr)) : -1;
      issue(0, orow >= 0 ? orow : 0);
    }
    if (t < TR) s_orow[t] = orow;
    if (t < BN) {
      const int64_t col = (int64_t)nbt * BN + t;
      s_bias[t] = ep.bias ? load_param(ep.bias, ep.bias_dt, col) : 0.f;
      channel_affine(ep, col, s_scale[t], s_shift[t]);
    }
    if (nbr_ordered != 2) {
      consume(0, orow);
      for (int k0 = 32; k0 < K; k0 += 32) {
        issue(k0, nbr_ordered ? (in ? tr : 0) : (orow >= 0 ? orow : 0));
        consume(k0, orow);
      }
    }
    uint32_t lo = static_cast<uint32_t>(m), hi = static_cast<uint32_t>(m >> 32);
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {  // within each 32-lane half: one 32-row block
      lo |= __shfl_xor(lo, off, kWave);
      hi |= __shfl_xor(hi, off, kWave);
    }
    if (t < TR && t % 32 == 0) s_bmask[t / 32] = (static_cast<uint64_t>(hi) << 32) | lo;
  }
  __syncthreads();
  auto uniform64 = [](uint64_t v) {
    return (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32))) << 32) |
           __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  };
  uint64_t umask_v = 0;
#pragma unroll
  for (int b = 0; b < TR / 32; ++b) umask_v |= s_bmask[b];
  const uint64_t umask = uniform64(umask_v);
  uint64_t bmask[RB];  // slots used by each of this wave's 32-row blocks
  uint64_t wmask = 0;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    bmask[rb] = uniform64(s_bmask[wave * RB + rb]);
    wmask |= bmask[rb];
  }

  auto advance = [&](int& k, int& c) {
    const bool done = k >= K;
    const bool more_c = c + 1 < nch;
    const uint64_t above = k + 1 < 64 ? umask >> (k + 1) : 0;
    const int nk = above ? k + 1 + __builtin_ctzll(above) : K;
    const int k2 = done ? K : (more_c ? k : nk);
    c = done ? c : (more_c ? c + 1 : 0);
    k = k2;
  };
  auto uses = [&](int k) { return k < K && ((wmask >> k) & 1); };  // this wave computes slot k
  // block rb of this wave computes slot k (a block none of whose rows uses
  // slot k would only add exact zeros: its loads and MFMAs are skipped)
  auto buses = [&](int rb, int k) { return k < K && ((bmask[rb] >> k) & 1); };
  // blocks set of slot k: bit rb for block rb
  auto blocks = [&](int k) {
    int set = 0;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) set |= buses(rb, k) ? 1 << rb : 0;
    return set;
  };

  const uint4* Wv = reinterpret_cast<const uint4*>(W);
  const int nbt_all = c_out / 32;
  uint64_t zero_addr = reinterpret_cast<uint64_t>(g_zero_row);
  asm volatile("" : "+s"(zero_addr));
  const char* zero_row = reinterpret_cast<const char*>(zero_addr);
  uint64_t none_addr = reinterpret_cast<uint64_t>(g_no_row);
  asm volatile("" : "+s"(none_addr));
  const int32_t* no_row = reinterpret_cast<const int32_t*>(none_addr);

  // LDS offsets for M0 (wave-uniform) and the same places as pointers
  const uint32_t w_lds = lds_offset(pool);                                   // slab P: + P * SLAB_BYTES
  const uint32_t a_lds = w_lds + W_BYTES + wave_u * A_BYTES;
  const uint32_t e_lds = w_lds + W_BYTES + 4 * A_BYTES + wave_u * 512;  // entries P: + P * 256
  const uint4* s_w = reinterpret_cast<const uint4*>(pool);
  uint4* s_split = reinterpret_cast<uint4*>(pool + SLAB_BYTES);  // f32: split slab P: + P * SPLIT_BYTES
  const char* s_a = pool + W_BYTES + wave * A_BYTES;
  const int32_t* s_e = reinterpret_cast<const int32_t*>(pool + W_BYTES + 4 * A_BYTES + wave * 512);

  // Map entries: lane l < WR loads the entry of its wave's row l (lanes
  // past WR load -1 from the no-row array).  Operand rows:
  // DMA instruction 2g + hh covers rows 16g..16g+15 of the wave and channel
  // half hh; the quad of lanes 4q..4q+3 reads row 16g + q, lane 4q + j its
  // 16-byte piece j ^ (q >> 2), which lands in LDS at (4q + j) * 16 of the
  // instruction's 1 KB.  So piece p of row 16g + q sits at (4q + (p ^ (q >>
  // 2))) * 16, and the MFMA's reads (lanes 0..15: rows q = 0..15, one piece)
  // hit sixteen different 16-byte bank groups.
  const int32_t orow_l = lane < WR ? s_orow[wave * WR + lane] : -1;
  const int64_t col_l = nbr_ordered ? tile0 + wave * WR + lane : (int64_t)orow_l;
  const int q = lane >> 2;
  const int piece = (lane & 3) ^ (q >> 2);

  auto dma_slab = [&](int P, int k, int c) {  // the slab of stage (k, c) into buffer P
    const uint4* src = Wv + (((int64_t)k * nch + c) * nbt_all + (int64_t)nbt * NB) * UB * 64 + t;
#pragma unroll
    for (int m = 0; m < WD; ++m)
      dma_b128(src + m * 256, w_lds + P * SLAB_BYTES + (m * 256 + wave_u * 64) * 16);
  };
  // f32: this wave's vectors of the loaded slab (block m, vector `wave`), as
  // three bf16 planes, into split slab P
  auto split_slab = [&](int P) {
#pragma unroll
    for (int m = 0; m < NB; ++m)
      store_split<NB>(s_split + P * (SPLIT_BYTES / 16), m, wave, lane, s_w[m * 256 + t]);
  };
  // DMA addresses.  A present row's is one 64-bit multiply-add (row times
  // row bytes plus the lane's base), an absent row's the zero row, chosen by a
  // lane-mask select: written as a C++ select, the compiler branches around
  // the multiply, an exec-masked block with its own 64-bit arithmetic per DMA.
  // Channel half hh of a stage is the same address plus 64 bytes, added in the
  // address register: the DMA's immediate offset would move its LDS
  // destination too.
  const uint64_t row_bytes = static_cast<uint64_t>(c_in) * sizeof(T);
  const uint64_t feat_lane = reinterpret_cast<uint64_t>(feat) + piece * 16;
  const uint64_t zero_lane = reinterpret_cast<uint64_t>(zero_row) + piece * 16;
  const uint64_t live_entries = __ballot(orow_l >= 0);
  const uint64_t entry_lane = reinterpret_cast<uint64_t>(nbr + col_l);  // slot 0's entry
  const uint64_t none_lane = reinterpret_cast<uint64_t>(no_row);
  auto lane_select = [](uint64_t m, uint64_t a, uint64_t b) {
    return reinterpret_cast<const char*>(select_lanes64(m, a, b));
  };
  auto dma_entries = [&](int P, int k) {  // slot k's entries of the wave's rows into buffer P
    const uint64_t a = entry_lane + static_cast<uint64_t>(k) * static_cast<uint64_t>(n_out) * 4u;
    dma_b32(lane_select(live_entries, a, none_lane), e_lds + P * 256);
  };
  // chunk c of the rows named by entry buffer P, for the blocks in set (four
  // DMAs per 32-row block)
  auto dma_rows = [&](int P, int c, int set) {
    int32_t j[2 * RB];
#pragma unroll
    for (int g = 0; g < 2 * RB; ++g) j[g] = s_e[P * 64 + 16 * g + q];
    const uint64_t base = feat_lane + static_cast<uint64_t>(c) * (CK * sizeof(T));
#pragma unroll
    for (int g = 0; g < 2 * RB; ++g) {
      if (!((set >> (g / 2)) & 1)) continue;
      const uint64_t a = static_cast<uint64_t>(static_cast<uint32_t>(j[g])) * row_bytes + base;
      const char* src = lane_select(__ballot(j[g] >= 0), a, zero_lane);
      dma_b128(src, a_lds + (2 * g) * 1024);
      dma_b128(src + 64, a_lds + (2 * g + 1) * 1024);
    }
  };
  auto wait_vm0 = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  // all but the youngest 4 * nblk: the row DMAs of the next stage, for nblk
  // blocks (the count must be exact: anything older, the slab and the
  // entries, has to have landed)
  auto wait_rows = [](int nblk) {
    if (nblk == 2)
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else if (nblk == 1)
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  auto wait_lgkm0 = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  const int qr = lane & 15;
  auto a_read = [&](int rb, int u) {  // operand u of row block rb (rows rb*32 + lane%32)
    const int g = rb * 2 + ((lane & 31) >> 4);
    return *reinterpret_cast<const uint4*>(s_a + (2 * g + h) * 1024 + (4 * qr + (u ^ (qr >> 2))) * 16);
  };

  f32x16 acc[RB][NB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[rb][nb][i] = 0.f;
  if constexpr (F32) Redo<RB, NB>::pad(acc, n_out - tile0 - wave * WR);

  // Stage s (slab and entry buffers S = s % 2), with the three waits:
  //  1. vmcnt(0): this wave's rows of s have landed (issued in stage s - 1);
  //  2. the slab of s + 1 and the entries of s + 2 go out; the rows of s and
  //     the entries of s + 1 are read; lgkmcnt(0): the reads are done, so the
  //     rows of s + 1 may overwrite the wave's one operand buffer;
  //  3. MFMAs of s; vmcnt(4 * RB) (or 0 when no rows went out): the slab and
  //     the entries have landed, the 4 * RB row loads of s + 1 may still be in
  //     flight; the barrier then publishes the slab to every wave.
  // f32 (split): the slab of s + 1 lands in the one load buffer, whose vectors
  // each wave splits into split slab S ^ 1 between wait 3 and the barrier; the
  // wait in 2 also covers those reads, so the slab of s + 2 may land there.
  // stages s (kc, cc), s + 1 (kn, cn) and s + 2 (kp, cp)
  const float limit = F32 ? split_limit(range) : 0.f;
  const bool no_split = F32 && limit > 3.4028235e38f;  // the f32 unit computes the whole tile, below
  int kc, cc, kn, cn, kp, cp;
  auto open = [&](auto split) {
    constexpr bool SPLIT = decltype(split)::value;
    kc = -1;
    cc = nch - 1;
    advance(kc, cc);
    kn = kc;
    cn = cc;
    advance(kn, cn);
    kp = kn;
    cp = cn;
    advance(kp, cp);
    if (kc < K) {
      dma_entries(0, kc);
      dma_slab(0, kc, cc);
    }
    if (kn < K) dma_entries(1, kn);
    wait_vm0();
    if constexpr (SPLIT) {
      if (kc < K) split_slab(0);
      wait_lgkm0();
    }
    dma_rows(0, cc, blocks(kc));
    wait_vm0();
    __syncthreads();
    if (SPLIT && no_split) kc = K;  // here, so that the first loads do not wait for it
  };
  auto body = [&](auto slot, auto split) {
    constexpr int S = decltype(slot)::value;
    constexpr bool SPLIT = decltype(split)::value;
    wait_vm0();
    if (kn < K) dma_slab(SPLIT ? 0 : S ^ 1, kn, cn);
    if (kp < K) dma_entries(S, kp);
    const int cur = blocks(kc);
    uint4 a[RB][UB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      if ((cur >> rb) & 1) {
#pragma unroll
        for (int u = 0; u < UB; ++u) a[rb][u] = a_read(rb, u);
      }
    }
    wait_lgkm0();
    const int nxt = blocks(kn);
    dma_rows(S ^ 1, cn, nxt);
    // the MFMAs of the blocks that use slot kc (a wave-uniform branch per
    // block; one loop, so the register allocation is that of a full wave)
    if (SPLIT && cur) {
      const uint4* sw = s_split + S * (SPLIT_BYTES / 16);
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        Split8 as[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          if ((cur >> rb) & 1) as[rb] = split8(a[rb][2 * t2], a[rb][2 * t2 + 1]);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const Split8 b = load_split<NB>(sw, nb, t2, lane);
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
            if ((cur >> rb) & 1) acc[rb][nb] = mfma_split(as[rb], b, acc[rb][nb]);
        }
      }
    } else if (cur) {
      const uint4* sw = s_w + S * SLAB_VECS;
#pragma unroll
      for (int u = 0; u < UB; ++u) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const uint4 bv = sw[(nb * UB + u) * 64 + lane];
          if constexpr (F32) {
            // four 32x32x2 steps per vector: step e uses element e of A and B
            const float4 b4 = __builtin_bit_cast(float4, bv);
            const float bs[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int rb = 0; rb < RB; ++rb) {
                if ((cur >> rb) & 1) {
                  const float4 a4 = __builtin_bit_cast(float4, a[rb][u]);
                  const float as[4] = {a4.x, a4.y, a4.z, a4.w};
                  acc[rb][nb] = Op::run(as[e], bs[e], acc[rb][nb]);
                }
              }
          } else {
            const V b = __builtin_bit_cast(V, bv);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
              if ((cur >> rb) & 1)
                acc[rb][nb] = Op::run(__builtin_bit_cast(V, a[rb][u]), b, acc[rb][nb]);
          }
        }
      }
    }
    wait_rows(__builtin_popcount(nxt));
    if constexpr (SPLIT) {
      if (kn < K) split_slab(S ^ 1);
    }
    __syncthreads();
    kc = kn;
    cc = cn;
    kn = kp;
    cn = cp;
    advance(kp, cp);
  };
  auto run = [&](auto split) {
    open(split);
    while (kc < K) {
      body(Slot<0>{}, split);
      body(Slot<1>{}, split);
    }
    wait_vm0();
    __syncthreads();
  };
  if constexpr (F32) {
    run(std::true_type{});
  } else {
    // in place: through the lambda the compiler tests kc < K again in each
    // stage (128->128 fp16, 500k rows 307 us in place, 311 so)
    open(std::false_type{});
    while (kc < K) {
      body(Slot<0>{}, std::false_type{});
      body(Slot<1>{}, std::false_type{});
    }
    wait_vm0();
    __syncthreads();
  }
  bool rerun = false;
  if constexpr (F32) rerun = __syncthreads_or(Redo<RB, NB>::any(acc, limit));

  // ---- epilogue, as in conv_mfma_kernel, staged in the pool
  const bool affine = ep.mean != nullptr;
  const bool relu = ep.relu != 0;
  const bool whole_lines = ((int64_t)c_out * (int64_t)sizeof(T)) % 128 == 0;
  constexpr int ROW_BYTES = BN * (int)sizeof(T);
  constexpr int STRIDE = ROW_BYTES + 16;
  constexpr int CHUNKS = ROW_BYTES / 16;
  constexpr int PR = mfma_stage_rows(ROW_BYTES);
  static_assert((size_t)4 * PR * STRIDE <= dma_pool_bytes<T, BN, RB>(), "staging exceeds the pool");
  static_assert(WR % PR == 0, "whole passes");
  char* stage = pool + wave * PR * STRIDE;
  // this lane's columns' bias and batch norm in registers (see conv_mfma_kernel)
  float cbias[NB], cscale[NB], cshift[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int cl = nb * 32 + (lane & 31);
    cbias[nb] = s_bias[cl];
    cscale[nb] = s_scale[cl];
    cshift[nb] = s_shift[cl];
  }
#pragma unroll
  for (int pass = 0; pass < WR / PR; ++pass) {
    if (no_split) break;
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int rblk = rb * 32 + (i >> 2) * 8;
        if (rblk / PR != pass) continue;
        const int row = rblk % PR + h * 4 + (i & 3);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int cl = nb * 32 + (lane & 31);
          *reinterpret_cast<T*>(stage + row * STRIDE + cl * (int)sizeof(T)) =
              from_f32<T>(finish(acc[rb][nb][i] + cbias[nb], cscale[nb], cshift[nb], affine,
                                 relu));
        }
      }
    __syncthreads();
    constexpr int NQ = PR * CHUNKS / 64;
    int32_t orows[NQ];
    uint4 vals[NQ];
#pragma unroll
    for (int qq = 0; qq < NQ; ++qq) {
      const int pc = qq * 64 + lane;
      const int row = pc / CHUNKS, ch = pc % CHUNKS;
      orows[qq] = s_orow[wave * WR + pass * PR + row];
      vals[qq] = *reinterpret_cast<const uint4*>(stage + row * STRIDE + ch * 16);
    }
#pragma unroll
    for (int qq = 0; qq < NQ; ++qq) {
      const int ch = (qq * 64 + lane) % CHUNKS;
      if (orows[qq] >= 0)
        store_out(out + (int64_t)orows[qq] * c_out + nbt * BN + ch * (16 / (int)sizeof(T)), vals[qq],
                  whole_lines);
    }
  }
  if constexpr (F32) {
    if (rerun) {  // workgroup-uniform, and rare
      Redo<RB, NB> bad;
      if (no_split) {
        bad.all();
      } else {
        const float* const flag = column_flag(W, (int64_t)K * nch * CK * c_out, c_in, c_out, nbt * BN + (lane & 31));
        const int flag_stride = c_in % 32 ? 1024 : 32;
        uint32_t vanish[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          const uint32_t zeros = Redo<RB, NB>::zero_rows(acc[rb], flag, flag_stride);
          vanish[rb] = zeros ? vanishing_rows(feat, c_in, nbr, nbr_ordered, n_out, K,
                                              s_orow + wave * WR + rb * 32, tile0 + wave * WR + rb * 32,
                                              zeros)
                             : 0u;
        }
        bad.find(acc, limit, vanish);
      }
      if (!__syncthreads_or(bad.some())) return;
      wait_vm0();  // the stores above are done
      __syncthreads();
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[rb][nb] = f32x16{};
      run(std::false_type{});
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int32_t o = s_orow[wave * WR + rb * 32 + (i >> 2) * 8 + h * 4 + (i & 3)];
            if (bad.has(rb, nb, i) && o >= 0)
              out[(int64_t)o * c_out + nbt * BN + nb * 32 + (lane & 31)] = from_f32<T>(
                  finish(acc[rb][nb][i] + cbias[nb], cscale[nb], cshift[nb], affine, relu));
          }
    }
  }
}

// ------------------------------------------------- small-layer split --
// Layers too small to give half the CUs a 256-row tile (a LiDAR encoder's
// deepest layers, ~10k rows).  There the 256-row kernel is bound by one
// tile's chain of 27 stages per CU.  This kernel takes 64-row tiles and splits
// the slots over the tile's four waves: wave w takes the slots k with
// k % 4 == w that some row of the tile uses, and loads its weight operands
// straight from global memory into registers (no shared slab, no barrier per
// stage).  The waves' partial sums meet in LDS and are added in wave order,
// ((p0 + p1) + p2) + p3.  Each row's p_w is its own slots of residue w in
// ascending order (a slot the row does not use adds exact zeros), so every
// output is still a fixed sequence of fp32 operations, independent of which
// rows share its tile.  f32 operands are split into three bf16 values by the
// wave that loads them (each wave has weights of its own, so there is no slab
// to split once): 64->64, 11k rows 47.4 us on the f32 unit, 35.8 this way;
// 32->32, 25k rows 28.6 and 23.2.
template <typename T, int BN, int CK>
__global__ void __launch_bounds__(256, 2) conv_split_kernel(
    const T* __restrict__ feat, int c_in, const T* __restrict__ W, Epilogue ep,
    const int32_t* __restrict__ nbr, const int32_t* __restrict__ order, int nbr_ordered,
    int64_t n_out, int K, int c_out, T* __restrict__ out) {
  using Op = MfmaOp<T>;
  using V = typename Op::V;
  constexpr bool F32 = std::is_same<T, float>::value;
  constexpr int VPL = 16 / (int)sizeof(T);  // values per 16-byte vector
  constexpr int UB = (CK / 2) / VPL;        // vectors per lane per row and stage
  static_assert(UB * VPL * 2 == CK && UB >= 1, "chunk must split into 16-byte runs");
  constexpr int NB = BN / 32;               // 32-wide column blocks
  constexpr int SR = kSplitRows;
  constexpr int PART = 2 * NB * 16 * 64;    // floats of one wave's partial sums

  __shared__ int32_t s_orow[SR];
  __shared__ float s_bias[BN], s_scale[BN], s_shift[BN];
  __shared__ uint64_t s_mask[4];
  extern __shared__ int32_t s_dyn[];  // [K][SR] map entries, then 3 waves' partial sums
  int32_t* s_nbr = s_dyn;
  float* s_part = reinterpret_cast<float*>(s_dyn + K * SR);

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int h = lane >> 5;
  const uint32_t ncol = static_cast<uint32_t>(c_out / BN);
  const uint32_t item = dealt_item(blockIdx.x, gridDim.x, ncol);
  const int64_t tile0 = static_cast<int64_t>(item / ncol) * SR;
  const int nbt = static_cast<int>(item % ncol);
  const int nch = (c_in + CK - 1) / CK;
  uint32_t range = 0;
  if constexpr (F32) range = *range_word(W, (int64_t)K * nch * CK * c_out, c_in, c_out);

  // ---- set-up: wave w reads the map entries of its own slots for the 64
  // rows, sixteen slots at a time, all in flight before any is used; a map
  // permuted into the execution order lets the first batch go out before the
  // order lookup
  {
    const int64_t tr = tile0 + lane;
    const bool in = tr < n_out;
    uint64_t m = 0;
    int32_t jv[16];
    auto issue = [&](int i0, int64_t src_row, int32_t self) {
      if (nbr) {
        const int32_t* col = nbr + src_row;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int k = wave + 4 * (i0 + i);
          jv[i] = col[(int64_t)(k < K ? k : K - 1) * n_out];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) jv[i] = self;
      }
    };
    auto consume = [&](int i0, int32_t orow) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int k = wave + 4 * (i0 + i);
        const int32_t j = orow >= 0 ? jv[i] : -1;
        if (k < K) {
          s_nbr[k * SR + lane] = j;
          m |= (j >= 0 ? uint64_t(1) : uint64_t(0)) << k;
        }
      }
    };
    int32_t orow;
    if (nbr && nbr_ordered) {
      issue(0, in ? tr : 0, 0);
      orow = in ? (order ? order[tr] : static_cast<int32_t>(tr)) : -1;
    } else {
      orow = in ? (order ? order[tr] : static_cast<int32_t>(tr)) : -1;
      issue(0, orow >= 0 ? orow : 0, orow >= 0 ? orow : 0);
    }
    if (wave == 0) s_orow[lane] = orow;
    if (t < BN) {
      const int64_t col = (int64_t)nbt * BN + t;
      s_bias[t] = ep.bias ? load_param(ep.bias, ep.bias_dt, col) : 0.f;
      channel_affine(ep, col, s_scale[t], s_shift[t]);
    }
    consume(0, orow);
    for (int i0 = 16; wave + 4 * i0 < K; i0 += 16) {
      issue(i0, nbr_ordered ? (in ? tr : 0) : (orow >= 0 ? orow : 0), orow >= 0 ? orow : 0);
      consume(i0, orow);
    }
    uint32_t lo = static_cast<uint32_t>(m), hi = static_cast<uint32_t>(m >> 32);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      lo |= __shfl_xor(lo, off, kWave);
      hi |= __shfl_xor(hi, off, kWave);
    }
    if (lane == 0) s_mask[wave] = (static_cast<uint64_t>(hi) << 32) | lo;
  }
  __syncthreads();
  // this wave's slots (wave-uniform, scalar registers)
  const uint64_t mine_v = s_mask[wave];
  const uint64_t mine =
      (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(mine_v >> 32))) << 32) |
      __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(mine_v));
  const int r0 = lane & 31;  // tile rows of this lane's A operands
  const int r1 = r0 + 32;

  auto advance = [&](int& k, int& c) {
    const bool done = k >= K;
    const bool more_c = c + 1 < nch;
    const uint64_t above = k + 1 < 64 ? mine >> (k + 1) : 0;
    const int nk = above ? k + 1 + __builtin_ctzll(above) : K;
    const int k2 = done ? K : (more_c ? k : nk);
    c = done ? c : (more_c ? c + 1 : 0);
    k = k2;
  };

  const uint4* Wv = reinterpret_cast<const uint4*>(W);
  const int nbt_all = c_out / 32;
  uint64_t zero_addr = reinterpret_cast<uint64_t>(g_zero_row);
  asm volatile("" : "+s"(zero_addr));
  const uint64_t feat_addr = reinterpret_cast<uint64_t>(feat);
  const uint32_t row_bytes = static_cast<uint32_t>(c_in) * static_cast<uint32_t>(sizeof(T));

  f32x16 acc[2][NB];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[rb][nb][i] = 0.f;
  if constexpr (F32) Redo<2, NB>::pad(acc, n_out - tile0);

  uint4 ring[2][2][UB];   // gathered operands: this stage and the next
  uint4 bring[2][NB][UB];  // weight operands: this stage and the next

  // Loads are issued whether or not the stage exists (past the last stage they
  // re-read stage 0 or the zero row), keeping the loop body straight-line.
  auto load_b = [&](auto slot, int k, int c) {
    constexpr int S = decltype(slot)::value;
    if (k >= K) k = c = 0;
    const uint4* src = Wv + (((int64_t)k * nch + c) * nbt_all + (int64_t)nbt * NB) * UB * 64 + lane;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int u = 0; u < UB; ++u) bring[S][nb][u] = src[(nb * UB + u) * 64];
  };
  auto load_a = [&](auto slot, int k, int c) {
    constexpr int S = decltype(slot)::value;
    const bool live = k < K;
    const int kk = live ? k : K - 1;
    const int32_t e0 = s_nbr[kk * SR + r0];
    const int32_t e1 = s_nbr[kk * SR + r1];
    const int32_t j0 = live ? e0 : -1;
    const int32_t j1 = live ? e1 : -1;
    const int coff = c * CK + h * (CK / 2);
    const bool pad = coff >= c_in;  // the upper half of a half-filled last chunk
    // one 64-bit multiply-add per row, the zero row by a lane-mask select
    const uint64_t base = feat_addr + static_cast<uint64_t>(coff) * sizeof(T);
    const uint64_t a0 = static_cast<uint64_t>(static_cast<uint32_t>(j0)) * static_cast<uint64_t>(row_bytes) + base;
    const uint64_t a1 = static_cast<uint64_t>(static_cast<uint32_t>(j1)) * static_cast<uint64_t>(row_bytes) + base;
    const uint4* p0 = global_ptr<uint4>(select_lanes64(__ballot(j0 >= 0 && !pad), a0, zero_addr));
    const uint4* p1 = global_ptr<uint4>(select_lanes64(__ballot(j1 >= 0 && !pad), a1, zero_addr));
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      ring[S][0][u] = p0[u];
      ring[S][1][u] = p1[u];
    }
  };
  auto compute = [&](auto slot, int k, auto split) {
    constexpr int S = decltype(slot)::value;
    if (k >= K) return;
    if constexpr (decltype(split)::value) {
#pragma unroll
      for (int t2 = 0; t2 < UB / 2; ++t2) {
        const Split8 a0 = split8(ring[S][0][2 * t2], ring[S][0][2 * t2 + 1]);
        const Split8 a1 = split8(ring[S][1][2 * t2], ring[S][1][2 * t2 + 1]);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const Split8 b = split8(bring[S][nb][2 * t2], bring[S][nb][2 * t2 + 1]);
          acc[0][nb] = mfma_split(a0, b, acc[0][nb]);
          acc[1][nb] = mfma_split(a1, b, acc[1][nb]);
        }
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const uint4 bv = bring[S][nb][u];
        if constexpr (F32) {
          const float4 a0 = __builtin_bit_cast(float4, ring[S][0][u]);
          const float4 a1 = __builtin_bit_cast(float4, ring[S][1][u]);
          const float4 b4 = __builtin_bit_cast(float4, bv);
          acc[0][nb] = Op::run(a0.x, b4.x, acc[0][nb]);
          acc[1][nb] = Op::run(a1.x, b4.x, acc[1][nb]);
          acc[0][nb] = Op::run(a0.y, b4.y, acc[0][nb]);
          acc[1][nb] = Op::run(a1.y, b4.y, acc[1][nb]);
          acc[0][nb] = Op::run(a0.z, b4.z, acc[0][nb]);
          acc[1][nb] = Op::run(a1.z, b4.z, acc[1][nb]);
          acc[0][nb] = Op::run(a0.w, b4.w, acc[0][nb]);
          acc[1][nb] = Op::run(a1.w, b4.w, acc[1][nb]);
        } else {
          const V b = __builtin_bit_cast(V, bv);
          acc[0][nb] = Op::run(__builtin_bit_cast(V, ring[S][0][u]), b, acc[0][nb]);
          acc[1][nb] = Op::run(__builtin_bit_cast(V, ring[S][1][u]), b, acc[1][nb]);
        }
      }
    }
  };

  const float limit = F32 ? split_limit(range) : 0.f;
  const bool no_split = F32 && limit > 3.4028235e38f;  // the f32 unit computes the whole tile, below
  auto run = [&](auto split) {
    int kc = -1, cc = nch - 1;
    advance(kc, cc);  // this wave's first slot
    int kn = kc, cn = cc;
    advance(kn, cn);
    load_b(Slot<0>{}, kc, cc);
    load_a(Slot<0>{}, kc, cc);
    if (decltype(split)::value && no_split) kc = K;  // here, so that the first loads do not wait for it
    auto body = [&](auto slot) {
      constexpr int S = decltype(slot)::value;
      load_b(Slot<(S + 1) % 2>{}, kn, cn);  // next stage's weights
      load_a(Slot<(S + 1) % 2>{}, kn, cn);  // and operands
      __builtin_amdgcn_sched_barrier(0);
      compute(Slot<S>{}, kc, split);
      kc = kn;
      cc = cn;
      advance(kn, cn);
    };
    while (kc < K) {
      body(Slot<0>{});
      body(Slot<1>{});
    }
    // waves 1-3 hand their partial sums to wave 0, which adds them in wave order
    if (wave > 0) {
      float* dst = s_part + (wave - 1) * PART;
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int i = 0; i < 16; ++i) dst[((rb * NB + nb) * 16 + i) * 64 + lane] = acc[rb][nb][i];
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            acc[rb][nb][i] += s_part[w * PART + ((rb * NB + nb) * 16 + i) * 64 + lane];
  };
  // wave 0 stores the elements that `which` picks.  32x32 accumulator layout:
  // register i of lane l holds row (i/4)*8 + (l/32)*4 + i%4 and column l%32 of
  // the block.
  auto store = [&](auto which) {
    const bool affine = ep.mean != nullptr;
    const bool relu = ep.relu != 0;
    T* const dst = out + nbt * BN + (lane & 31);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = rb * 32 + (i >> 2) * 8 + h * 4 + (i & 3);
        const int32_t orow = s_orow[row];
        if (orow < 0) continue;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int cl = nb * 32 + (lane & 31);
          if (which(rb, nb, i))
            dst[(int64_t)orow * c_out + nb * 32] =
                from_f32<T>(finish(acc[rb][nb][i] + s_bias[cl], s_scale[cl], s_shift[cl], affine, relu));
        }
      }
  };
  auto every = [](int, int, int) { return true; };
  if constexpr (!F32) {
    run(std::false_type{});
    if (wave != 0) return;
    store(every);
  } else {
    run(std::true_type{});
    if (wave == 0 && !no_split) store(every);
    if (!__syncthreads_or(wave == 0 && Redo<2, NB>::any(acc, limit))) return;
    Redo<2, NB> bad;
    if (no_split) {
      bad.all();
    } else if (wave == 0) {
      const float* const flag = column_flag(W, (int64_t)K * nch * CK * c_out, c_in, c_out, nbt * BN + (lane & 31));
      const int flag_stride = c_in % 32 ? 1024 : 32;
      uint32_t vanish[2];
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const uint32_t zeros = Redo<2, NB>::zero_rows(acc[rb], flag, flag_stride);
        vanish[rb] = zeros ? vanishing_rows(feat, c_in, nbr, nbr_ordered, n_out, K, s_orow + rb * 32,
                                            tile0 + rb * 32, zeros)
                           : 0u;
      }
      bad.find(acc, limit, vanish);
    }
    if (!__syncthreads_or(wave == 0 && bad.some())) return;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[rb][nb] = f32x16{};
    run(std::false_type{});
    if (wave == 0) store([&](int rb, int nb, int i) { return bad.has(rb, nb, i); });
  }
}

// --------------------------------------------------------- narrow MFMA --
// Layers that the 32x32 tile does not take.  The reduction runs over
// r = k * cp + c (slot k, channel c, cp = C_in rounded up to a multiple of 4)
// in steps of 4*LV values, LV = 16 / sizeof(T): one v_mfma_f32_16x16x32 for
// f16/bf16, four v_mfma_f32_16x16x4_f32 for f32.  A wave owns 16 output rows
// and NT 16-column tiles.  Lane l supplies row l%16's values
// r = 4*LV*i + LV*(l/16) .. +LV-1 of step i, gathered straight from the input
// rows the map names (zeros for absent neighbours and padding), in one of
// three forms:
//   * kWhole, C_in % 4 == 0 and aligned features: one 16-byte piece, or for
//     f16/bf16 with C_in % 8 == 4 two 8-byte pieces of four channels each;
//   * kRagged, any C_in and element-aligned features: the same pieces, read
//     unaligned.  A piece may run past its row's end (the channels past C_in
//     are cleared, whatever they hold) but never past the buffer's: it then
//     starts earlier and is shifted back into place;
//   * kSingle, feature buffers smaller than one piece: element by element.
// C_out that is no multiple of 16 has zero-weight columns that are not stored.
// These widths ran one row per lane on the vector ALU before, 20 class scores
// with every feature row read by five column groups.  Before and after: 96 -> 20
// f16 over 120k rows 70 -> 14 us a pass; a 3 -> 32 f16 layer with 125 slots over
// 80k rows, its launch 121 -> 29 us; 5 -> 16 and 16 -> 16 f16 over 60k LiDAR
// rows, a pass with the build 90 -> 81 us.
// A group of steps loads all its map entries, then all its gathers and
// weight operands, then runs its MFMAs, so a 3x3x3 layer with C_in = 4 (four
// steps) costs two dependent memory round trips.  Each output is the same
// sequence of MFMAs whatever the row order, so results are bitwise
// reproducible and independent of the execution order.
typedef float f32x4 __attribute__((ext_vector_type(4)));

// One step on 16-byte operands per lane: a 16x16x32 MFMA for f16/bf16, four
// 16x16x4 MFMAs for f32 (MFMA e takes element e of every lane's vectors).
template <typename T> struct Mfma16;
template <> struct Mfma16<__half> {
  static __device__ __forceinline__ f32x4 step(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma16<__hip_bfloat16> {
  static __device__ __forceinline__ f32x4 step(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma16<float> {
  static __device__ __forceinline__ f32x4 step(uint4 a, uint4 b, f32x4 c) {
    const float4 fa = __builtin_bit_cast(float4, a);
    const float4 fb = __builtin_bit_cast(float4, b);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa.x, fb.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa.y, fb.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa.z, fb.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(fa.w, fb.w, c, 0, 0, 0);
  }
};

constexpr int kNarrowRows = 16;  // output rows per wave (the MFMA's M)

enum NarrowRead { kWhole = 0, kRagged = 1, kSingle = 2 };

template <int BYTES> struct VecOf;
template <> struct VecOf<16> { using type = uint4; };
template <> struct VecOf<8> { using type = uint2; };
template <> struct VecOf<4> { using type = uint32_t; };
template <> struct VecOf<2> { using type = uint16_t; };

// The NP pieces of a lane and step as one operand vector.
__device__ __forceinline__ uint4 join_pieces(const uint4* v) { return v[0]; }
__device__ __forceinline__ uint4 join_pieces(const uint2* v) {
  return make_uint4(v[0].x, v[0].y, v[1].x, v[1].y);
}
__device__ __forceinline__ uint4 join_pieces(const uint32_t* v) {
  return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint4 join_pieces(const uint16_t* v) {
  return make_uint4(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16,
                    v[4] | (uint32_t)v[5] << 16, v[6] | (uint32_t)v[7] << 16);
}

// Four channels read at the byte address p: shifted down by `shift` bytes, of
// which the first `bytes` are wanted and the rest cleared.
__device__ __forceinline__ uint2 ragged_piece(const char* p, uint32_t shift, uint32_t bytes,
                                              uint2) {
  uint64_t v;
  __builtin_memcpy(&v, p, 8);
  v >>= 8 * shift;
  v &= bytes >= 8 ? ~0ull : (1ull << (8 * bytes)) - 1;
  return make_uint2(static_cast<uint32_t>(v), static_cast<uint32_t>(v >> 32));
}
__device__ __forceinline__ uint4 ragged_piece(const char* p, uint32_t shift, uint32_t bytes,
                                              uint4) {
  uint4 v;
  __builtin_memcpy(&v, p, 16);
  if (shift & 8) v = make_uint4(v.z, v.w, 0u, 0u);
  if (shift & 4) v = make_uint4(v.y, v.z, v.w, 0u);
  return make_uint4(bytes > 0 ? v.x : 0u, bytes > 4 ? v.y : 0u, bytes > 8 ? v.z : 0u,
                    bytes > 12 ? v.w : 0u);
}

// Sixteen bytes of packed weights, of which only the words need be aligned.
__device__ __forceinline__ uint4 load_words(const uint4* p) {
  uint4 v;
  __builtin_memcpy(&v, __builtin_assume_aligned(reinterpret_cast<const uint32_t*>(p), 4), 16);
  return v;
}

// Entry i of a per-channel parameter, or dflt where the pointer is null.  The
// load is issued either way (from the zero row), so a run of these issues
// back to back instead of one branch and wait at a time.
__device__ __forceinline__ float param_or(const void* p, int dt, int64_t i, float dflt) {
  const float v = load_param(p ? p : static_cast<const void*>(g_zero_row), dt, p ? i : 0);
  return p ? v : dflt;
}

// PIECE: bytes per gather (16 or 8, or one element); NT: 16-column tiles per
// wave.  A group is SG steps: 8 / NT gathers and 32 / NP weight registers per
// lane.
// B32: layers whose features and map stay below 2^31 bytes (NarrowB32::fits).
// The gathers and map loads then go through buffer loads with 32-bit
// offsets: an offset past the buffer's end reads zeros, which gives absent
// neighbours their zero row and the identity map (a buffer of no bytes) its
// zero entries, and the slot of a reduction index is one multiply-high by
// cp's rounded-up reciprocal.  The 64-bit addresses and the division cost
// each step about three times the vector instructions (a wave of the 20k-row
// 16->16 fp32 layer executed 1,623 of them for 108 MFMAs).  Both forms sum
// the same products in the same order.
struct NarrowB32 {
  uint32_t feat_bytes;  // n_in * C_in * sizeof(T)
  uint32_t map_bytes;   // K * n_out * 4, 0 for the identity map
  uint32_t row_bytes;   // C_in * sizeof(T)
  uint32_t cp_mag;      // ceil(2^32 / cp)
  static bool fits(int64_t n_in, int c_in, int elem, int64_t n_out, int K, int64_t nsteps,
                   int lv) {
    const int64_t r_end = 4 * lv * nsteps;  // reduction indices stay below this
    return n_in * c_in * elem < (int64_t(1) << 31) && (int64_t)K * n_out * 4 < (int64_t(1) << 31) &&
           n_in < (int64_t(1) << 24) && (int64_t)c_in * elem < (int64_t(1) << 24) &&
           r_end * narrow_cp(c_in) < (int64_t(1) << 32);
  }
};
constexpr int kBufferWord3 = 0x00020000;  // raw buffer, 32-bit data (gfx9 family)

template <typename T, int READ, int PIECE, int NT, bool B32>
__global__ void __launch_bounds__(256) conv_narrow_kernel(
    const T* __restrict__ feat, int64_t feat_bytes, int c_in, const T* __restrict__ W,
    const uint32_t* __restrict__ form, Epilogue ep, const int32_t* __restrict__ nbr,
    const int32_t* __restrict__ order, int nbr_ordered, int64_t n_out, int K, int c_out, int nsteps,
    NarrowB32 nb32, T* __restrict__ out) {
  using Op = Mfma16<T>;
  using Piece = typename VecOf<PIECE>::type;
  constexpr int LV = 16 / (int)sizeof(T);      // reduction values per lane and step
  constexpr int VPP = PIECE / (int)sizeof(T);  // values per piece
  constexpr int NP = 16 / PIECE;               // pieces per lane and step
  constexpr int SG = 8 / (NP * NT) > 0 ? 8 / (NP * NT) : 1;
  static_assert(READ == kSingle ? PIECE == (int)sizeof(T)
                                : PIECE == 16 || (PIECE == 8 && sizeof(T) == 2), "piece size");
  static_assert(READ != kRagged || VPP == 4, "a ragged piece is four channels");
  const int lane = threadIdx.x & 63;
  const uint32_t q = lane >> 4;  // which 8 values of a step this lane supplies
  const int rl = lane & 15;      // A row, B and D column of this lane
  const int64_t p0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * kNarrowRows;
  const int64_t pa = p0 + rl;  // processing position of this lane's A row
  const bool va = pa < n_out;
  const int32_t oa = va ? (order ? order[pa] : static_cast<int32_t>(pa)) : 0;
  // its column of the map; lanes past the last row read column 0 (their
  // loads are issued too, and then discarded)
  const int64_t col = va ? (nbr_ordered ? pa : oa) : 0;
  const int nt_all = (c_out + 15) / 16;
  const int nt0 = blockIdx.y * NT;
  const uint32_t cp = READ == kWhole ? c_in : (c_in + 3) / 4 * 4;
  uint64_t zero_addr = reinterpret_cast<uint64_t>(g_zero_row);
  asm volatile("" : "+s"(zero_addr));
  // global (not flat) loads for both the gathered rows and the zero row
  const Piece* zero_piece =
      (const Piece*)reinterpret_cast<const __attribute__((address_space(1))) Piece*>(zero_addr);
  const uint4* Wv = reinterpret_cast<const uint4*>(W);
  uint32_t form_word = kNarrowForm;  // the weights' form: the buffer's last word

  // the epilogue's per-column parameters: loaded before the main loop (their
  // latency overlaps the map loads), combined after it
  float bias[NT], mean[NT], var[NT], gamma[NT], beta[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int col_n = (nt0 + n) * 16 + rl;
    const int co = col_n < c_out ? col_n : c_out - 1;  // padding columns are not stored
    bias[n] = param_or(ep.bias, ep.bias_dt, co, 0.f);
    mean[n] = param_or(ep.mean, ep.bn_dt, co, 0.f);
    var[n] = param_or(ep.var, ep.bn_dt, co, 1.f);
    gamma[n] = param_or(ep.gamma, ep.bn_dt, co, 1.f);
    beta[n] = param_or(ep.beta, ep.bn_dt, co, 0.f);
  }
  // The identity map (1x1x1 layers): its map loads read 0 from the zero row
  // and its row is added on, so the loop has no branch on which map it reads.
  const int32_t* map = nbr ? nbr : reinterpret_cast<const int32_t*>(g_zero_row);
  const int64_t map_mask = nbr ? ~int64_t(0) : 0;
  const int32_t ident_row = nbr ? 0 : oa;

  f32x4 acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};

  // B32: buffers over the features and the map (no bytes for the identity map)
  const __amdgpu_buffer_rsrc_t feat_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(feat), 0, static_cast<int>(nb32.feat_bytes), kBufferWord3);
  const __amdgpu_buffer_rsrc_t map_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int32_t*>(nbr), 0, static_cast<int>(nb32.map_bytes), kBufferWord3);
  const uint32_t col4 = static_cast<uint32_t>(col) * 4u;
  const uint32_t n_out4 = static_cast<uint32_t>(n_out) * 4u;

  for (int i0 = 0; i0 < nsteps; i0 += SG) {
    int32_t j[SG * NP];
    uint32_t ch[SG * NP];
#pragma unroll
    for (int u = 0; u < SG * NP; ++u) {
      const int i = i0 + u / NP;
      const uint32_t r = 4u * LV * static_cast<uint32_t>(i) + LV * q + VPP * static_cast<uint32_t>(u % NP);
      const uint32_t k = B32 ? __umulhi(r, nb32.cp_mag) : r / cp;
      ch[u] = r - k * cp;
      const bool live = va && i < nsteps && k < static_cast<uint32_t>(K) &&
                        (READ != kSingle || ch[u] < static_cast<uint32_t>(c_in));
      // every lane loads (dead ones from slot K-1 of their column), so the
      // group's map loads issue back to back; dead lanes then use -1
      int32_t e;
      if constexpr (B32) {
        const uint32_t kk = live ? k : static_cast<uint32_t>(K - 1);
        e = __builtin_amdgcn_raw_buffer_load_b32(map_rs, kk * n_out4 + col4, 0, 0);
      } else {
        const int64_t kk = live ? k : K - 1;
        e = map[(kk * n_out + col) & map_mask];
      }
      // an OR rather than a select: the load's value is then always used, and
      // the compiler keeps it unconditional instead of branching around it
      j[u] = (e + ident_row) | (live ? 0 : -1);
    }
    Piece v[SG * NP];
#pragma unroll
    for (int u = 0; u < SG * NP; ++u) {
      if constexpr (READ == kSingle) {
        const T* src = j[u] >= 0 ? feat + (int64_t)j[u] * c_in + ch[u]
                                 : reinterpret_cast<const T*>(zero_piece);
        v[u] = __builtin_bit_cast(Piece, *src);
      } else if constexpr (READ == kRagged) {
        // the wanted channels of this piece, none of an absent row's; a piece
        // that would end past the buffer starts earlier (feat_bytes >= PIECE)
        const uint32_t bytes = j[u] >= 0 ? (static_cast<uint32_t>(c_in) - ch[u]) * (uint32_t)sizeof(T) : 0u;
        const uint32_t row = j[u] >= 0 ? static_cast<uint32_t>(j[u]) : 0u;
        if constexpr (B32) {
          const uint32_t off = __umul24(row, nb32.row_bytes) + ch[u] * static_cast<uint32_t>(sizeof(T));
          const uint32_t last = nb32.feat_bytes - PIECE;
          const uint32_t at = off < last ? off : last;
          v[u] = ragged_piece(reinterpret_cast<const char*>(feat) + at, off - at, bytes, Piece{});
        } else {
          const int64_t off = ((int64_t)row * c_in + ch[u]) * (int64_t)sizeof(T);
          const int64_t last = feat_bytes - PIECE;
          const int64_t at = off < last ? off : last;
          v[u] = ragged_piece(reinterpret_cast<const char*>(feat) + at,
                              static_cast<uint32_t>(off - at), bytes, Piece{});
        }
      } else if constexpr (B32) {
        // absent rows read past the buffer's end: zeros
        const uint32_t off = j[u] >= 0 ? __umul24(static_cast<uint32_t>(j[u]), nb32.row_bytes) +
                                             ch[u] * static_cast<uint32_t>(sizeof(T))
                                       : 0x80000000u;
        if constexpr (PIECE == 16)
          v[u] = __builtin_bit_cast(Piece, __builtin_amdgcn_raw_buffer_load_b128(feat_rs, off, 0, 0));
        else
          v[u] = __builtin_bit_cast(Piece, __builtin_amdgcn_raw_buffer_load_b64(feat_rs, off, 0, 0));
      } else {
        const Piece* src = j[u] >= 0
                               ? reinterpret_cast<const Piece*>(feat + (int64_t)j[u] * c_in + ch[u])
                               : zero_piece;
        v[u] = *src;
      }
    }
    uint4 b[SG][NT];
#pragma unroll
    for (int u = 0; u < SG; ++u)
#pragma unroll
      for (int n = 0; n < NT; ++n)
        b[u][n] = i0 + u < nsteps
                      ? load_words(Wv + ((int64_t)(i0 + u) * nt_all + nt0 + n) * 64 + lane)
                      : make_uint4(0u, 0u, 0u, 0u);
    if constexpr (sizeof(T) == 2) {
      // Behind the group's loads, which it then shares the wait with; it is used
      // after the loop, whose sums over f32 weights (reads inside the buffer
      // too) are dropped.  Loaded at the kernel's start it is waited for with the
      // kernel's other scalars: 96 -> 20, 120k rows 13.95 -> 14.3 us a pass, 14.0
      // so.  The barrier keeps the compiler from moving it there.
      const uint32_t* f = form;
      asm volatile("" : "+s"(f));
      form_word = *f;
    }
#pragma unroll
    for (int u = 0; u < SG; ++u) {
      if (i0 + u >= nsteps) break;
      const uint4 a = join_pieces(v + u * NP);
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n] = Op::step(a, b[u][n], acc[n]);
    }
  }

  // f32 weights under 16-bit features (rare: a program packs weights of the
  // features' type): each output's products one by one in f32, slots and channels
  // ascending
  if (sizeof(T) == 2 && (c_in % 4 || c_out % 16) && form_word != kNarrowForm) {
    const float* const wf = reinterpret_cast<const float*>(W);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t p = p0 + 4 * q + e;
      const int64_t o = p < n_out ? (order ? order[p] : p) : 0;
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n][e] = 0.f;
      for (int k = 0; k < K && p < n_out; ++k) {
        const int64_t j = nbr ? nbr[(int64_t)k * n_out + (nbr_ordered ? p : o)] : o;
        if (j < 0) continue;
        for (int c = 0; c < c_in; ++c) {
          const float x = to_f32<T>(feat[j * c_in + c]);
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            const int co = (nt0 + n) * 16 + rl;
            acc[n][e] = fmaf(x, wf[((int64_t)k * c_in + c) * c_out + (co < c_out ? co : c_out - 1)],
                             acc[n][e]);
          }
        }
      }
    }
  }

  // D: lane l holds rows 4(l/16) + 0..3 of the wave's 16, column l%16; the
  // output row of wave row r is lane r's oa
  int32_t orow[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 4 * static_cast<int>(q) + e;
    const int32_t o = __shfl(oa, r, kWave);
    orow[e] = p0 + r < n_out ? o : -1;
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int co = (nt0 + n) * 16 + rl;
    // the batch norm as v * sc + sh, in the order channel_affine computes it
    const float sc = gamma[n] * (1.f / sqrtf(var[n] + ep.eps));
    const float sh = beta[n] - mean[n] * sc;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (orow[e] >= 0 && co < c_out)
        out[(int64_t)orow[e] * c_out + co] = from_f32<T>(
            finish(acc[n][e] + bias[n], sc, sh, ep.mean != nullptr, ep.relu != 0));
  }
}

template <typename T, int BN, int CK>
int launch_mfma(const void* feat, int c_in, const void* W, const Epilogue& ep,
                const int32_t* nbr, const int32_t* order, int nbr_ordered, int64_t n_out, int K,
                int c_out, void* out, hipStream_t s) {
  const int64_t items = ceil_div(n_out, kTileRows) * (c_out / BN);
  TSC_REQUIRE(items < (int64_t(1) << 31), "conv: %lld workgroups exceed the grid limit",
              static_cast<long long>(items));
  dim3 grid(static_cast<unsigned>(items));
  // dynamic LDS: the tile's slot lists, later reused to stage the output
  const size_t lds_nbr = (size_t)K * kTileRows * sizeof(int32_t);
  const int row_bytes = BN * (int)sizeof(T);
  const size_t lds_out = (size_t)4 * mfma_stage_rows(row_bytes) * (row_bytes + 16);  // 4 waves
  const size_t lds = lds_nbr > lds_out ? lds_nbr : lds_out;
  // with the weight slabs it may pass 64 KB (K <= 64 slots)
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&conv_mfma_kernel<T, BN, CK>),
                                 64 * kTileRows * (int)sizeof(int32_t)))
    return rc;
  conv_mfma_kernel<T, BN, CK><<<grid, 256, lds, s>>>(
      static_cast<const T*>(feat), c_in, static_cast<const T*>(W), ep, nbr, order,
      nbr_ordered, n_out, K, c_out, static_cast<T*>(out));
  TSC_LAUNCH_CHECK("conv_mfma");
  return 0;
}

template <typename T, int BN, int RB>
int launch_dma(const void* feat, int c_in, const void* W, const Epilogue& ep,
               const int32_t* nbr, const int32_t* order, int nbr_ordered, int64_t n_out, int K,
               int c_out, void* out, hipStream_t s) {
  const int64_t items = ceil_div(n_out, 128 * RB) * (c_out / BN);
  TSC_REQUIRE(items < (int64_t(1) << 31), "conv: %lld workgroups exceed the grid limit",
              static_cast<long long>(items));
  constexpr int CK = 128 / (int)sizeof(T);
  TSC_REQUIRE(nbr != nullptr && c_in % CK == 0, "conv: the DMA kernel needs a map and C_in %% %d == 0",
              CK);
  constexpr size_t pool = dma_pool_bytes<T, BN, RB>();
  // more than 64 KB of dynamic LDS for the larger tiles
  if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&conv_dma_kernel<T, BN, RB>),
                                 static_cast<int>(pool)))
    return rc;
  conv_dma_kernel<T, BN, RB><<<dim3(static_cast<unsigned>(items)), 256, pool, s>>>(
      static_cast<const T*>(feat), c_in, static_cast<const T*>(W), ep, nbr, order, nbr_ordered,
      n_out, K, c_out, static_cast<T*>(out));
  TSC_LAUNCH_CHECK("conv_dma");
  return 0;
}

template <typename T, int BN, int CK>
int launch_split(const void* feat, int c_in, const void* W, const Epilogue& ep,
                 const int32_t* nbr, const int32_t* order, int nbr_ordered, int64_t n_out, int K,
                 int c_out, void* out, hipStream_t s) {
  const int64_t items = ceil_div(n_out, kSplitRows) * (c_out / BN);
  TSC_REQUIRE(items < (int64_t(1) << 31), "conv: %lld workgroups exceed the grid limit",
              static_cast<long long>(items));
  // dynamic LDS: the tile's map entries, then three waves' partial sums
  const size_t lds = (size_t)K * kSplitRows * sizeof(int32_t) +
                     (size_t)3 * 2 * (BN / 32) * 16 * 64 * sizeof(float);
  conv_split_kernel<T, BN, CK><<<dim3(static_cast<unsigned>(items)), 256, lds, s>>>(
      static_cast<const T*>(feat), c_in, static_cast<const T*>(W), ep, nbr, order,
      nbr_ordered, n_out, K, c_out, static_cast<T*>(out));
  TSC_LAUNCH_CHECK("conv_split");
  return 0;
}

// Which 32x32-tile kernel runs a layer, and with which column tile width.
struct MfmaChoice {
  int bn;      // column tile width
  int ck;      // input-channel chunk of one stage
  bool split;  // the 64-row slot-split kernel instead of the 256-row one
  bool dma;    // the 256-row kernel's direct-to-LDS variant
  int rb;      // its 32-row blocks per wave (tiles of 128 * rb rows)
};

// Layers of at least this many 256-row tiles always run the direct-to-LDS
// kernel at 64 rows per wave: the sum of all tiles' work bounds them, and two
// 64-row waves share each weight slab read from LDS (the 500k-row 128->128
// fp16 layer, 1954 tiles: 327 us, 339 us at 32 rows per wave).
constexpr int64_t kShortTiles = 1024;
constexpr int64_t kCus = 256;

// Workgroups of the direct-to-LDS kernel a CU's 160 KB of LDS hold (its pool
// and up to 3 KB of static arrays).
int dma_per_cu(int dtype, int bn, int rb) {
  return 163840 / ((dtype == TSC_F32 ? 4 : 2) * bn * 128 + 16384 * rb + 2048 + 3072);
}

// Column tile width, kernel and rows per wave of a 32x32-tile layer.  Below a
// few workgroups per CU a layer's time is one tile's chain of stages (27 slots
// x the channel chunks), which a narrower or shorter tile shortens, against
// repeated gathers per column tile; the lines are where the two meet, from a
// sweep of every width and row count over layers of 16-768 channels and 3k-400k
// rows, all dtypes.  Times in us are of one launch from a captured graph.
//   * Column tile.  The widest that leaves enough tiles: direct-to-LDS f16/bf16
//     128-row tiles, 400 at 128 columns and 180 at 64; f32 512 at 64 (its
//     stages are longer); other layers 256-row tiles, 360 at 128 columns and
//     128 at 64 (300 for f32 and for K < 12).  64->64 fp16: 120k rows 59 -> 41
//     with 64 columns for 32, 16k rows 18.7 with 64 and 16.2 with 32; 128->128
//     fp16: 70k rows 96 at 64 and 89 at 128, 40k rows 56 and 59; 192->192, 40k
//     rows 142 -> 107; 64->64 f32: 70k rows 138 -> 118, 40k rows 88 at 64 and
//     79 at 32.  Short slot lists (K < 8) keep the line at 512 256-row tiles.
//   * Slot split (conv_split_kernel, 64-row tiles of 32 columns, K >= 8) up to
//     one tile per CU for f16/bf16 layers the direct-to-LDS kernel takes
//     (64->64, 8k rows 14.1 against 15.7; 10k rows 18.5 against 15.9), two for
//     a single column tile (inverse 64->32, 30k rows 15.2 against 17.1), for
//     strided and inverse layers, whose rows use few slots (inverse 128->64,
//     15k rows 21.4 against 27.8; strided 64->128, 6k rows 15.5 against 16.6) and
//     for K < 12 (32->64 with 8 slots, 20k rows 10.2 against 8.6), and two and a
//     half for the other f16/bf16 layers (32->32, 28k rows 12.8 against 15.7;
//     48->64, 20k rows 20.2 against 24.3, 28k 25.1 against 24.5) and for f32
//     (32->32, 40k rows 31.5 against 33.3, 50k 36.9 against 33.6; 64->64, 18k rows
//     44.5 against 59.4; 128->128, 9k rows 76 against 113).  f32 strided and
//     inverse layers and those of the register-gather kernel with more than one
//     column tile up to four (inverse 128->64, 24k rows 36.4 against 46.0;
//     48->96, 16k rows 44.6 against 65.9; 16->64, 32k rows 36.3 against 37.4).
//     SubM layers of the direct-to-LDS kernel would gain up to five (64->64, 40k
//     rows 72.9 against 78.4); their line is not where the times cross, but below
//     the 752 tiles of a 64->128 layer of 12k rows, whose sums a test compares
//     bit for bit with the 256-row kernels'.
//   * Rows per wave of the direct-to-LDS kernel: 32 (128-row tiles) below
//     kShortTiles 256-row tiles, as halving a wave's rows halves each stage's
//     MFMAs and the smaller pool lets more workgroups share a CU; but 64 where
//     256-row tiles fit the chip at once and 128-row ones do not (128->128
//     fp16, 120k rows: 106 -> 91; 256->256 bf16, 60k: 207 -> 162; 64->64 f32,
//     120k: 149 -> 132).  Not with fewer input than output rows: an inverse
//     layer's tiles use from one slot to eight, and its launch lasts as long
//     as the chain of those with eight (768->256, 60k rows: 142 against 180).
// column_tile != 0 forces the 256-row register-gather kernel with that width.
// Every width and both 256-row kernels sum each output in the same order, so
// all give the same bits.  The direct-to-LDS kernel serves layers whose stages
// are 128 bytes of each row (f16/bf16 with C_in % 64 == 0, f32 with C_in % 32
// == 0) and that have a map (K > 1).
MfmaChoice choose_mfma(int dtype, int c_in, int c_out, int K, int64_t n_in, int64_t n_out,
                       int column_tile) {
  MfmaChoice c{pick_bn(c_out), pick_ck(dtype, c_in), false, false, 2};
  if (column_tile) {
    c.bn = column_tile;
    return c;
  }
  const bool f32 = dtype == TSC_F32;
  if (f32 && c.bn > 64) c.bn = 64;  // split slabs of 128 columns leave one workgroup per CU
  const bool dma = K > 1 && c.ck * dtype_bytes(dtype) == 128 && c_in % c.ck == 0;
  auto tiles = [&](int rows) { return ceil_div(n_out, rows) * (c_out / c.bn); };
  auto few = [&] {
    if (K < 8) return tiles(256) < 512;
    if (dma) return tiles(128) < (f32 ? 512 : c.bn == 128 ? 400 : 180);
    return tiles(256) < (c.bn == 128 ? 360 : f32 || K < 12 ? 300 : 128);
  };
  while (c.bn > 32 && few()) c.bn /= 2;
  const bool two = dma ? c_out == 32 || n_in != n_out : K < 12;
  const int64_t split_tiles = f32   ? (c_out > 32 && (n_in != n_out || !dma) ? 4 * kCus : 5 * kCus / 2)
                              : two ? 2 * kCus
                              : dma ? kCus
                                    : 5 * kCus / 2;
  c.split = c.bn == 32 && K >= 8 && tiles(kSplitRows) <= split_tiles;
  c.dma = dma && !c.split;
  if (c.dma && tiles(256) < kShortTiles) {
    const bool one_round = tiles(256) <= kCus * dma_per_cu(dtype, c.bn, 2) &&
                           tiles(128) > kCus * dma_per_cu(dtype, c.bn, 1);
    c.rb = n_in >= n_out && one_round ? 2 : 1;
  }
  return c;
}

template <typename T>
int dispatch_mfma(const void* feat, int64_t n_in, int c_in, const void* W, const Epilogue& ep,
                  const int32_t* nbr, const int32_t* order, int nbr_ordered, int64_t n_out, int K,
                  int c_out, int column_tile, void* out, hipStream_t s) {
  constexpr int dt = std::is_same<T, float>::value ? TSC_F32
                     : std::is_same<T, __half>::value ? TSC_F16 : TSC_BF16;
  const MfmaChoice ch = choose_mfma(dt, c_in, c_out, K, n_in, n_out, column_tile);
#define TSC_MFMA_CASE(BN_, CK_)                                                              \
  if (ch.bn == BN_ && ch.ck == CK_) {                                                        \
    if constexpr (BN_ == 32)                                                                 \
      if (ch.split)                                                                          \
        return launch_split<T, BN_, CK_>(feat, c_in, W, ep, nbr, order, nbr_ordered, n_out,  \
                                         K, c_out, out, s);                                  \
    if constexpr (CK_ * sizeof(T) == 128 && !(sizeof(T) == 4 && BN_ == 128))                 \
      if (ch.dma)                                                                            \
        return ch.rb == 1 ? launch_dma<T, BN_, 1>(feat, c_in, W, ep, nbr, order, nbr_ordered,  \
                                                  n_out, K, c_out, out, s)                   \
                          : launch_dma<T, BN_, 2>(feat, c_in, W, ep, nbr, order, nbr_ordered,  \
                                                  n_out, K, c_out, out, s);                  \
    return launch_mfma<T, BN_, CK_>(feat, c_in, W, ep, nbr, order, nbr_ordered,          \
                                    n_out, K, c_out, out, s);                                \
  }
  if constexpr (!std::is_same<T, float>::value) {
    TSC_MFMA_CASE(128, 64)
    TSC_MFMA_CASE(64, 64)
    TSC_MFMA_CASE(32, 64)
  }
  TSC_MFMA_CASE(128, 32)
  TSC_MFMA_CASE(64, 32)
  TSC_MFMA_CASE(32, 32)
#undef TSC_MFMA_CASE
  return set_error(TSC_EUNSUPPORTED, "conv: no MFMA tile for c_in=%d c_out=%d", c_in, c_out);
}

template <typename T, int READ, int PIECE, int NT>
int launch_narrow(const void* feat, int64_t n_in, int c_in, const void* W, const Epilogue& ep,
                  const int32_t* nbr, const int32_t* order, int nbr_ordered, int64_t n_out, int K,
                  int c_out, void* out, hipStream_t s) {
  constexpr int dt = std::is_same<T, float>::value ? TSC_F32
                     : std::is_same<T, __half>::value ? TSC_F16 : TSC_BF16;
  const int64_t nsteps = narrow_steps(dt, K, c_in);
  TSC_REQUIRE(nsteps < (int64_t(1) << 26), "conv: K * C_in too large");
  constexpr int elem = static_cast<int>(sizeof(T));
  const int64_t feat_bytes = n_in * c_in * elem;
  const uint32_t* form = static_cast<const uint32_t*>(W);  // read, and not looked at, where there is one form
  if (has_forms(dt, c_in, c_out))
    form += tsc_packed_weight_bytes(K, c_in, c_out, dt) / 4 - 1;
  const int64_t cols = ceil_div(c_out, 16) / NT;
  TSC_REQUIRE(cols < 65536, "conv: C_out too large");
  dim3 grid(static_cast<unsigned>(ceil_div(n_out, 4 * kNarrowRows)), static_cast<unsigned>(cols));
  if (NarrowB32::fits(n_in, c_in, elem, n_out, K, nsteps, 16 / elem)) {
    const int cp = narrow_cp(c_in);
    const NarrowB32 nb32{static_cast<uint32_t>(feat_bytes),
                         nbr ? static_cast<uint32_t>((int64_t)K * n_out * 4) : 0u,
                         static_cast<uint32_t>(c_in * elem),
                         static_cast<uint32_t>(((uint64_t(1) << 32) + cp - 1) / cp)};
    conv_narrow_kernel<T, READ, PIECE, NT, true><<<grid, 256, 0, s>>>(
        static_cast<const T*>(feat), feat_bytes, c_in, static_cast<const T*>(W), form, ep, nbr, order,
        nbr_ordered, n_out, K, c_out, static_cast<int>(nsteps), nb32, static_cast<T*>(out));
  } else {
    conv_narrow_kernel<T, READ, PIECE, NT, false><<<grid, 256, 0, s>>>(
        static_cast<const T*>(feat), feat_bytes, c_in, static_cast<const T*>(W), form, ep, nbr, order,
        nbr_ordered, n_out, K, c_out, static_cast<int>(nsteps), NarrowB32{}, static_cast<T*>(out));
  }
  TSC_LAUNCH_CHECK("conv_narrow");
  return 0;
}

template <typename T>
int dispatch_narrow(const void* feat, int64_t n_in, int c_in, const void* W, const Epilogue& ep,
                    const int32_t* nbr, const int32_t* order, int nbr_ordered, int64_t n_out,
                    int K, int c_out, void* out, hipStream_t s) {
  constexpr int elem = static_cast<int>(sizeof(T));
  // Column tiles per wave: up to 4, fewer while that leaves the chip short of
  // workgroups, since each extra column group gathers its rows again (from
  // cache).  Measured per launch, f16, 1 / 2 / 4 tiles: 20->64, 15k rows (235
  // row groups) 15.1 / 10.9 / 11.4 us, 40k rows 30.8 / 21.2 / 18.6; 3->32 with
  // 125 slots, 80k rows 41.6 / 28.5, 3k rows 9.4 / 10.2; f32 128->20, 15k rows
  // 69.7 / 75.1, 40k rows 168 / 145.  One and three tiles: 48->48, 40k rows
  // 36.4 / 27.1, 150k rows 112 / 79.
  const int nt_all = static_cast<int>(ceil_div(c_out, 16));
  const int64_t blocks = ceil_div(n_out, 4 * kNarrowRows);
  auto enough = [&](int nt, int64_t groups) {
    return nt_all % nt == 0 && blocks * (nt_all / nt) >= groups;
  };
  int nt = enough(4, 600) ? 4 : enough(3, 400) ? 3 : enough(2, elem == 4 ? 400 : 200) ? 2 : 1;
  const int whole = (c_in % 8 == 0 || elem == 4) ? 16 : 8;  // bytes of an aligned piece
  const uintptr_t f = reinterpret_cast<uintptr_t>(feat);
  TSC_REQUIRE(f % elem == 0, "conv: features must be aligned to their elements");
  // Widths of whole pieces and tiles are refused features or weights that are
  // not aligned to them; the others take any that are aligned to elements
  // (weights: to words), as they always have.
  const bool regular = c_in % 4 == 0 && c_out % 16 == 0;
  TSC_REQUIRE(!regular || ((f & (whole - 1)) == 0 && (reinterpret_cast<uintptr_t>(W) & 15) == 0),
              "conv: features must be %d-byte and weights 16-byte aligned", whole);
  TSC_REQUIRE((reinterpret_cast<uintptr_t>(W) & 3) == 0, "conv: weights must be 4-byte aligned");
  constexpr int ragged = 4 * elem;  // bytes of a ragged piece
  int read = c_in % 4 == 0 && (f & (whole - 1)) == 0 ? kWhole : kRagged;
  if (read == kRagged && n_in * c_in * elem < ragged) read = kSingle;
  const int piece = read == kWhole ? whole : read == kRagged ? ragged : elem;
  if (read == kSingle) nt = 1;
#define TSC_NARROW_CASE(R_, P_, NT_)                                                         \
  if (read == R_ && piece == P_ && nt == NT_)                                                \
    return launch_narrow<T, R_, P_, NT_>(feat, n_in, c_in, W, ep, nbr, order, nbr_ordered,   \
                                         n_out, K, c_out, out, s);
#define TSC_NARROW_CASES(R_, P_)                                                             \
  TSC_NARROW_CASE(R_, P_, 1)                                                                 \
  TSC_NARROW_CASE(R_, P_, 2)                                                                 \
  TSC_NARROW_CASE(R_, P_, 3)                                                                 \
  TSC_NARROW_CASE(R_, P_, 4)
  TSC_NARROW_CASES(kWhole, 16)
  if constexpr (sizeof(T) == 2) {
    TSC_NARROW_CASES(kWhole, 8)
  }
  TSC_NARROW_CASES(kRagged, ragged)
  TSC_NARROW_CASE(kSingle, elem, 1)
#undef TSC_NARROW_CASES
#undef TSC_NARROW_CASE
  return set_error(TSC_EUNSUPPORTED, "conv: no narrow tile for c_in=%d c_out=%d", c_in, c_out);
}

}  // namespace
}  // namespace tsc

using namespace tsc;

extern "C" int64_t tsc_packed_weight_bytes(int32_t k_vol, int32_t c_in, int32_t c_out,
                                           int32_t dtype) {
  if (pick_path(dtype, c_in, c_out, k_vol) == kMfma) {
    const int ck = pick_ck(dtype, c_in);
    return ((int64_t)k_vol * mfma_chunks(c_in, ck) * ck * c_out +
            (dtype == TSC_F32 ? range_tail(c_in, c_out) : 0)) * dtype_bytes(dtype);
  }
  const int64_t bytes = narrow_bytes(dtype, k_vol, c_in, c_out);
  // widths that do not fill their pieces and tiles: no less than an fp32
  // (K, C_in, C_out) copy, the size these weights have always had, and for
  // 16-bit features a word past the narrow layout for the form
  const int64_t fp32 = (int64_t)k_vol * c_in * c_out * 4;
  if ((c_in % 4 || c_out % 16) && fp32 > bytes) return fp32;
  return bytes + (has_forms(dtype, c_in, c_out) ? 16 : 0);
}

extern "C" int tsc_pack_weight(const void* w, int32_t w_dtype, int32_t layout, int32_t k_vol,
                               int32_t c_in, int32_t c_out, int32_t dtype, void* packed,
                               tsc_stream_t stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  TSC_REQUIRE(dtype_ok(dtype) && dtype_ok(w_dtype), "pack: unsupported dtype");
  TSC_REQUIRE(layout == 0 || layout == 1, "pack: layout must be 0 (KRSC) or 1 (flat)");
  TSC_REQUIRE(k_vol > 0 && c_in > 0 && c_out > 0, "pack: sizes must be positive");
  TSC_REQUIRE(w && packed, "pack: null pointer");
  const int64_t total = (int64_t)k_vol * (c_in + 32) * (c_out + 15);  // covers padded chunks and tiles
  const int grid = static_cast<int>(ceil_div(total, 256) < 2048 ? ceil_div(total, 256) : 2048);
  const Path path = pick_path(dtype, c_in, c_out, k_vol);
  if (path == kNarrow) {
    const int64_t nsteps = narrow_steps(dtype, k_vol, c_in);
    uint32_t* form = nullptr;
    if (has_forms(dtype, c_in, c_out))
      form = static_cast<uint32_t*>(packed) + tsc_packed_weight_bytes(k_vol, c_in, c_out, dtype) / 4 - 1;
    if (form && w_dtype != dtype)
      pack_wide_kernel<<<grid, 256, 0, s>>>(w, w_dtype, layout, k_vol, c_in, c_out,
                                            static_cast<float*>(packed), form);
    else if (dtype == TSC_F32)
      pack_narrow_kernel<float><<<grid, 256, 0, s>>>(w, w_dtype, layout, k_vol, c_in, c_out, nsteps,
                                                     static_cast<float*>(packed), form);
    else if (dtype == TSC_F16)
      pack_narrow_kernel<__half><<<grid, 256, 0, s>>>(w, w_dtype, layout, k_vol, c_in, c_out, nsteps,
                                                      static_cast<__half*>(packed), form);
    else
      pack_narrow_kernel<__hip_bfloat16><<<grid, 256, 0, s>>>(w, w_dtype, layout, k_vol, c_in, c_out, nsteps,
                                                              static_cast<__hip_bfloat16*>(packed), form);
  } else if (path == kMfma) {
    const int ck = pick_ck(dtype, c_in);
    if (dtype == TSC_F32) {
      float* const p = static_cast<float*>(packed);
      pack_mfma_kernel<float><<<grid, 256, 0, s>>>(w, w_dtype, layout, k_vol, c_in, c_out, ck, p);
      const int64_t rows = (int64_t)k_vol * c_in;
      const int64_t elems = (int64_t)k_vol * mfma_chunks(c_in, ck) * ck * c_out;
      if (layout == 0)
        weight_range_kernel<true><<<dim3(c_out, static_cast<unsigned>(std::min<int64_t>(ceil_div(rows, 8192), 16))),
                                    1024, 0, s>>>(w, w_dtype, rows, c_in, c_out, p, elems);
      else
        weight_range_kernel<false><<<dim3(c_out / 32, static_cast<unsigned>(std::min<int64_t>(ceil_div(rows, 256), 64))),
                                     1024, 0, s>>>(w, w_dtype, rows, c_in, c_out, p, elems);
    } else if (dtype == TSC_F16)
      pack_mfma_kernel<__half><<<grid, 256, 0, s>>>(w, w_dtype, layout, k_vol, c_in, c_out, ck,
                                                    static_cast<__half*>(packed));
    else
      pack_mfma_kernel<__hip_bfloat16><<<grid, 256, 0, s>>>(
          w, w_dtype, layout, k_vol, c_in, c_out, ck, static_cast<__hip_bfloat16*>(packed));
  }
  TSC_LAUNCH_CHECK("pack_weight");
  return 0;
}

static int conv_forward(const void* feat, int32_t dtype, int64_t n_in, int32_t c_in,
                        const void* packed_w, const Epilogue& ep, const int32_t* nbr,
                        const int32_t* order, int32_t nbr_ordered, int64_t n_out, int32_t k_vol,
                        int32_t c_out, int32_t column_tile, void* out, hipStream_t s) {
  TSC_REQUIRE(dtype_ok(dtype), "conv: unsupported dtype %d", dtype);
  TSC_REQUIRE(!ep.bias || dtype_ok(ep.bias_dt), "conv: unsupported bias dtype %d", ep.bias_dt);
  TSC_REQUIRE((ep.mean == nullptr) == (ep.var == nullptr),
              "conv: batch-norm mean and variance come together");
  TSC_REQUIRE(ep.mean || (!ep.gamma && !ep.beta),
              "conv: batch-norm weight or bias without running statistics");
  TSC_REQUIRE(!ep.mean || dtype_ok(ep.bn_dt), "conv: unsupported batch-norm dtype %d", ep.bn_dt);
  TSC_REQUIRE(!ep.mean || ep.eps >= 0.f, "conv: batch-norm eps must be non-negative");
  TSC_REQUIRE(c_in > 0 && c_out > 0 && k_vol > 0, "conv: sizes must be positive");
  TSC_REQUIRE(n_out >= 0 && n_out < (int64_t(1) << 31) && n_in >= 0 && n_in < (int64_t(1) << 31),
              "conv: row counts out of range");
  TSC_REQUIRE(nbr || k_vol == 1, "conv: identity map needs k_vol == 1");
  TSC_REQUIRE(nbr || n_in >= n_out, "conv: identity map needs n_in >= n_out");
  TSC_REQUIRE(!nbr_ordered || (order && nbr), "conv: an ordered map needs its order");
  TSC_REQUIRE(nbr_ordered >= 0 && nbr_ordered <= 2, "conv: nbr_ordered must be 0, 1 or 2");
  TSC_REQUIRE(nbr_ordered != 2 || k_vol <= 32,
              "conv: a map with its slot-mask row (nbr_ordered = 2) needs k_vol <= 32");
  const Path path = pick_path(dtype, c_in, c_out, k_vol);
  TSC_REQUIRE(column_tile == 0 || (path == kMfma && (column_tile == 32 || column_tile == 64 ||
                                                     column_tile == 128) &&
                                   c_out % column_tile == 0),
              "conv: %d is not a column tile width of this layer (32, 64 or 128 dividing "
              "c_out=%d, on a 32x32-tile layer)", column_tile, c_out);
  if (n_out == 0) return 0;
  TSC_REQUIRE(packed_w && out && (feat || n_in == 0), "conv: null pointer");
  if (n_in == 0) {
    // no inputs: every output is the epilogue of zero
    TSC_REQUIRE(nbr != nullptr, "conv: empty input");
  }
  if (path == kMfma) {
    TSC_REQUIRE((reinterpret_cast<uintptr_t>(feat) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(packed_w) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(out) & 15) == 0,
                "conv: feature, weight and output buffers must be 16-byte aligned");
    if (dtype == TSC_F32)
      return dispatch_mfma<float>(feat, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered, n_out, k_vol,
                                  c_out, column_tile, out, s);
    if (dtype == TSC_F16)
      return dispatch_mfma<__half>(feat, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered, n_out, k_vol,
                                   c_out, column_tile, out, s);
    return dispatch_mfma<__hip_bfloat16>(feat, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered, n_out,
                                         k_vol, c_out, column_tile, out, s);
  }
  if (dtype == TSC_F32)
    return dispatch_narrow<float>(feat, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered, n_out,
                                  k_vol, c_out, out, s);
  if (dtype == TSC_F16)
    return dispatch_narrow<__half>(feat, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered, n_out,
                                   k_vol, c_out, out, s);
  return dispatch_narrow<__hip_bfloat16>(feat, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered,
                                         n_out, k_vol, c_out, out, s);
}

extern "C" int tsc_conv_forward(const void* feat, int32_t dtype, int64_t n_in, int32_t c_in,
                                const void* packed_w, const void* bias, int32_t bias_dtype,
                                const int32_t* nbr, const int32_t* order, int32_t nbr_ordered,
                                int64_t n_out, int32_t k_vol, int32_t c_out, void* out,
                                tsc_stream_t stream) {
  const Epilogue ep{bias, bias_dtype, nullptr, nullptr, nullptr, nullptr, 0, 0.f, 0};
  return conv_forward(feat, dtype, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered, n_out, k_vol,
                      c_out, 0, out, static_cast<hipStream_t>(stream));
}

extern "C" int tsc_conv_forward_ep(const void* feat, int32_t dtype, int64_t n_in, int32_t c_in,
                                   const void* packed_w, const void* bias, int32_t bias_dtype,
                                   const void* bn_mean, const void* bn_var,
                                   const void* bn_weight, const void* bn_bias, int32_t bn_dtype,
                                   float bn_eps, int32_t relu, const int32_t* nbr,
                                   const int32_t* order, int32_t nbr_ordered, int64_t n_out,
                                   int32_t k_vol, int32_t c_out, void* out, tsc_stream_t stream) {
  const Epilogue ep{bias,      bias_dtype, bn_mean, bn_var, bn_weight,
                    bn_bias,   bn_dtype,   bn_eps,  relu != 0 ? 1 : 0};
  return conv_forward(feat, dtype, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered, n_out, k_vol,
                      c_out, 0, out, static_cast<hipStream_t>(stream));
}

extern "C" int tsc_conv_forward_tile(const void* feat, int32_t dtype, int64_t n_in, int32_t c_in,
                                     const void* packed_w, const void* bias, int32_t bias_dtype,
                                     const int32_t* nbr, const int32_t* order,
                                     int32_t nbr_ordered, int64_t n_out, int32_t k_vol,
                                     int32_t c_out, int32_t column_tile, void* out,
                                     tsc_stream_t stream) {
  const Epilogue ep{bias, bias_dtype, nullptr, nullptr, nullptr, nullptr, 0, 0.f, 0};
  return conv_forward(feat, dtype, n_in, c_in, packed_w, ep, nbr, order, nbr_ordered, n_out, k_vol,
                      c_out, column_tile, out, static_cast<hipStream_t>(stream));
}

extern "C" const char* tsc_conv_kernel_name(int32_t dtype, int32_t c_in, int32_t c_out,
                                            int32_t k_vol, int64_t n_out) {
  if (!dtype_ok(dtype) || c_in <= 0 || c_out <= 0 || k_vol <= 0 || n_out < 0) return "";
  switch (pick_path(dtype, c_in, c_out, k_vol)) {
    case kMfma: {
      const MfmaChoice ch = choose_mfma(dtype, c_in, c_out, k_vol, n_out, n_out, 0);
      return ch.split ? "conv_split_kernel" : ch.dma ? "conv_dma_kernel" : "conv_mfma_kernel";
    }
    default:
      return "conv_narrow_kernel";
  }
}

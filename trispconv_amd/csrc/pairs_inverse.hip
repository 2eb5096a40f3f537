// Inverse (transposed) indice pairs on the GPU.
//
// Reference algorithm: trispconv/pytorch/modules.py:175-212.  The inverse of a
// strided layer reuses its pairs with roles swapped: output rows are the
// forward input rows that took part in at least one forward pair, kept in
// ascending row order (the sorted unique of the concatenated pairs_in,
// :178-182), and slot k maps forward output pairs_out[k][j] to the compact id
// of forward input pairs_in[k][j] (:193-194).
//
// MI355X design: no unique() — a participation flag per forward input row, an
// exclusive scan of the flags (the compact ids, already in ascending row
// order), then one pass that writes the remapped ids, the output-major
// neighbour map and the gathered output coordinates.
#include "common.hpp"

#include <algorithm>

namespace tsc {
namespace {

__global__ void __launch_bounds__(256) inverse_mark_kernel(const int32_t* __restrict__ fwd_pin,
                                                           const int32_t* __restrict__ fwd_cnt,
                                                           int64_t cap, uint32_t* flags) {
  const int k = blockIdx.y;
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j >= fwd_cnt[k]) return;
  flags[fwd_pin[(int64_t)k * cap + j]] = 1u;
}

__global__ void __launch_bounds__(256) inverse_emit_kernel(const uint32_t* __restrict__ flags,
                                                           const uint32_t* __restrict__ id_map,
                                                           const int4* __restrict__ in_coords,
                                                           int64_t n, int4* __restrict__ out_coords,
                                                           int64_t n_out) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n || !flags[i]) return;
  if (id_map[i] < n_out) out_coords[id_map[i]] = in_coords[i];  // holds by construction
}

__global__ void __launch_bounds__(256) inverse_fill_kernel(const int32_t* __restrict__ fwd_pin,
                                                           const int32_t* __restrict__ fwd_pout,
                                                           const int32_t* __restrict__ fwd_cnt,
                                                           int64_t cap, int K, int64_t n_out,
                                                           const uint32_t* __restrict__ id_map,
                                                           int32_t* __restrict__ nbr,
                                                           int32_t* __restrict__ inv_pout) {
  const int k = blockIdx.y;
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j >= fwd_cnt[k]) return;
  const int64_t e = (int64_t)k * cap + j;
  const int32_t o = static_cast<int32_t>(id_map[fwd_pin[e]]);
  inv_pout[e] = o;
  if (o < n_out) nbr[(int64_t)k * n_out + o] = fwd_pout[e];  // holds by construction
}

// The fill's first launch for ids made by the forward build: blocks below
// emit_blocks write out_coords[id] = the row's coordinates for the rows with
// an id; the others fill the map with -1.
__global__ void __launch_bounds__(256) inverse_emit_ids_kernel(const int32_t* __restrict__ in_ids,
                                                               const int4* __restrict__ in_coords,
                                                               int64_t n, int4* __restrict__ out_coords,
                                                               int64_t n_out, int emit_blocks,
                                                               uint32_t* __restrict__ nbr,
                                                               int64_t nbr_words) {
  if (static_cast<int>(blockIdx.x) >= emit_blocks) {
    for (int64_t j = (blockIdx.x - emit_blocks) * (int64_t)blockDim.x + threadIdx.x; j < nbr_words;
         j += (int64_t)(gridDim.x - emit_blocks) * blockDim.x)
      nbr[j] = 0xffffffffu;
    return;
  }
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t id = in_ids[i];
  if (id >= 0 && id < n_out) out_coords[id] = in_coords[i];  // id < n_out holds by construction
}

// --------------------------------------------------- grouped columns --
// Which slots of an inverse layer's row have a pair is decided by its residues
// (coordinate + padding) mod stride: with stride 2 and a 3-wide kernel an axis
// reaches one or two output cells, so a row uses one to eight of the 27 slots,
// and rows of one residue class the same ones (away from the borders).  In row
// order every tile of the convolution meets all classes and runs all slots;
// with the map's columns grouped by class a tile runs only its class's, as
// after a sort by slot mask, for two launches more than the row-order map's two
// instead of the execution order's fourteen, so already the first convolution
// over a new map gains.  Classes with more slots go first: the convolution's long tiles then
// start first.  Measured, 4 x 150k blob voxels, stride 2, 3x3x3: the 64->32
// bf16 inverse convolution 140 -> 63 us (54 once the columns' masks are made, on
// a second use), the inverse build 40 -> 51 us (count 9.4, scan 5.0, emit 18.9,
// fill 17.8; row order: emit 14.2, fill 25.8).
// A row's class only places its column: whatever the coordinates hold, the
// columns are a permutation of the rows.
constexpr int kMaxClasses = 64;
constexpr int kGroupRows = 1024;  // rows of a count block: four per thread

struct Residues {
  int32_t s[3], p[3];          // stride and padding (z, y, x)
  uint8_t rank[kMaxClasses];   // class -> its place, classes with more slots first
  __device__ __forceinline__ int place(int4 c) const {
    auto res = [](int v, int m) {  // v mod m, in 0..m-1 also for negative v
      const int r = v % m;
      return r < 0 ? r + m : r;
    };
    return rank[(res(c.y + p[0], s[0]) * s[1] + res(c.z + p[1], s[1])) * s[2] + res(c.w + p[2], s[2])];
  }
};

// Rows of each class per block, [class][block].
__global__ void __launch_bounds__(256) group_count_kernel(const int32_t* __restrict__ in_ids,
                                                          const int4* __restrict__ in_coords,
                                                          int64_t n, Residues rs, int classes,
                                                          uint32_t* __restrict__ blk_cnt, int nblk) {
  __shared__ uint32_t s_cnt[kMaxClasses];
  if (threadIdx.x < kMaxClasses) s_cnt[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kGroupRows / 256; ++j) {
    const int64_t i = blockIdx.x * (int64_t)kGroupRows + j * 256 + threadIdx.x;
    const bool in = i < n && in_ids[i] >= 0;
    const int c = in ? rs.place(in_coords[i]) : -1;
    uint64_t left = __ballot(in);
    while (left) {  // one LDS add per class of the wave
      const int first = __builtin_amdgcn_readlane(c, __builtin_ctzll(left));
      const uint64_t same = __ballot(c == first);
      if (__lane_id() == 0) atomicAdd(&s_cnt[first], static_cast<uint32_t>(__popcll(same)));
      left &= ~same;
    }
  }
  __syncthreads();
  if (threadIdx.x < classes) blk_cnt[(int64_t)threadIdx.x * nblk + blockIdx.x] = s_cnt[threadIdx.x];
}

// Exclusive scan of m words in place, one workgroup (a thousand rows per word
// and class: 5k words for 600k rows and 8 classes).
__global__ void __launch_bounds__(1024) group_scan_kernel(uint32_t* __restrict__ v, int64_t m) {
  __shared__ uint32_t s_wave[33];
  uint32_t carry = 0;
  for (int64_t base = 0; base < m; base += 4096) {
    const int64_t i0 = base + 4 * (int64_t)threadIdx.x;
    uint32_t x[4], acc = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[j] = i0 + j < m ? v[i0 + j] : 0u;
      acc += x[j];
    }
    uint32_t tot;
    uint32_t run = carry + block_exclusive(acc, s_wave, &tot);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (i0 + j < m) v[i0 + j] = run;
      run += x[j];
    }
    carry += tot;
  }
}

// inverse_emit_ids_kernel with the columns' places: cols_row[column] = id and
// col_of[input row] = column (-1 for rows without a pair).
__global__ void __launch_bounds__(256) group_emit_kernel(
    const int32_t* __restrict__ in_ids, const int4* __restrict__ in_coords, int64_t n, Residues rs,
    int classes, const uint32_t* __restrict__ blk_off, int nblk, int4* __restrict__ out_coords,
    int32_t* __restrict__ cols_row, int32_t* __restrict__ col_of, int64_t n_out, uint32_t* __restrict__ nbr,
    int64_t nbr_words) {
  if (static_cast<int>(blockIdx.x) >= nblk) {
    for (int64_t j = (blockIdx.x - nblk) * (int64_t)blockDim.x + threadIdx.x; j < nbr_words;
         j += (int64_t)(gridDim.x - nblk) * blockDim.x)
      nbr[j] = 0xffffffffu;
    return;
  }
  __shared__ uint32_t s_run[kMaxClasses];                 // next column of each class
  __shared__ uint32_t s_wc[256 / kWave][kMaxClasses];     // this round, per wave
  const int t = threadIdx.x, w = t / kWave;
  if (t < classes) s_run[t] = blk_off[(int64_t)t * nblk + blockIdx.x];
  for (int j = 0; j < kGroupRows / 256; ++j) {
    for (int q = t; q < (256 / kWave) * kMaxClasses; q += 256) (&s_wc[0][0])[q] = 0;
    __syncthreads();
    const int64_t i = blockIdx.x * (int64_t)kGroupRows + j * 256 + t;
    const int32_t id = i < n ? in_ids[i] : -1;
    const bool in = id >= 0;
    const int4 co = in ? in_coords[i] : make_int4(0, 0, 0, 0);
    const int c = in ? rs.place(co) : -1;
    uint32_t rank = 0;
    uint64_t left = __ballot(in);
    while (left) {
      const int first = __builtin_amdgcn_readlane(c, __builtin_ctzll(left));
      const uint64_t same = __ballot(c == first);
      if (c == first) rank = rank_in_wave(same);
      if (__lane_id() == 0) s_wc[w][first] = static_cast<uint32_t>(__popcll(same));
      left &= ~same;
    }
    __syncthreads();
    if (in && id < n_out) {  // id < n_out holds by construction
      uint32_t at = s_run[c] + rank;
      for (int ww = 0; ww < w; ++ww) at += s_wc[ww][c];
      const int64_t column = at < n_out ? at : 0;  // at < n_out too
      out_coords[id] = co;
      cols_row[column] = id;
      col_of[i] = static_cast<int32_t>(column);
    } else if (i < n) {
      col_of[i] = -1;
    }
    __syncthreads();
    if (t < classes)
#pragma unroll
      for (int ww = 0; ww < 256 / kWave; ++ww) s_run[t] += s_wc[ww][t];
    __syncthreads();
  }
}

// inverse_fill_kernel with the map written by column.
__global__ void __launch_bounds__(256) group_fill_kernel(const int32_t* __restrict__ fwd_pin,
                                                         const int32_t* __restrict__ fwd_pout,
                                                         const int32_t* __restrict__ fwd_cnt,
                                                         int64_t cap, int64_t n_out,
                                                         const int32_t* __restrict__ in_ids,
                                                         const int32_t* __restrict__ col_of,
                                                         int32_t* __restrict__ nbr,
                                                         int32_t* __restrict__ inv_pout) {
  const int k = blockIdx.y;
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j >= fwd_cnt[k]) return;
  const int64_t e = (int64_t)k * cap + j;
  const int32_t r = fwd_pin[e];
  inv_pout[e] = in_ids[r];
  const int32_t column = col_of[r];  // rows that a pair names have one
  if (column >= 0) nbr[(int64_t)k * n_out + column] = fwd_pout[e];
}

struct GroupBuffers {
  uint32_t* blk;    // [classes][blocks]: rows, then first columns
  int32_t* col_of;  // [n_fwd_in]
};

GroupBuffers carve_grouped(void* ws, int64_t n, int classes, int64_t* used) {
  Carver c(ws);
  const int64_t m = n > 0 ? n : 1;
  GroupBuffers b;
  b.blk = c.take<uint32_t>(ceil_div(m, kGroupRows) * classes);
  b.col_of = c.take<int32_t>(m);
  if (used) *used = c.used;
  return b;
}

// The product of the strides, 0 when it is not 1..kMaxClasses.
int residue_classes(const int32_t stride[3]) {
  int64_t c = 1;
  for (int a = 0; a < 3; ++a) {
    if (stride[a] <= 0 || stride[a] > kMaxClasses) return 0;
    c *= stride[a];
  }
  return c <= kMaxClasses ? static_cast<int>(c) : 0;
}

struct Buffers {
  uint32_t* flags;
  uint32_t* id_map;
  uint32_t* scratch;
};

Buffers carve(void* ws, int64_t n, int64_t* used) {
  Carver c(ws);
  Buffers b;
  const int64_t m = n > 0 ? n : 1;
  b.flags = c.take<uint32_t>(m);
  b.id_map = c.take<uint32_t>(m);
  b.scratch = c.take<uint32_t>(scan_scratch_words(m));
  if (used) *used = c.used;
  return b;
}

}  // namespace
}  // namespace tsc

using namespace tsc;

extern "C" int64_t tsc_inverse_workspace_bytes(int64_t n_fwd_in) {
  int64_t used = 0;
  carve(nullptr, n_fwd_in, &used);
  return used;
}

extern "C" int tsc_inverse_count(const int32_t* fwd_pairs_in, const int32_t* fwd_counts,
                                 int32_t k_vol, int64_t cap, int64_t n_fwd_in, void* ws,
                                 int64_t ws_bytes, int32_t* counts, tsc_stream_t stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  TSC_REQUIRE(k_vol > 0 && k_vol <= 65535, "inverse: invalid kernel volume %d", k_vol);
  TSC_REQUIRE(n_fwd_in >= 0 && n_fwd_in < (int64_t(1) << 31) && cap >= n_fwd_in,
              "inverse: invalid sizes");
  TSC_REQUIRE(ws && ws_bytes >= tsc_inverse_workspace_bytes(n_fwd_in),
              "inverse: workspace too small");
  TSC_REQUIRE(counts && fwd_counts, "inverse: null counts");
  Buffers b = carve(ws, n_fwd_in, nullptr);
  int rc;
  if ((rc = fill_u32(reinterpret_cast<uint32_t*>(counts), 1, 0u, s))) return rc;
  if (n_fwd_in == 0) return 0;
  TSC_REQUIRE(fwd_pairs_in != nullptr, "inverse: null pair table");
  if ((rc = fill_u32(b.flags, n_fwd_in, 0u, s))) return rc;
  if (cap > 0) {
    dim3 grid(static_cast<unsigned>(ceil_div(cap, 256)), static_cast<unsigned>(k_vol));
    inverse_mark_kernel<<<grid, 256, 0, s>>>(fwd_pairs_in, fwd_counts, cap, b.flags);
    TSC_LAUNCH_CHECK("inverse_mark");
  }
  return exclusive_scan_u32(b.flags, 1, n_fwd_in, b.id_map, counts, b.scratch, s);
}

extern "C" int tsc_inverse_fill(const int32_t* fwd_pairs_in, const int32_t* fwd_pairs_out,
                                const int32_t* fwd_counts, int32_t k_vol, int64_t cap,
                                const int32_t* fwd_in_coords, int64_t n_fwd_in, void* ws,
                                int64_t ws_bytes, int64_t n_out, int32_t* out_coords, int32_t* nbr,
                                int32_t* inv_pairs_out, tsc_stream_t stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  TSC_REQUIRE(k_vol > 0 && k_vol <= 65535, "inverse: invalid kernel volume %d", k_vol);
  TSC_REQUIRE(n_fwd_in >= 0 && cap >= n_fwd_in && n_out >= 0 && n_out <= n_fwd_in,
              "inverse: invalid sizes");
  TSC_REQUIRE(ws && ws_bytes >= tsc_inverse_workspace_bytes(n_fwd_in),
              "inverse: workspace too small");
  if (n_out == 0) return 0;
  TSC_REQUIRE(fwd_pairs_in && fwd_pairs_out && fwd_counts && fwd_in_coords && out_coords && nbr &&
                  inv_pairs_out,
              "inverse: null pointer");
  Buffers b = carve(ws, n_fwd_in, nullptr);
  int rc;
  inverse_emit_kernel<<<ceil_div(n_fwd_in, 256), 256, 0, s>>>(
      b.flags, b.id_map, reinterpret_cast<const int4*>(fwd_in_coords), n_fwd_in,
      reinterpret_cast<int4*>(out_coords), n_out);
  TSC_LAUNCH_CHECK("inverse_emit");
  if ((rc = fill_u32(reinterpret_cast<uint32_t*>(nbr), n_out * k_vol, 0xffffffffu, s))) return rc;
  dim3 grid(static_cast<unsigned>(ceil_div(cap, 256)), static_cast<unsigned>(k_vol));
  inverse_fill_kernel<<<grid, 256, 0, s>>>(fwd_pairs_in, fwd_pairs_out, fwd_counts, cap, k_vol,
                                           n_out, b.id_map, nbr, inv_pairs_out);
  TSC_LAUNCH_CHECK("inverse_fill");
  return 0;
}

extern "C" int tsc_inverse_fill_ids(const int32_t* fwd_pairs_in, const int32_t* fwd_pairs_out,
                                    const int32_t* fwd_counts, int32_t k_vol, int64_t cap,
                                    const int32_t* in_ids, const int32_t* fwd_in_coords,
                                    int64_t n_fwd_in, int64_t n_out, int32_t* out_coords,
                                    int32_t* nbr, int32_t* inv_pairs_out, tsc_stream_t stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  TSC_REQUIRE(k_vol > 0 && k_vol <= 65535, "inverse: invalid kernel volume %d", k_vol);
  TSC_REQUIRE(n_fwd_in >= 0 && n_fwd_in < (int64_t(1) << 31) && cap >= n_fwd_in && n_out >= 0 &&
                  n_out <= n_fwd_in,
              "inverse: invalid sizes");
  if (n_out == 0) return 0;
  TSC_REQUIRE(fwd_pairs_in && fwd_pairs_out && fwd_counts && in_ids && fwd_in_coords &&
                  out_coords && nbr && inv_pairs_out,
              "inverse: null pointer");
  const int emit_blocks = static_cast<int>(ceil_div(n_fwd_in, 256));
  const int64_t nbr_words = n_out * k_vol;
  const int fill_blocks =
      static_cast<int>(std::min<int64_t>(std::max<int64_t>(ceil_div(nbr_words, 256), 1), 4096));
  inverse_emit_ids_kernel<<<emit_blocks + fill_blocks, 256, 0, s>>>(
      in_ids, reinterpret_cast<const int4*>(fwd_in_coords), n_fwd_in,
      reinterpret_cast<int4*>(out_coords), n_out, emit_blocks, reinterpret_cast<uint32_t*>(nbr),
      nbr_words);
  TSC_LAUNCH_CHECK("inverse_emit_ids");
  // every row a forward pair names has an id (it has that pair), so the ids
  // read through pairs_in are never -1
  dim3 grid(static_cast<unsigned>(ceil_div(cap, 256)), static_cast<unsigned>(k_vol));
  inverse_fill_kernel<<<grid, 256, 0, s>>>(fwd_pairs_in, fwd_pairs_out, fwd_counts, cap, k_vol,
                                           n_out, reinterpret_cast<const uint32_t*>(in_ids), nbr,
                                           inv_pairs_out);
  TSC_LAUNCH_CHECK("inverse_fill");
  return 0;
}

extern "C" int64_t tsc_inverse_grouped_workspace_bytes(int64_t n_fwd_in, const int32_t stride[3]) {
  const int classes = stride ? residue_classes(stride) : 0;
  if (n_fwd_in < 0 || classes == 0) return -1;
  int64_t used = 0;
  carve_grouped(nullptr, n_fwd_in, classes, &used);
  return used;
}

extern "C" int tsc_inverse_fill_grouped(
    const int32_t* fwd_pairs_in, const int32_t* fwd_pairs_out, const int32_t* fwd_counts,
    int32_t k_vol, int64_t cap, const int32_t* in_ids, const int32_t* fwd_in_coords,
    int64_t n_fwd_in, const int32_t ksize[3], const int32_t stride[3], const int32_t padding[3],
    const int32_t dilation[3], void* ws, int64_t ws_bytes, int64_t n_out, int32_t* out_coords,
    int32_t* cols_row, int32_t* nbr, int32_t* inv_pairs_out, tsc_stream_t stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  TSC_REQUIRE(ksize && stride && padding && dilation, "inverse: null geometry");
  const int classes = residue_classes(stride);
  TSC_REQUIRE(classes > 0, "inverse: grouped columns need strides of 1..%d residue classes",
              kMaxClasses);
  for (int a = 0; a < 3; ++a)
    TSC_REQUIRE(ksize[a] > 0 && dilation[a] > 0 && padding[a] >= 0, "inverse: invalid geometry");
  TSC_REQUIRE(k_vol > 0 && k_vol <= 65535, "inverse: invalid kernel volume %d", k_vol);
  TSC_REQUIRE(n_fwd_in >= 0 && n_fwd_in < (int64_t(1) << 31) && cap >= n_fwd_in && n_out >= 0 &&
                  n_out <= n_fwd_in,
              "inverse: invalid sizes");
  if (n_out == 0) return 0;
  TSC_REQUIRE(ws && ws_bytes >= tsc_inverse_grouped_workspace_bytes(n_fwd_in, stride),
              "inverse: workspace too small");
  TSC_REQUIRE(fwd_pairs_in && fwd_pairs_out && fwd_counts && in_ids && fwd_in_coords &&
                  out_coords && cols_row && nbr && inv_pairs_out,
              "inverse: null pointer");
  // slots of each class: per axis the offsets a with a * dilation = residue mod stride
  Residues rs;
  int slots[kMaxClasses], by[kMaxClasses];
  for (int a = 0; a < 3; ++a) {
    rs.s[a] = stride[a];
    rs.p[a] = padding[a] % stride[a];
  }
  for (int c = 0; c < classes; ++c) {
    const int r[3] = {c / (stride[1] * stride[2]), c / stride[2] % stride[1], c % stride[2]};
    slots[c] = 1;
    by[c] = c;
    for (int a = 0; a < 3; ++a) {
      int hits = 0;
      for (int64_t o = 0; o < ksize[a]; ++o) hits += o * dilation[a] % stride[a] == r[a];
      slots[c] *= hits;
    }
  }
  std::stable_sort(by, by + classes, [&](int a, int b) { return slots[a] > slots[b]; });
  for (int i = 0; i < classes; ++i) rs.rank[by[i]] = static_cast<uint8_t>(i);

  const GroupBuffers b = carve_grouped(ws, n_fwd_in, classes, nullptr);
  const int4* c4 = reinterpret_cast<const int4*>(fwd_in_coords);
  const int nblk = static_cast<int>(ceil_div(n_fwd_in, kGroupRows));
  group_count_kernel<<<nblk, 256, 0, s>>>(in_ids, c4, n_fwd_in, rs, classes, b.blk, nblk);
  TSC_LAUNCH_CHECK("inverse_group_count");
  group_scan_kernel<<<1, 1024, 0, s>>>(b.blk, (int64_t)nblk * classes);
  TSC_LAUNCH_CHECK("inverse_group_scan");
  const int64_t nbr_words = n_out * k_vol;
  const int fill_blocks =
      static_cast<int>(std::min<int64_t>(std::max<int64_t>(ceil_div(nbr_words, 256), 1), 4096));
  group_emit_kernel<<<nblk + fill_blocks, 256, 0, s>>>(
      in_ids, c4, n_fwd_in, rs, classes, b.blk, nblk, reinterpret_cast<int4*>(out_coords), cols_row,
      b.col_of, n_out, reinterpret_cast<uint32_t*>(nbr), nbr_words);
  TSC_LAUNCH_CHECK("inverse_group_emit");
  dim3 grid(static_cast<unsigned>(ceil_div(cap, 256)), static_cast<unsigned>(k_vol));
  group_fill_kernel<<<grid, 256, 0, s>>>(fwd_pairs_in, fwd_pairs_out, fwd_counts, cap, n_out,
                                         in_ids, b.col_of, nbr, inv_pairs_out);
  TSC_LAUNCH_CHECK("inverse_group_fill");
  return 0;
}

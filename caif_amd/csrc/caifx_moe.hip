// MoE token routing around the grouped dequant-GEMMs: dispatch map, gather into the token-sorted
// expert buffer, weighted combine, and the backward passes of the two.  All of it is HBM-bound
// integer / row-copy work: one wave moves one row segment with 16-byte accesses; nothing is
// reshaped into a GEMM.
//
// The dispatch map is built in three small launches without touching the host:
//   1. every wave counts, per expert, the assignments of its 64-entry slice of the flat
//      [num_tokens*top_k] index array                         -> counts[wave][expert]
//   2. one thread per expert turns its column of counts into exclusive prefix sums over the waves
//      (arrival order) and clamps the total by the capacity; a single wave then scans the totals
//      into the offsets
//   3. every wave ranks its 64 entries among equal experts (stable, by lane order) and writes
//      base[wave][expert] + rank, or -1 past the clamped count.
// The result is the reference's: positions in token-major, k-minor arrival order.
#include "caifx_internal.hpp"

#include <atomic>

namespace caifx {
namespace {

constexpr int kRouteThreads = 256;

// number of lanes below `lane` in `mask`
__device__ __forceinline__ int rank_below(unsigned long long mask, int lane)
{
  return __builtin_popcountll(mask & ((1ull << lane) - 1ull));
}

// The lanes of the wave whose expert id equals this lane's (e < 0: no expert, an empty mask): one ballot per bit of
// the id, each lane keeping the side of the ballot its own bit is on, instead of one round per distinct id.
__device__ __forceinline__ unsigned long long lanes_with_same_expert(int e, int num_experts)
{
  const bool valid = e >= 0;
  unsigned long long same = __ballot(valid);
  const int bits = 32 - __builtin_clz(static_cast<unsigned>(num_experts > 1 ? num_experts - 1 : 1));
  for (int b = 0; b < bits; ++b) {
    const bool one = valid && ((e >> b) & 1);
    const unsigned long long with = __ballot(one);
    same &= one ? with : ~with;
  }
  return valid ? same : 0ull;
}

__global__ __launch_bounds__(kRouteThreads) void map_count_kernel(const int32_t *idx, int64_t total, int num_experts,
                                                                   int32_t *counts)
{
  const int lane = threadIdx.x & 63;
  const int64_t slice = (static_cast<int64_t>(blockIdx.x) * kRouteThreads + threadIdx.x) >> 6;
  const int64_t i = slice * 64 + lane;
  int e = -1;
  if (i < total) {
    e = idx[i];
    if (e < 0 || e >= num_experts) e = -1;
  }
  int32_t *row = counts + slice * num_experts;
  if (slice * 64 < total) {
    for (int x = lane; x < num_experts; x += 64) row[x] = 0;
  }
  __builtin_amdgcn_wave_barrier();
  // the first lane of every expert value writes how many lanes hold it
  const unsigned long long same = lanes_with_same_expert(e, num_experts);
  if (e >= 0 && rank_below(same, lane) == 0) row[e] = __builtin_popcountll(same);
}

// counts[w][e] -> exclusive prefix over w (in place), one wave per expert walking the slices 64 at a
// time; the total, clamped by the capacity, goes to clamped[e]
__global__ __launch_bounds__(64) void map_scan_kernel(int32_t *counts, int64_t slices, int num_experts, int capacity,
                                                       int32_t *clamped)
{
  const int e = blockIdx.x;
  const int lane = threadIdx.x;
  int32_t carry = 0;
  for (int64_t base = 0; base < slices; base += 64) {
    const int64_t w = base + lane;
    const int32_t c = w < slices ? counts[w * num_experts + e] : 0;
    int32_t v = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t up = __shfl_up(v, o, 64);
      if (lane >= o) v += up;
    }
    if (w < slices) counts[w * num_experts + e] = carry + v - c;
    carry += __shfl(v, 63, 64);
  }
  if (capacity > 0 && carry > capacity) carry = capacity;
  if (lane == 0) clamped[e] = carry;
}

__global__ __launch_bounds__(64) void map_offsets_kernel(const int32_t *clamped, int num_experts, int32_t *offsets)
{
  const int lane = threadIdx.x;
  int32_t carry = 0;
  if (lane == 0) offsets[0] = 0;
  for (int base = 0; base < num_experts; base += 64) {
    const int e = base + lane;
    int32_t v = e < num_experts ? clamped[e] : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t up = __shfl_up(v, o, 64);
      if (lane >= o) v += up;
    }
    if (e < num_experts) offsets[e + 1] = carry + v;
    carry += __shfl(v, 63, 64);
  }
}

__global__ __launch_bounds__(kRouteThreads) void map_rank_kernel(const int32_t *idx, int64_t total, int num_experts,
                                                                  const int32_t *base, const int32_t *clamped,
                                                                  int32_t *map)
{
  const int lane = threadIdx.x & 63;
  const int64_t slice = (static_cast<int64_t>(blockIdx.x) * kRouteThreads + threadIdx.x) >> 6;
  const int64_t i = slice * 64 + lane;
  int e = -1;
  if (i < total) {
    e = idx[i];
    if (e < 0 || e >= num_experts) e = -1;
  }
  int pos = -1;
  const unsigned long long same = lanes_with_same_expert(e, num_experts);
  if (e >= 0) {
    pos = base[slice * num_experts + e] + rank_below(same, lane);
    if (pos >= clamped[e]) pos = -1;               // dropped by the capacity limit
  }
  if (i < total) map[i] = pos;
}

// The three steps above in one workgroup of 16 waves, for short index arrays (decode batches: up to 3072
// assignments, three 64-entry slices per wave) whose counts[slice][expert] table fits LDS: four launches back to back
// cost 10-12 us in a graph however little they do, this one 5.5 us at 16 x 6 assignments over 64 experts and 7.0 us at
// 340 x 6 (at 1024 x 6 it measured 12.8 us: no gain left).  A wave asks for all its slices' ids before it looks at
// the first (one memory round trip, not one per slice) and keeps them for the ranking.  Row pitch of the table odd,
// so that a wave walking one expert's column touches 64 different banks.
constexpr int kMapOneThreads = 1024;
constexpr int kMapOneWaves = kMapOneThreads / 64;
constexpr int kMapOneSlices = 3;                                  // slices per wave
constexpr size_t kMapOneLdsMax = 144 * 1024;
__global__ __launch_bounds__(kMapOneThreads) void map_one_kernel(const int32_t *idx, int64_t total, int num_experts, int capacity,
                                                                  int32_t *map, int32_t *offsets)
{
  extern __shared__ int32_t map_lds[];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int slices = static_cast<int>((total + 63) >> 6);
  const int pitch = num_experts | 1;
  int32_t *counts = map_lds;                                      // [slices][pitch]
  int32_t *clamped = map_lds + static_cast<size_t>(slices) * pitch;       // [num_experts]
  int ev[kMapOneSlices];                                          // slice wave + 16 u: this lane's expert id, -1 for none
#pragma unroll
  for (int u = 0; u < kMapOneSlices; ++u) {
    const int64_t i = static_cast<int64_t>(wave + kMapOneWaves * u) * 64 + lane;
    ev[u] = -1;
    if (i < total) ev[u] = idx[i];
    if (ev[u] >= num_experts) ev[u] = -1;
  }
  for (int i = threadIdx.x; i < slices * pitch; i += kMapOneThreads) counts[i] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kMapOneSlices; ++u) {
    const int slice = wave + kMapOneWaves * u;
    if (slice >= slices) break;                                   // the same for every lane of the wave
    const unsigned long long same = lanes_with_same_expert(ev[u], num_experts);
    if (ev[u] >= 0 && rank_below(same, lane) == 0) counts[slice * pitch + ev[u]] = __builtin_popcountll(same);
  }
  __syncthreads();
  // one wave per expert: exclusive prefix over the slices (arrival order), the total clamped by the capacity
  for (int e = wave; e < num_experts; e += kMapOneWaves) {
    int32_t carry = 0;
    for (int base = 0; base < slices; base += 64) {
      const int w = base + lane;
      const int32_t c = w < slices ? counts[w * pitch + e] : 0;
      int32_t v = c;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int32_t up = __shfl_up(v, o, 64);
        if (lane >= o) v += up;
      }
      if (w < slices) counts[w * pitch + e] = carry + v - c;
      carry += __shfl(v, 63, 64);
    }
    if (capacity > 0 && carry > capacity) carry = capacity;
    if (lane == 0) clamped[e] = carry;
  }
  __syncthreads();
  if (wave == 0) {
    int32_t carry = 0;
    if (lane == 0) offsets[0] = 0;
    for (int base = 0; base < num_experts; base += 64) {
      const int e = base + lane;
      int32_t v = e < num_experts ? clamped[e] : 0;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int32_t up = __shfl_up(v, o, 64);
        if (lane >= o) v += up;
      }
      if (e < num_experts) offsets[e + 1] = carry + v;
      carry += __shfl(v, 63, 64);
    }
  }
#pragma unroll
  for (int u = 0; u < kMapOneSlices; ++u) {
    const int slice = wave + kMapOneWaves * u;
    if (slice >= slices) break;
    const int64_t i = static_cast<int64_t>(slice) * 64 + lane;
    const unsigned long long same = lanes_with_same_expert(ev[u], num_experts);
    int pos = -1;
    if (ev[u] >= 0) {
      pos = counts[slice * pitch + ev[u]] + rank_below(same, lane);
      if (pos >= clamped[ev[u]]) pos = -1;           // dropped by the capacity limit
    }
    if (i < total) map[i] = pos;
  }
}

// destination / source row of assignment a = t*top_k + k, or -1
__device__ __forceinline__ int64_t routed_row(const int32_t *idx, const int32_t *map, const int32_t *offsets, int64_t a,
                                              int num_experts)
{
  const int e = idx[a];
  const int p = map[a];
  if (e < 0 || e >= num_experts || p < 0) return -1;
  return static_cast<int64_t>(offsets[e]) + p;
}

template <typename T> struct Vec16 {
  static constexpr int kN = 16 / sizeof(T);
  typedef T type __attribute__((ext_vector_type(16 / sizeof(T))));
};

// Zeroes the rows of [0, rows) that no assignment maps to, for a buffer that holds nothing yet: the first `blocks` workgroups of the
// launch that writes the mapped ones take a row each wave, look through all assignments for it and clear it if there is none.
struct Clear {
  int64_t rows;
  int blocks;                                        // 0: the buffer has been cleared
};
__device__ __forceinline__ void clear_unmapped(const Clear &c, const int32_t *idx, const int32_t *map, const int32_t *offsets, int64_t assignments,
                                               int num_experts, void *buf, int64_t row_bytes)
{
  const int lane = threadIdx.x & 63;
  const int64_t r = (static_cast<int64_t>(blockIdx.x) * kRouteThreads + threadIdx.x) >> 6;
  if (r >= c.rows) return;
  bool mapped = false;
  for (int64_t a0 = lane; a0 < assignments; a0 += 64 * 8) {      // eight at a time: a memory round trip each otherwise
    int e[8], p[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t a = a0 + 64 * u < assignments ? a0 + 64 * u : a0;
      e[u] = idx[a];
      p[u] = map[a];
    }
    int64_t at[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool valid = e[u] >= 0 && e[u] < num_experts && p[u] >= 0;
      const int64_t first = offsets[valid ? e[u] : 0];
      at[u] = valid ? first + p[u] : -1;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) mapped |= at[u] == r;
  }
  if (__ballot(mapped) == 0) zero_bytes(static_cast<unsigned char *>(buf), r * row_bytes, (r + 1) * row_bytes, lane, 64);
}

// one wave per assignment: copy a row, 16 bytes per lane and step
template <typename T>
__global__ __launch_bounds__(kRouteThreads) void dispatch_kernel(const T *in, const int32_t *idx, const int32_t *map,
                                                                  const int32_t *offsets, T *buf, int64_t assignments,
                                                                  int64_t dim, int top_k, int num_experts, bool vec, Clear clear)
{
  if (static_cast<int>(blockIdx.x) < clear.blocks) {
    clear_unmapped(clear, idx, map, offsets, assignments, num_experts, buf, dim * static_cast<int64_t>(sizeof(T)));
    return;
  }
  const int lane = threadIdx.x & 63;
  const int64_t a = (static_cast<int64_t>(blockIdx.x - clear.blocks) * kRouteThreads + threadIdx.x) >> 6;
  if (a >= assignments) return;
  const int64_t row = routed_row(idx, map, offsets, a, num_experts);
  if (row < 0) return;
  const T *src = in + (a / top_k) * dim;
  T *dst = buf + row * dim;
  if (vec) {
    typedef typename Vec16<T>::type v_t;
    constexpr int n = Vec16<T>::kN;
    for (int64_t d = lane * n; d < dim; d += 64 * n) *reinterpret_cast<v_t *>(dst + d) = *reinterpret_cast<const v_t *>(src + d);
  } else {
    for (int64_t d = lane; d < dim; d += 64) dst[d] = src[d];
  }
}

// grad_expert_buffer[row(t,k)] = T(w[t,k] * grad_output[t]); one wave per assignment
template <typename T, bool kVec>
__global__ __launch_bounds__(kRouteThreads) void combine_bwd_kernel(const T *gout, const int32_t *idx, const T *w,
                                                                     const int32_t *map, const int32_t *offsets, T *gbuf,
                                                                     int64_t assignments, int64_t dim, int top_k,
                                                                     int num_experts, Clear clear)
{
  if (static_cast<int>(blockIdx.x) < clear.blocks) {
    clear_unmapped(clear, idx, map, offsets, assignments, num_experts, gbuf, dim * static_cast<int64_t>(sizeof(T)));
    return;
  }
  const int lane = threadIdx.x & 63;
  const int64_t a = (static_cast<int64_t>(blockIdx.x - clear.blocks) * kRouteThreads + threadIdx.x) >> 6;
  if (a >= assignments) return;
  const int64_t row = routed_row(idx, map, offsets, a, num_experts);
  if (row < 0) return;
  const float wt = to_f32<T>(w[a]);
  const T *src = gout + (a / top_k) * dim;
  T *dst = gbuf + row * dim;
  if constexpr (kVec) {
    typedef typename Vec16<T>::type v_t;
    constexpr int n = Vec16<T>::kN;
    for (int64_t d = lane * n; d < dim; d += 64 * n) {
      const v_t g = *reinterpret_cast<const v_t *>(src + d);
      v_t o;
#pragma unroll
      for (int i = 0; i < n; ++i) o[i] = from_f32<T>(wt * to_f32<T>(g[i]));
      *reinterpret_cast<v_t *>(dst + d) = o;
    }
  } else {
    for (int64_t d = lane; d < dim; d += 64) dst[d] = from_f32<T>(wt * to_f32<T>(src[d]));
  }
}

// out[t] = T(sum_k w[t,k] * buf[row(t,k)])  (kWeighted) or T(sum_k buf[row(t,k)]); per element the additions run over k in
// order.  A wave takes one 64-lane piece of a token's row (and every gather_waves-th after it), so that a decode step's few
// tokens still spread over the chip, and asks for the pieces of up to eight rows before it adds the first: with one wave per
// token and one row at a time 16 tokens of 2048 took 14.4 us, a chain of 24 memory round trips.
// The rows and weights of a token are fetched once per batch of 8 assignments by lanes 0..7 and broadcast.
constexpr int kGatherWavesMax = 8;
__host__ __device__ inline int gather_waves(int64_t dim, int n, int64_t num_tokens)
{
  const int64_t pieces = (dim + 64 * n - 1) / (64 * n);
  int waves = pieces < kGatherWavesMax ? static_cast<int>(pieces) : kGatherWavesMax;
  while (waves > 1 && num_tokens * waves > (int64_t{1} << 26) - 4) waves /= 2;      // a grid has fewer than 2^32 threads
  return waves;
}
template <typename T, bool kWeighted, bool kVec>
__global__ __launch_bounds__(kRouteThreads) void gather_sum_kernel(const T *buf, const int32_t *idx, const T *w,
                                                                    const int32_t *map, const int32_t *offsets, T *out,
                                                                    int64_t num_tokens, int64_t dim, int top_k,
                                                                    int num_experts)
{
  constexpr int n = kVec ? Vec16<T>::kN : 1;
  typedef typename Vec16<T>::type v_t;
  const int lane = threadIdx.x & 63;
  const int per_token = gather_waves(dim, n, num_tokens);
  const int64_t wave = (static_cast<int64_t>(blockIdx.x) * kRouteThreads + threadIdx.x) >> 6;
  const int64_t t = wave / per_token;
  if (t >= num_tokens) return;
  for (int64_t d0 = (wave - t * per_token) * 64 * n; d0 < dim; d0 += static_cast<int64_t>(per_token) * 64 * n) {
    const int64_t d = d0 + static_cast<int64_t>(lane) * n;
    float sum[n];
#pragma unroll
    for (int i = 0; i < n; ++i) sum[i] = 0.0f;
    for (int k0 = 0; k0 < top_k; k0 += 8) {
      int64_t my_row = -1;
      float my_w = 0.0f;
      if (lane < 8 && k0 + lane < top_k) {
        const int64_t a = t * top_k + k0 + lane;
        my_row = routed_row(idx, map, offsets, a, num_experts);
        if constexpr (kWeighted) my_w = to_f32<T>(w[a]);
      }
      int64_t row[8];
      v_t v[8];          // (element 0 alone when not kVec)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        row[k] = __shfl(my_row, k, 64);          // -1 past top_k
        if (row[k] >= 0 && d < dim) {
          if constexpr (kVec) v[k] = *reinterpret_cast<const v_t *>(buf + row[k] * dim + d);
          else v[k][0] = buf[row[k] * dim + d];
        }
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float wt = __shfl(my_w, k, 64);
        if (row[k] < 0 || d >= dim) continue;
#pragma unroll
        for (int i = 0; i < n; ++i) {
          if constexpr (kWeighted) sum[i] = __builtin_fmaf(wt, to_f32<T>(v[k][i]), sum[i]);
          else sum[i] += to_f32<T>(v[k][i]);
        }
      }
    }
    if (d < dim) {
      if constexpr (kVec) {
        v_t o;
#pragma unroll
        for (int i = 0; i < n; ++i) o[i] = from_f32<T>(sum[i]);
        *reinterpret_cast<v_t *>(out + t * dim + d) = o;
      } else {
        out[t * dim + d] = from_f32<T>(sum[0]);
      }
    }
  }
}

// one wave per assignment: grad_weights[t,k] = T(sum_d grad_output[t,d] * buffer[row(t,k),d]), fp32;
// 0 for assignments that moved no data.  Lane l adds elements l, l+64, ... in order, then the 64 partial
// sums are added pairwise (xor 32, 16, ..., 1): a fixed order, so results repeat bit for bit.
template <typename T>
__global__ __launch_bounds__(kRouteThreads) void combine_bwd_weights_kernel(const T *gout, const T *buf, const int32_t *idx,
                                                                             const int32_t *map, const int32_t *offsets,
                                                                             T *gw, int64_t assignments, int64_t dim,
                                                                             int top_k, int num_experts)
{
  const int lane = threadIdx.x & 63;
  const int64_t a = (static_cast<int64_t>(blockIdx.x) * kRouteThreads + threadIdx.x) >> 6;
  if (a >= assignments) return;
  const int64_t row = routed_row(idx, map, offsets, a, num_experts);
  float sum = 0.0f;
  if (row >= 0) {
    const T *g = gout + (a / top_k) * dim;
    const T *b = buf + row * dim;
    int64_t d = lane;
    // sixteen pairs asked for before the first is added: the order of the additions is a chain, the loads need not be
    for (; d - lane + 16 * 64 <= dim; d += 16 * 64) {
      T x[16], y[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        x[i] = g[d + 64 * i];
        y[i] = b[d + 64 * i];
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) sum = __builtin_fmaf(to_f32<T>(x[i]), to_f32<T>(y[i]), sum);
    }
    for (; d - lane + 4 * 64 <= dim; d += 4 * 64) {
      T x[4], y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = g[d + 64 * i];
        y[i] = b[d + 64 * i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sum = __builtin_fmaf(to_f32<T>(x[i]), to_f32<T>(y[i]), sum);
    }
    for (; d < dim; d += 64) sum = __builtin_fmaf(to_f32<T>(g[d]), to_f32<T>(b[d]), sum);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  }
  if (lane == 0) gw[a] = from_f32<T>(sum);
}

int check_route(const void *a, const void *b, const int32_t *idx, const int32_t *map, const int32_t *offsets,
                int64_t num_tokens, int64_t dim, int top_k, int num_experts, int dtype)
{
  if (num_tokens < 0 || dim < 0 || top_k < 0 || num_experts <= 0 || !valid_dtype(dtype)) return CAIFX_ERR_INVALID_ARGUMENT;
  if (num_tokens == 0 || dim == 0 || top_k == 0) return CAIFX_OK;
  if (!a || !b || !idx || !map || !offsets) return CAIFX_ERR_INVALID_ARGUMENT;
  if (!aligned_to(a, dtype_size(dtype)) || !aligned_to(b, dtype_size(dtype)) || !aligned_to(idx, 4) || !aligned_to(map, 4) ||
      !aligned_to(offsets, 4))
    return CAIFX_ERR_MISALIGNED;
  return -1;      // go on
}

unsigned wave_blocks(int64_t waves) { return static_cast<unsigned>((waves * 64 + kRouteThreads - 1) / kRouteThreads); }

constexpr int64_t kClearAssignments = 1024, kClearRows = 1024;
// A 16-byte piece a thread and no loop, as fast as the framework's fill (with zero_bytes' loop, four pieces a thread, up to 0.2 us slower: 1716
// rows of 1288 columns and the launch behind it 5.6 us, 5.4 here); single bytes at the ends by the first workgroup.
__global__ __launch_bounds__(256) void zero_all_kernel(unsigned char *y, int64_t bytes)
{
  const int64_t before = (16 - (reinterpret_cast<uintptr_t>(y) & 15)) & 15, head = before < bytes ? before : bytes;
  const int64_t pieces = (bytes - head) / 16, i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, tail = head + 16 * pieces;
  if (i < pieces) reinterpret_cast<u32x4_t *>(y + head)[i] = u32x4_t{0, 0, 0, 0};
  if (i < head) y[i] = 0;
  if (i < 16 && tail + i < bytes) y[tail + i] = 0;
}

// How a buffer of total_rows that holds nothing yet gets its unmapped rows zeroed.  Few rows and assignments: by the launch that fills
// the others (graph replay, clearing launch and this one / this one: 96 rows of 2048 bf16 columns 5.1 / 3.4 us, 1020 rows of 4096 7.7 /
// 5.8, with every other assignment dropped 7.2 / 6.1; 2048 rows of 64 4.8 / 7.1, a wave for each looking through all of them).
// Many: all of the buffer in a launch of its own.  (24576 rows of 2048: 37 us; with 64 workgroups that look for unmapped ones in a
// bitmap 32, but 41 instead of 27 where half of the assignments are dropped.)
int plan_clear(void *buf, int64_t total_rows, int64_t dim, int64_t assignments, int dtype, Clear &c, hipStream_t s)
{
  c = Clear{total_rows, 0};
  const int64_t row_bytes = dim * static_cast<int64_t>(dtype_size(dtype));
  if (total_rows == 0 || row_bytes == 0) return CAIFX_OK;
  if (!buf || total_rows > INT64_MAX / row_bytes) return CAIFX_ERR_INVALID_ARGUMENT;
  if (assignments > 0 && assignments <= kClearAssignments && total_rows <= kClearRows) {
    c.blocks = static_cast<int>(wave_blocks(total_rows));
    return CAIFX_OK;
  }
  const int64_t bytes = total_rows * row_bytes, most = int64_t{1} << 34;      // of a launch: 2^22 workgroups
  for (int64_t at = 0; at < bytes; at += most) {
    const int64_t part = bytes - at < most ? bytes - at : most;
    hipLaunchKernelGGL(zero_all_kernel, dim3(static_cast<unsigned>(part / (256 * 16) + 1)), dim3(256), 0, s, static_cast<unsigned char *>(buf) + at, part);
  }
  return launch_status();
}

}  // namespace
}  // namespace caifx

using namespace caifx;

namespace caifx {
namespace {

// Zeroes rows [0, offsets[0]) and [offsets[E], rows) of a grouped result: the segments' rows are all written by the
// launch behind it (the steps upwards from offsets[0] to offsets[E] cover every row between the two, whatever the order
// of the entries).  Usually there is nothing to do and the launch takes 4.7 us (any does), where clearing the whole result took 11
// (24576 x 1408 bf16) to 15 us (24576 x 2048).
__global__ __launch_bounds__(256) void zero_rest_kernel(const int32_t *offsets, int num_experts, int64_t rows, int64_t row_bytes,
                                                        unsigned char *y)
{
  const int64_t first = offsets[0], end = offsets[num_experts];
  const int64_t lo = first < 0 ? 0 : first > rows ? rows : first, hi = end < 0 ? 0 : end > rows ? rows : end;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, threads = static_cast<int64_t>(gridDim.x) * 256;
  zero_bytes(y, 0, lo * row_bytes, t, threads);
  zero_bytes(y, (hi > lo ? hi : lo) * row_bytes, rows * row_bytes, t, threads);
}

}  // namespace
}  // namespace caifx

extern "C" {

int caifx_qlinear_grouped_zero_rest(int num_experts, const int32_t *offsets, int64_t total_rows, int64_t row_bytes, void *y,
                                    caifx_stream_t stream)
{
  if (num_experts < 0 || total_rows < 0 || row_bytes < 0) return CAIFX_ERR_INVALID_ARGUMENT;
  if (total_rows == 0 || row_bytes == 0) return CAIFX_OK;
  if (!offsets || !y || total_rows > INT64_MAX / row_bytes) return CAIFX_ERR_INVALID_ARGUMENT;
  // 8 pieces a thread where everything is to be cleared; never more than 1024 workgroups, which mostly find nothing to do
  const int64_t blocks = total_rows * row_bytes / (256 * 16 * 8) + 1;
  hipLaunchKernelGGL(caifx::zero_rest_kernel, dim3(static_cast<unsigned>(blocks < 1024 ? blocks : 1024)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), offsets, num_experts, total_rows, row_bytes, static_cast<unsigned char *>(y));
  return caifx::launch_status();
}

size_t caifx_moe_dispatch_map_workspace_bytes(int64_t num_tokens, int top_k, int num_experts)
{
  if (num_tokens <= 0 || top_k <= 0 || num_experts <= 0) return 0;
  const int64_t slices = (num_tokens * top_k + 63) / 64;
  return static_cast<size_t>(slices + 1) * static_cast<size_t>(num_experts) * sizeof(int32_t);
}

int caifx_moe_build_dispatch_map(const int32_t *expert_indices, int64_t num_tokens, int top_k, int num_experts,
                                 int capacity_per_expert, int32_t *dispatch_map, int32_t *expert_offsets,
                                 void *workspace, size_t workspace_bytes, caifx_stream_t stream)
{
  if (num_tokens < 0 || top_k < 0 || num_experts <= 0 || capacity_per_expert < 0 || !expert_offsets) return CAIFX_ERR_INVALID_ARGUMENT;
  const int64_t total = num_tokens * top_k;
  if (total > (int64_t{1} << 31) - 64) return CAIFX_ERR_UNSUPPORTED;
  hipStream_t s = as_stream(stream);
  if (total > 0 && (!expert_indices || !dispatch_map)) return CAIFX_ERR_INVALID_ARGUMENT;
  if (!aligned_to(expert_indices, 4) || !aligned_to(dispatch_map, 4) || !aligned_to(expert_offsets, 4) || !aligned_to(workspace, 4))
    return CAIFX_ERR_MISALIGNED;
  const size_t need = total > 0 ? caifx_moe_dispatch_map_workspace_bytes(num_tokens, top_k, num_experts)
                                : static_cast<size_t>(num_experts) * sizeof(int32_t);
  if (!workspace || workspace_bytes < need) return CAIFX_ERR_WORKSPACE_TOO_SMALL;
  {
    // short index arrays: everything in one workgroup's LDS (the workspace is checked all the same and not used)
    const size_t one = ((static_cast<size_t>((total + 63) / 64)) * static_cast<size_t>(num_experts | 1) + static_cast<size_t>(num_experts)) *
                       sizeof(int32_t);
    if (one <= kMapOneLdsMax && (total + 63) / 64 <= kMapOneWaves * kMapOneSlices) {
      static std::atomic<bool> raised{false};
      if (!raised.load(std::memory_order_relaxed)) {
        if (hipFuncSetAttribute(reinterpret_cast<const void *>(map_one_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(kMapOneLdsMax)) != hipSuccess)
          return CAIFX_ERR_LAUNCH_FAILED;
        raised.store(true, std::memory_order_relaxed);
      }
      hipLaunchKernelGGL(map_one_kernel, dim3(1), dim3(kMapOneThreads), one, s, expert_indices, total, num_experts,
                         capacity_per_expert, dispatch_map, expert_offsets);
      return launch_status();
    }
  }
  const int64_t slices = (total + 63) / 64;
  int32_t *counts = static_cast<int32_t *>(workspace);            // [slices][num_experts]
  int32_t *clamped = counts + slices * num_experts;               // [num_experts]
  if (total > 0)
    hipLaunchKernelGGL(map_count_kernel, dim3(wave_blocks(slices)), dim3(kRouteThreads), 0, s, expert_indices, total,
                       num_experts, counts);
  hipLaunchKernelGGL(map_scan_kernel, dim3(num_experts), dim3(64), 0, s, counts, slices, num_experts, capacity_per_expert,
                     clamped);
  hipLaunchKernelGGL(map_offsets_kernel, dim3(1), dim3(64), 0, s, clamped, num_experts, expert_offsets);
  if (total > 0)
    hipLaunchKernelGGL(map_rank_kernel, dim3(wave_blocks(slices)), dim3(kRouteThreads), 0, s, expert_indices, total,
                       num_experts, counts, clamped, dispatch_map);
  return launch_status();
}

static int moe_dispatch(const void *input, const int32_t *expert_indices, const int32_t *dispatch_map, const int32_t *expert_offsets,
                        void *expert_buffer, int64_t fresh_rows, int64_t num_tokens, int64_t dim, int top_k, int num_experts, int dtype,
                        caifx_stream_t stream)
{
  const int st = check_route(input, expert_buffer, expert_indices, dispatch_map, expert_offsets, num_tokens, dim, top_k,
                             num_experts, dtype);
  if (st > 0) return st;
  const int64_t assignments = st == 0 ? 0 : num_tokens * top_k;
  Clear clear;
  const int cl = plan_clear(expert_buffer, fresh_rows, dim, assignments, dtype, clear, as_stream(stream));
  if (st >= 0 || cl != CAIFX_OK) return cl;
  const size_t es = dtype_size(dtype);
  const bool vec = (dim * es) % 16 == 0 && aligned_to(input, 16) && aligned_to(expert_buffer, 16);
  const dim3 grid(wave_blocks(assignments) + clear.blocks), block(kRouteThreads);
  hipStream_t s = as_stream(stream);
  if (dtype == CAIFX_F32)
    hipLaunchKernelGGL(dispatch_kernel<float>, grid, block, 0, s, static_cast<const float *>(input), expert_indices,
                       dispatch_map, expert_offsets, static_cast<float *>(expert_buffer), assignments, dim, top_k,
                       num_experts, vec, clear);
  else      // fp16 and bf16 rows are copied as 16-bit patterns
    hipLaunchKernelGGL(dispatch_kernel<uint16_t>, grid, block, 0, s, static_cast<const uint16_t *>(input), expert_indices,
                       dispatch_map, expert_offsets, static_cast<uint16_t *>(expert_buffer), assignments, dim, top_k,
                       num_experts, vec, clear);
  return launch_status();
}

int caifx_moe_dispatch(const void *input, const int32_t *expert_indices, const int32_t *dispatch_map,
                       const int32_t *expert_offsets, void *expert_buffer, int64_t num_tokens, int64_t dim, int top_k,
                       int num_experts, int dtype, caifx_stream_t stream)
{
  return moe_dispatch(input, expert_indices, dispatch_map, expert_offsets, expert_buffer, 0, num_tokens, dim, top_k, num_experts, dtype, stream);
}

int caifx_moe_dispatch_fresh(const void *input, const int32_t *expert_indices, const int32_t *dispatch_map, const int32_t *expert_offsets,
                             void *expert_buffer, int64_t total_rows, int64_t num_tokens, int64_t dim, int top_k, int num_experts, int dtype,
                             caifx_stream_t stream)
{
  if (total_rows < 0) return CAIFX_ERR_INVALID_ARGUMENT;
  return moe_dispatch(input, expert_indices, dispatch_map, expert_offsets, expert_buffer, total_rows, num_tokens, dim, top_k, num_experts, dtype,
                      stream);
}

int caifx_moe_combine(const void *expert_buffer, const int32_t *expert_indices, const void *expert_weights,
                      const int32_t *dispatch_map, const int32_t *expert_offsets, void *output, int64_t num_tokens,
                      int64_t dim, int top_k, int num_experts, int dtype, caifx_stream_t stream)
{
  const int st = check_route(expert_buffer, output, expert_indices, dispatch_map, expert_offsets, num_tokens, dim, top_k,
                             num_experts, dtype);
  if (st >= 0) return st;
  if (!expert_weights) return CAIFX_ERR_INVALID_ARGUMENT;
  hipStream_t s = as_stream(stream);
  const bool vec = (dim * dtype_size(dtype)) % 16 == 0 && aligned_to(expert_buffer, 16) && aligned_to(output, 16);
  const dim3 grid(wave_blocks(num_tokens * gather_waves(dim, vec ? 16 / static_cast<int>(dtype_size(dtype)) : 1, num_tokens))), block(kRouteThreads);
#define CAIFX_GO(T)                                                                                                    \
  if (vec)                                                                                                             \
    hipLaunchKernelGGL((gather_sum_kernel<T, true, true>), grid, block, 0, s, static_cast<const T *>(expert_buffer),   \
                       expert_indices, static_cast<const T *>(expert_weights), dispatch_map, expert_offsets,          \
                       static_cast<T *>(output), num_tokens, dim, top_k, num_experts);                                \
  else                                                                                                                 \
    hipLaunchKernelGGL((gather_sum_kernel<T, true, false>), grid, block, 0, s, static_cast<const T *>(expert_buffer),  \
                       expert_indices, static_cast<const T *>(expert_weights), dispatch_map, expert_offsets,          \
                       static_cast<T *>(output), num_tokens, dim, top_k, num_experts)
  if (dtype == CAIFX_F32) {
    CAIFX_GO(float);
  } else if (dtype == CAIFX_F16) {
    CAIFX_GO(f16_t);
  } else {
    CAIFX_GO(bf16_t);
  }
#undef CAIFX_GO
  return launch_status();
}

static int moe_combine_backward_grad_expert(const void *grad_output, const int32_t *expert_indices, const void *expert_weights,
                                            const int32_t *dispatch_map, const int32_t *expert_offsets, void *grad_expert_buffer,
                                            int64_t fresh_rows, int64_t num_tokens, int64_t dim, int top_k, int num_experts, int dtype,
                                            caifx_stream_t stream)
{
  const int st = check_route(grad_output, grad_expert_buffer, expert_indices, dispatch_map, expert_offsets, num_tokens, dim,
                             top_k, num_experts, dtype);
  if (st > 0) return st;
  if (st < 0 && !expert_weights) return CAIFX_ERR_INVALID_ARGUMENT;
  const int64_t assignments = st == 0 ? 0 : num_tokens * top_k;
  Clear clear;
  const int cl = plan_clear(grad_expert_buffer, fresh_rows, dim, assignments, dtype, clear, as_stream(stream));
  if (st >= 0 || cl != CAIFX_OK) return cl;
  const dim3 grid(wave_blocks(assignments) + clear.blocks), block(kRouteThreads);
  hipStream_t s = as_stream(stream);
  const bool vec = (dim * dtype_size(dtype)) % 16 == 0 && aligned_to(grad_output, 16) && aligned_to(grad_expert_buffer, 16);
#define CAIFX_GO(T)                                                                                                    \
  if (vec)                                                                                                             \
    hipLaunchKernelGGL((combine_bwd_kernel<T, true>), grid, block, 0, s, static_cast<const T *>(grad_output),          \
                       expert_indices, static_cast<const T *>(expert_weights), dispatch_map, expert_offsets,          \
                       static_cast<T *>(grad_expert_buffer), assignments, dim, top_k, num_experts, clear);            \
  else                                                                                                                 \
    hipLaunchKernelGGL((combine_bwd_kernel<T, false>), grid, block, 0, s, static_cast<const T *>(grad_output),         \
                       expert_indices, static_cast<const T *>(expert_weights), dispatch_map, expert_offsets,          \
                       static_cast<T *>(grad_expert_buffer), assignments, dim, top_k, num_experts, clear)
  if (dtype == CAIFX_F32) {
    CAIFX_GO(float);
  } else if (dtype == CAIFX_F16) {
    CAIFX_GO(f16_t);
  } else {
    CAIFX_GO(bf16_t);
  }
#undef CAIFX_GO
  return launch_status();
}

int caifx_moe_combine_backward_grad_expert(const void *grad_output, const int32_t *expert_indices,
                                           const void *expert_weights, const int32_t *dispatch_map,
                                           const int32_t *expert_offsets, void *grad_expert_buffer, int64_t num_tokens,
                                           int64_t dim, int top_k, int num_experts, int dtype, caifx_stream_t stream)
{
  return moe_combine_backward_grad_expert(grad_output, expert_indices, expert_weights, dispatch_map, expert_offsets, grad_expert_buffer, 0,
                                          num_tokens, dim, top_k, num_experts, dtype, stream);
}

int caifx_moe_combine_backward_grad_expert_fresh(const void *grad_output, const int32_t *expert_indices, const void *expert_weights,
                                                 const int32_t *dispatch_map, const int32_t *expert_offsets, void *grad_expert_buffer,
                                                 int64_t total_rows, int64_t num_tokens, int64_t dim, int top_k, int num_experts, int dtype,
                                                 caifx_stream_t stream)
{
  if (total_rows < 0) return CAIFX_ERR_INVALID_ARGUMENT;
  return moe_combine_backward_grad_expert(grad_output, expert_indices, expert_weights, dispatch_map, expert_offsets, grad_expert_buffer, total_rows,
                                          num_tokens, dim, top_k, num_experts, dtype, stream);
}

int caifx_moe_combine_backward_grad_weights(const void *grad_output, const void *expert_buffer,
                                            const int32_t *expert_indices, const int32_t *dispatch_map,
                                            const int32_t *expert_offsets, void *grad_weights, int64_t num_tokens,
                                            int64_t dim, int top_k, int num_experts, int dtype, caifx_stream_t stream)
{
  const int st = check_route(grad_output, expert_buffer, expert_indices, dispatch_map, expert_offsets, num_tokens, dim, top_k,
                             num_experts, dtype);
  if (st >= 0) return st;
  if (!grad_weights) return CAIFX_ERR_INVALID_ARGUMENT;
  const int64_t assignments = num_tokens * top_k;
  const dim3 grid(wave_blocks(assignments)), block(kRouteThreads);
  hipStream_t s = as_stream(stream);
#define CAIFX_GO(T)                                                                                                    \
  hipLaunchKernelGGL(combine_bwd_weights_kernel<T>, grid, block, 0, s, static_cast<const T *>(grad_output),            \
                     static_cast<const T *>(expert_buffer), expert_indices, dispatch_map, expert_offsets,             \
                     static_cast<T *>(grad_weights), assignments, dim, top_k, num_experts)
  if (dtype == CAIFX_F32) {
    CAIFX_GO(float);
  } else if (dtype == CAIFX_F16) {
    CAIFX_GO(f16_t);
  } else {
    CAIFX_GO(bf16_t);
  }
#undef CAIFX_GO
  return launch_status();
}

int caifx_moe_dispatch_backward(const void *grad_expert_buffer, const int32_t *expert_indices, const int32_t *dispatch_map,
                                const int32_t *expert_offsets, void *grad_input, int64_t num_tokens, int64_t dim, int top_k,
                                int num_experts, int dtype, caifx_stream_t stream)
{
  const int st = check_route(grad_expert_buffer, grad_input, expert_indices, dispatch_map, expert_offsets, num_tokens, dim,
                             top_k, num_experts, dtype);
  if (st >= 0) return st;
  hipStream_t s = as_stream(stream);
  const bool vec = (dim * dtype_size(dtype)) % 16 == 0 && aligned_to(grad_expert_buffer, 16) && aligned_to(grad_input, 16);
  const dim3 grid(wave_blocks(num_tokens * gather_waves(dim, vec ? 16 / static_cast<int>(dtype_size(dtype)) : 1, num_tokens))), block(kRouteThreads);
#define CAIFX_GO(T)                                                                                                    \
  if (vec)                                                                                                             \
    hipLaunchKernelGGL((gather_sum_kernel<T, false, true>), grid, block, 0, s,                                         \
                       static_cast<const T *>(grad_expert_buffer), expert_indices, static_cast<const T *>(nullptr),   \
                       dispatch_map, expert_offsets, static_cast<T *>(grad_input), num_tokens, dim, top_k, num_experts); \
  else                                                                                                                 \
    hipLaunchKernelGGL((gather_sum_kernel<T, false, false>), grid, block, 0, s,                                        \
                       static_cast<const T *>(grad_expert_buffer), expert_indices, static_cast<const T *>(nullptr),   \
                       dispatch_map, expert_offsets, static_cast<T *>(grad_input), num_tokens, dim, top_k, num_experts)
  if (dtype == CAIFX_F32) {
    CAIFX_GO(float);
  } else if (dtype == CAIFX_F16) {
    CAIFX_GO(f16_t);
  } else {
    CAIFX_GO(bf16_t);
  }
#undef CAIFX_GO
  return launch_status();
}

}  // extern "C"

// Expert-major row order of a MoE routing map: the row map behind TE's
// moe_permute for MXFP4 inputs (code/transformer_engine-2.8.diff:220-356).
// map [T, E] is one byte per (token, expert), non-zero where routed. Output
// row r of the permutation is the r-th routed pair by expert, then token:
//   src[r]     = its token
//   dest[t][e] = r, or -1 where (t, e) is not routed (optional)
//
// Two launches. route_counts_kernel counts the routed tokens of every
// (expert, chunk of tokens); laid out [E, chunks], the counts are in output
// order, so the first output row of a (expert, chunk) is the sum of all
// counts before its own. route_rows_kernel recomputes the flags and ranks
// each routed token within its chunk by ballots. A workgroup covers one chunk
// of tokens for four experts (one map dword per token where E allows it);
// the map is small (256 KB for 4096 tokens x 64 experts) and stays in L2, so
// both launches are bound by latency: one load, a few ballots, one store.
// The torch composition they replace (nonzero, bincount, index_put and their
// fills: 18 launches, 65 us of kernels, three waits of the host) made a
// permute + FP8 requant of 4096 tokens x 7168, 8 of 64 experts, 193.9 us a
// call, of which the requant is 51.8; these two launches take 3.5 + 4.7 us
// (kernel trace) and the call 67.3. The host waits for the first alone; the
// permute + requant enqueues the second before it waits.
#include <algorithm>

#include "omo_internal.h"

namespace omo_hip {

constexpr int kRouteThreads = 256;
constexpr int kRouteExperts = 4;      // experts per workgroup

// Tokens per chunk: whole workgroup steps. At most 64 chunks (a wave sums one
// expert's counts with one load), fewer where experts are many, since every
// workgroup of the second launch sums the counts before its own: about 4096
// counts in all, at least 8 chunks.
static int64_t route_span(int64_t T, int64_t E) {
  const int64_t most = std::min<int64_t>(64, std::max<int64_t>(8, 4096 / E));
  const int64_t steps = (T + kRouteThreads - 1) / kRouteThreads;
  return kRouteThreads * ((steps + most - 1) / most);
}

int64_t route_chunks(int64_t T, int64_t E) {
  if (T == 0 || E == 0) return 0;
  const int64_t span = route_span(T, E);
  return (T + span - 1) / span;
}

// Flags of experts e0 .. e0 + 3 of token t as the four bytes of a dword
// (non-zero: routed); 0 past the map. VEC: E % 4 == 0 and a 4 B aligned map.
template <bool VEC>
__device__ __forceinline__ uint32_t route_flags(const uint8_t* __restrict__ map, int64_t T, int E, int64_t t, int e0) {
  if (t >= T) return 0u;
  const uint8_t* p = map + t * E + e0;
  if (VEC) return *reinterpret_cast<const uint32_t*>(p);
  uint32_t w = 0u;
#pragma unroll
  for (int k = 0; k < kRouteExperts; k++)
    if (e0 + k < E) w |= (uint32_t)p[k] << (8 * k);
  return w;
}

__device__ __forceinline__ bool route_flag(uint32_t w, int k) { return ((w >> (8 * k)) & 0xFFu) != 0u; }

template <bool VEC>
__global__ __launch_bounds__(kRouteThreads) void route_counts_kernel(const uint8_t* __restrict__ map, int64_t T, int E,
                                                                     int64_t span, int chunks,
                                                                     int32_t* __restrict__ counts,
                                                                     int32_t* __restrict__ host_counts) {
  __shared__ int part[kRouteThreads / 64][kRouteExperts];
  const int chunk = blockIdx.x, e0 = blockIdx.y * kRouteExperts;
  const int t = threadIdx.x, wave = t >> 6;
  int n[kRouteExperts] = {0, 0, 0, 0};
  for (int64_t i = 0; i < span; i += kRouteThreads) {
    const uint32_t w = route_flags<VEC>(map, T, E, chunk * span + i + t, e0);
#pragma unroll
    for (int k = 0; k < kRouteExperts; k++) n[k] += __popcll(__ballot(route_flag(w, k)));
  }
  if ((t & 63) == 0) {
#pragma unroll
    for (int k = 0; k < kRouteExperts; k++) part[wave][k] = n[k];
  }
  __syncthreads();
  if (t < kRouteExperts && e0 + t < E) {
    const int sum = part[0][t] + part[1][t] + part[2][t] + part[3][t];
    const int64_t at = (int64_t)(e0 + t) * chunks + chunk;
    counts[at] = sum;
    if (host_counts) host_counts[at] = sum;
  }
}

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
  for (int x = 32; x >= 1; x >>= 1) v += __shfl_xor(v, x);
  return v;
}

// Output rows at or past src_len are not written (a map that changed after
// it was counted, or a caller's src shorter than the routed pairs); rows from
// the routed count to pad_to are set to -1 by the last grid row.
template <bool VEC>
__global__ __launch_bounds__(kRouteThreads) void route_rows_kernel(const uint8_t* __restrict__ map, int64_t T, int E,
                                                                   int64_t span, int chunks,
                                                                   const int32_t* __restrict__ counts,
                                                                   int32_t* __restrict__ src, int64_t src_len,
                                                                   int64_t pad_to, int32_t* __restrict__ dest) {
  constexpr int kWaves = kRouteThreads / 64;
  __shared__ int head[kWaves], seg[kRouteExperts], part[2][kWaves][kRouteExperts];
  const int chunk = blockIdx.x, e0 = blockIdx.y * kRouteExperts;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const bool pad_row = e0 >= E;  // the grid row after the experts, present when there are rows to pad
  // counts before (e0, chunk): all of them for the padding row
  const int64_t before = pad_row ? (int64_t)E * chunks : (int64_t)e0 * chunks + chunk;
  int h = 0;
  for (int64_t i = t; i < before; i += kRouteThreads) h += counts[i];
  h = wave_sum(h);
  // wave k: the counts from (e0 + k, chunk) up to (e0 + k + 1, chunk)
  int g = 0;
  const int64_t at = (int64_t)(e0 + wave) * chunks + chunk + lane;
  if (lane < chunks && at < (int64_t)E * chunks) g = counts[at];
  g = wave_sum(g);
  if (lane == 0) {
    head[wave] = h;
    seg[wave] = g;
  }
  __syncthreads();
  const int base0 = head[0] + head[1] + head[2] + head[3];
  if (pad_row) {
    for (int64_t r = base0 + (int64_t)chunk * kRouteThreads + t; r < pad_to; r += (int64_t)chunks * kRouteThreads)
      src[r] = -1;
    return;
  }
  int base[kRouteExperts];
  base[0] = base0;
#pragma unroll
  for (int k = 1; k < kRouteExperts; k++) base[k] = base[k - 1] + seg[k - 1];
  int buf = 0;
  for (int64_t i = 0; i < span; i += kRouteThreads, buf ^= 1) {
    const int64_t tok = chunk * span + i + t;
    const uint32_t w = route_flags<VEC>(map, T, E, tok, e0);
    int rank[kRouteExperts];
#pragma unroll
    for (int k = 0; k < kRouteExperts; k++) {
      const uint64_t b = __ballot(route_flag(w, k));
      rank[k] = __popcll(b & ((1ull << lane) - 1));
      if (lane == 0) part[buf][wave][k] = __popcll(b);
    }
    __syncthreads();  // the two buffers keep this step's reads apart from the next step's writes
    int pos[kRouteExperts];
#pragma unroll
    for (int k = 0; k < kRouteExperts; k++) {
      int lower = 0, all = 0;
#pragma unroll
      for (int v = 0; v < kWaves; v++) {
        const int c = part[buf][v][k];
        lower += v < wave ? c : 0;
        all += c;
      }
      pos[k] = route_flag(w, k) ? base[k] + lower + rank[k] : -1;
      base[k] += all;
      if (pos[k] >= 0 && pos[k] < src_len) src[pos[k]] = (int32_t)tok;
    }
    if (dest && tok < T) {
      int32_t* d = dest + tok * E + e0;
#pragma unroll
      for (int k = 0; k < kRouteExperts; k++)
        if (e0 + k < E) d[k] = pos[k];
    }
  }
}

static bool route_vec(const void* map, int64_t E) { return E % 4 == 0 && (reinterpret_cast<uintptr_t>(map) & 3) == 0; }

hipError_t launch_route_counts(const void* map, int64_t T, int64_t E, int32_t* counts, int32_t* host_counts,
                               hipStream_t stream) {
  const int64_t chunks = route_chunks(T, E);
  const dim3 grid((unsigned)chunks, (unsigned)((E + kRouteExperts - 1) / kRouteExperts));
  auto kernel = route_vec(map, E) ? route_counts_kernel<true> : route_counts_kernel<false>;
  return launch(kernel, grid, dim3(kRouteThreads), 0, stream, static_cast<const uint8_t*>(map), T, (int)E,
                route_span(T, E), (int)chunks, counts, host_counts);
}

hipError_t launch_route_rows(const void* map, int64_t T, int64_t E, const int32_t* counts, int32_t* src,
                             int64_t src_len, bool pad, int32_t* dest, hipStream_t stream) {
  const int64_t chunks = route_chunks(T, E);
  const dim3 grid((unsigned)chunks, (unsigned)((E + kRouteExperts - 1) / kRouteExperts + (pad ? 1 : 0)));
  auto kernel = route_vec(map, E) ? route_rows_kernel<true> : route_rows_kernel<false>;
  return launch(kernel, grid, dim3(kRouteThreads), 0, stream, static_cast<const uint8_t*>(map), T, (int)E,
                route_span(T, E), (int)chunks, counts, src, src_len, pad ? src_len : (int64_t)0, dest);
}

}  // namespace omo_hip

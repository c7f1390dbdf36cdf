// Fused dual-layout BF16 -> MXFP4 quantize: rowwise 1x32 blocks along K and
// columnwise 32x1 blocks along M from one read of the input.
//
// The columnwise output is defined by the TE integration as
// quant_rowwise(X.T.contiguous()) (code/transformer_engine-2.8.diff:1463-1466):
// codes [K, M/2] and scales [K, M/32]. The reference pays a full transpose
// copy plus a second quantize pass for it. Both layouts here use the
// reference block rule (code/kernel/per_token_quant_mxfp4.cu:151-254) with
// fp4_min = -6, fp4_max = 6, the constants of the quantize wrapper
// (code/kernel/api/mxfp4.py:11-12, 152-154).
//
// Tiles are 64 rows x 256 columns (32 KiB of bf16), 512 threads. Each lane
// loads 4 chunks of 16 B (rows r0 + 16k of one 16 B column chunk); the
// rowwise blocks are quantized from registers exactly as in the rowwise
// kernel (a block is a DPP quad) and their codes leave as full 128 B lines
// (non-temporal stores). The tile is staged in LDS without padding: the 16 B
// chunks of each 16-row band are XOR-swizzled so the column pass reads four
// bands from four different 64 B bank ranges. In the column pass, lanes
// 4i..4i+3 own column pair i, one 16-row half of a 32-row block each: a lane
// reads one dword (two adjacent columns) from 16 rows, repacks the columns
// into bf16 pairs with v_perm_b32, combines the block amax with its partner
// lane (DPP), and converts its half block to 8 code bytes per column. The
// four lanes' 8 B stores then write each column's 32 B piece of the
// transposed codes as one contiguous run. (With the two 16 B halves of a
// piece stored by different waves, each store instruction touched 64
// different lines; pairing them cut the 7168 x 18432 kernel from 93 to 83 us.)
//
#include <algorithm>

#include "omo_internal.h"
#include "omo_quant.cuh"

namespace omo_hip {

constexpr int kDualRows = 64;
constexpr int kDualCols = 256;
constexpr int kDualPitch = kDualCols * 2;  // bytes per LDS row (no padding: swizzled)
constexpr int kXcds = 8;
constexpr int kDualGroupMax = 32;
constexpr int kDualThreads = 512;

// Half of a 32-element column block: 8 packed bf16 pairs (rows 2j low, 2j+1
// high); amax_bits is the whole block's max |x| bit pattern (< 0x7F80).
// Returns the 8 code bytes.
__device__ __forceinline__ uint2 quant_half16_fast(const uint32_t (&p)[8], uint32_t amax_bits, int c_eps,
                                                   uint32_t* byte) {
  const float y_s = fast_block_scale(amax_bits, c_eps, byte);
  uint2 out;
  uint32_t r = p[0];  // all four bytes are written
  r = cvt_pk_fp4<0>(r, p[0], y_s);
  r = cvt_pk_fp4<1>(r, p[1], y_s);
  r = cvt_pk_fp4<2>(r, p[2], y_s);
  r = cvt_pk_fp4<3>(r, p[3], y_s);
  out.x = r;
  r = p[4];
  r = cvt_pk_fp4<0>(r, p[4], y_s);
  r = cvt_pk_fp4<1>(r, p[5], y_s);
  r = cvt_pk_fp4<2>(r, p[6], y_s);
  r = cvt_pk_fp4<3>(r, p[7], y_s);
  out.y = r;
  return out;
}

// Reference emulation for a half block; the two lanes holding a block's
// halves (lanes 2i, 2i+1) call it together.
__device__ __forceinline__ uint2 quant_half16_ref(const uint32_t (&p)[8], float eps, uint32_t* byte) {
  float amax = eps;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    amax = fmax_abs_bf16(amax, p[k]);
    amax = fmax_abs_bf16(amax, p[k] >> 16);
  }
  amax = fmaxf(amax, __uint_as_float(dpp_quad_xor1(__float_as_uint(amax))));
  float inv;
  *byte = ref_scale(amax, 6.0f, &inv);
  uint32_t o[2];
#pragma unroll
  for (int w = 0; w < 2; w++) {
    uint32_t v = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t pk = p[4 * w + k];
      const float qx = fminf(fmaxf(bf16_to_f32(pk & 0xFFFFu) * inv, -6.0f), 6.0f);
      const float qy = fminf(fmaxf(bf16_to_f32(pk >> 16) * inv, -6.0f), 6.0f);
      v |= (e2m1_from_f32_ref(qx) | (e2m1_from_f32_ref(qy) << 4)) << (8 * k);
    }
    o[w] = v;
  }
  return make_uint2(o[0], o[1]);
}

// One 64 x 256 tile (tile row mt, band kt) of the [M, K] tensor x,
// 512 threads. FULL: every tile of the tensor is whole (M % 64 == 0, K % 256
// == 0): no clamping, no store under a bounds test (512 x 7168 4.90 -> 4.72
// us, 2048 x 7168 11.6 -> 11.3, 8192 x 7168 35.0 -> 34.8). LINES: K % 256 ==
// 0, so that the 128 B of codes a tile gives a row are a whole line and are
// stored non-temporally (1056 x 7168 7.0 us, 7.5 with ordinary stores).
// Without, every such piece shares its lines with the next tile's, and
// ordinary stores let L2 complete them (4096 x 2880 10.7 -> 10.4 us, 4064 x
// 7136 22.2 -> 22.0, 8192 x 5344 31.2 -> 30.8). A row's 8 scale
// bytes and a column's 2 leave as one store at any alignment (byte by byte
// where rows of K / 32 bytes are not 8 B aligned, 4096 x 2880 took 10.9 us
// against 10.7).
template <bool FULL, bool LINES>
__device__ __forceinline__ void dual_tile(const uint16_t* __restrict__ x, uint32_t* __restrict__ row_q,
                                          uint8_t* __restrict__ row_s, uint8_t* __restrict__ col_q,
                                          uint8_t* __restrict__ col_s, int64_t M, int64_t K, int64_t mt, int64_t kt,
                                          float eps, int c_eps, uint8_t* tile, uint8_t* rs_tile) {
  const int t = threadIdx.x;
  const int64_t m0 = mt * kDualRows, k0 = kt * kDualCols;
  const int rows_valid = FULL ? kDualRows : (int)(M - m0 < kDualRows ? M - m0 : kDualRows);  // 32 or 64
  // lane t owns 16 B column chunk cc of rows r0 + 16k (k = 0..3)
  const int r0 = t >> 5, cc = t & 31;
  const int64_t col = k0 + cc * 8;
  const int64_t cl = FULL || col < K ? col : K - 8;
  u32x4 d[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int r = r0 + 16 * k;
    const int rr = FULL || r < rows_valid ? r : rows_valid - 1;
    d[k] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(x + (m0 + rr) * K + cl));
  }
  const bool quad_leader = (t & 3) == 0;
  uint32_t* rq = row_q + (m0 + r0) * (K / 8) + col / 8;
  uint32_t codes[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    // row r0 + 16k is in 16-row band k: its chunks are stored XORed by 4k,
    // so the four bands sit in four different 64 B bank ranges
    *reinterpret_cast<u32x4*>(tile + (r0 + 16 * k) * kDualPitch + ((cc ^ (k << 2)) * 16)) = d[k];
    uint32_t byte;
    const uint32_t am = quad_max_u32(chunk_absmax_bits(d[k]));
    if (__builtin_expect(am < 0x7F80u, 1)) {
      codes[k] = quant_chunk_fast(d[k], am, c_eps, &byte);
    } else {
      quant_chunk_ref(d[k], eps, -6.0f, 6.0f, &codes[k], &byte);
    }
    // the 8 scale bytes of a tile row are gathered in LDS and leave as one store
    if (quad_leader) rs_tile[(r0 + 16 * k) * 8 + (cc >> 2)] = (uint8_t)byte;
  }
  // The code stores follow all four conversions: a store under the bounds
  // test ahead of the next chunk made the wait for that chunk's load wait
  // for the store as well (loads and stores share one counter).
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (FULL || (r0 + 16 * k < rows_valid && col < K)) {
      if (LINES) __builtin_nontemporal_store(codes[k], rq + k * 2 * K);  // 16 rows down
      else rq[k * 2 * K] = codes[k];
    }
  __syncthreads();
  if (t < rows_valid) {
    uint8_t* rs = row_s + (m0 + t) * (K / 32) + k0 / 32;
    const int nsc = FULL ? 8 : (int)((K - k0) / 32 < 8 ? (K - k0) / 32 : 8);
    if (FULL || nsc == 8) {
      const uint2 v = *reinterpret_cast<const uint2*>(rs_tile + t * 8);
      __builtin_memcpy(rs, &v, 8);
    } else {
      for (int j = 0; j < nsc; j++) rs[j] = rs_tile[t * 8 + j];
    }
  }
  // ---- columnwise: lanes 4i..4i+3 own column pair i; lane 4i + 2g + h holds
  // rows 32g + 16h .. +15 (half h of row block g), so the four lanes' 8 B
  // code stores form the column's 32 B piece
  const int h = t & 1, g = (t >> 1) & 1, p = t >> 2;
  const int64_t kc = k0 + 2 * p;
  // every lane runs the column pass (rows and columns past the tensor read
  // the tile's clamped copies) so that the scale exchange below sees all
  // lanes; only valid results are stored
  const bool active = FULL || (32 * g < rows_valid && kc < K);
  const int band = 2 * g + h;
  const int pp = 4 * (p ^ (band << 4));
  uint32_t ca[8], cb[8];
  uint32_t amax_a = 0, amax_b = 0;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const uint32_t w0 = *reinterpret_cast<const uint32_t*>(tile + (16 * band + 2 * j) * kDualPitch + pp);
    const uint32_t w1 = *reinterpret_cast<const uint32_t*>(tile + (16 * band + 2 * j + 1) * kDualPitch + pp);
    ca[j] = __builtin_amdgcn_perm(w1, w0, 0x05040100u);  // column 2p: rows 2j (low), 2j+1 (high)
    cb[j] = __builtin_amdgcn_perm(w1, w0, 0x07060302u);  // column 2p+1
    amax_a = pk_max_u16(amax_a, ca[j] & 0x7FFF7FFFu);
    amax_b = pk_max_u16(amax_b, cb[j] & 0x7FFF7FFFu);
  }
  amax_a = max(amax_a & 0xFFFFu, amax_a >> 16);
  amax_b = max(amax_b & 0xFFFFu, amax_b >> 16);
  amax_a = max(amax_a, dpp_quad_xor1(amax_a));  // the other half of the block
  amax_b = max(amax_b, dpp_quad_xor1(amax_b));
  uint32_t byte_a, byte_b;
  uint2 qa, qb;
  if (__builtin_expect(amax_a < 0x7F80u, 1)) qa = quant_half16_fast(ca, amax_a, c_eps, &byte_a);
  else qa = quant_half16_ref(ca, eps, &byte_a);
  if (__builtin_expect(amax_b < 0x7F80u, 1)) qb = quant_half16_fast(cb, amax_b, c_eps, &byte_b);
  else qb = quant_half16_ref(cb, eps, &byte_b);
  const int64_t mo = (m0 + 16 * band) / 2;
  if (active) {
    *reinterpret_cast<uint2*>(col_q + kc * (M / 2) + mo) = qa;
    *reinterpret_cast<uint2*>(col_q + (kc + 1) * (M / 2) + mo) = qb;
  }
  // A column's two scale bytes of this tile (row blocks g = 0, 1) sit in
  // lanes 4p + 2g; swapping them (quad lane ^ 2) lets lane 4p write column
  // kc's pair and lane 4p + 2 column kc + 1's as one 2-byte store each.
  const uint32_t oa = dpp_quad_xor2(byte_a), ob = dpp_quad_xor2(byte_b);
  if (h == 0 && (FULL || kc < K)) {
    const int64_t so = m0 / 32;  // even: m0 is a multiple of 64
    uint8_t* const cs = col_s + (kc + g) * (M / 32) + so;
    if (FULL || rows_valid == kDualRows) {
      const uint16_t pair = (uint16_t)(g == 0 ? (byte_a | (oa << 8)) : (ob | (byte_b << 8)));
      __builtin_memcpy(cs, &pair, 2);
    } else if (active) {
      col_s[kc * (M / 32) + so + g] = (uint8_t)byte_a;
      col_s[(kc + 1) * (M / 32) + so + g] = (uint8_t)byte_b;
    }
  }
}

// Band-group order of S x B units (S along M, B bands of 256 columns; a unit
// is a tile or a column of four, below). Numbered M-fastest (L = band * S +
// row), the units are cut into eight contiguous ranges of per_xcd = ceil(S *
// B / 8), one per XCD, so each XCD owns a group of whole bands (the ends of its
// range may be parts of bands). Each XCD walks its range row by row: all of its
// bands of row m, then those of m + 1. The eight XCDs thus sweep the tensor's
// rows together: at any moment the chip reads a few whole stripes of the
// input, each row's codes are written by all XCDs at about the same time, and
// each XCD's column codes fill its own contiguous region. Memory-only copies
// at 7168 x 18432 (256-row stripes, heavy-tailed weights, rotating buffers):
// 68.0 us against 73.3 us for M-fastest ranges (each XCD finishing one band
// before the next) and 73.4 us for K-fastest ones (the XCDs on different
// stripes), which also write 10 MB more (scale lines leaving L2 partly
// filled).
struct BandUnits {
  int rows, count;  // S; S * B
  int per_xcd;      // ceil(S * B / 8)
  int shift;        // log2 of the tiles per unit
  int last;         // tiles of a unit of the last row: 1 .. 1 << shift
};

static BandUnits band_units(int64_t tiles_m, int64_t bands, int shift) {
  const int64_t rows = (tiles_m + (1 << shift) - 1) >> shift, count = rows * bands;
  return {(int)rows, (int)count, (int)((count + kXcds - 1) / kXcds), shift,
          (int)(tiles_m - (rows - 1) * (1 << shift))};
}

// Tiles of XCD xcd's range: hi / rows - lo / rows of its units are in the last
// row.
static int band_group_tiles(int xcd, const BandUnits& u) {
  const int lo = xcd * u.per_xcd, end = lo + u.per_xcd, hi = end < u.count ? end : u.count;
  if (hi <= lo || u.rows == 0) return 0;
  return ((hi - lo) << u.shift) - ((1 << u.shift) - u.last) * (hi / u.rows - lo / u.rows);
}

// Tile row and band of tile j of XCD xcd's walk; false past its range. The
// last row of units, which may hold fewer tiles each, comes last in the walk,
// so no position is without a tile (with four positions for each of its units
// 64 x 786432 took 67.1 us against 28.7, 576 x 196608 78.7 against 65.1, 32
// items of 64 x 32768 109.7 against 36.0; and 32 x 2^29 passed the 2^32 - 1
// work-items of a launch).
// TILES: units of one tile (shift 0).
template <bool TILES>
__device__ __forceinline__ bool band_group_tile(int xcd, int j, const BandUnits& u, int* ms, int* kb) {
  const int S = u.rows, lo = xcd * u.per_xcd, hi = min(u.count, lo + u.per_xcd);
  const int kb0 = lo / S, ms0 = lo - kb0 * S;  // first unit of the range
  const int kb1 = hi / S, ms1 = hi - kb1 * S;  // one past the last
  if (TILES ? j >= hi - lo : hi <= lo) return false;
  int tile = 0;
  if (!TILES) {
    const int upper = hi - lo - (kb1 - kb0);  // units above the last row
    if (j < upper << u.shift) {
      tile = j & ((1 << u.shift) - 1);
      j >>= u.shift;
    } else {
      const int k = j - (upper << u.shift);
      const int q = u.last == 3 ? k / 3 : k >> (u.last >> 1);  // k / last
      if (q >= kb1 - kb0) return false;
      j = upper + q;
      tile = k - q * u.last;
    }
  }
  // units of the range in rows below m: band kb0 holds rows
  // [ms0, S) (or [ms0, ms1) when kb0 == kb1), bands kb0 + 1 .. kb1 - 1 all,
  // band kb1 [0, ms1)
  auto below = [&](int m) {
    if (kb0 == kb1) return max(0, min(m, ms1) - ms0);
    return m * (kb1 - kb0 - 1) + max(0, m - ms0) + min(m, ms1);
  };
  int a = 0, b = S;  // below(a) <= j < below(b) = hi - lo
  while (b - a > 1) {
    const int mid = (a + b) >> 1;
    if (below(mid) <= j) a = mid;
    else b = mid;
  }
  *ms = TILES ? a : (a << u.shift) + tile;
  *kb = kb0 + (a >= ms0 ? 0 : 1) + (j - below(a));
  return true;
}

// Unit of the band-group order for one tensor: four vertically adjacent tiles,
// handed out one after the other. They fill the 128 B lines of the column
// codes (256 rows) and the 8-byte runs of the column scales, which so are
// complete in L2 soon after they were begun, however many bands an XCD owns:
// 2048 x 65536 77.5 us tile by tile, 72.1 in fours; 7168 x 18432 68.8 and
// 69.0; 16384 x 7168 63.8 and 63.5. A kernel that kept four tiles' column
// codes in registers and wrote whole lines (80 VGPRs, three workgroups per CU
// where this one has four) is level or up to 2% ahead on some large tensors in
// back-to-back launches and behind on others (2048 x 65536 73.2 us, this one
// 74.7; 12288 x 12288 80.0, 81.3; 7168 x 18432 70.7, 71.1; 16384 x 18432 180.3,
// 179.8; 16384 x 7168 65.7, 65.0; 5120 x 20480 60.4, 58.0; 28672 x 8192 128.2,
// 124.3), and behind on all of them after a 512 MB fill (84.8, 84.0; 97.1,
// 89.4; 84.8, 80.0; 185.1, 183.0; 76.4, 72.0; 70.3, 64.9; 151.0, 139.0). From
// about 1.5 to 15 ms after a load begins the GPU's clocks dip; there it was
// 1-4% ahead at 7168 x 18432 (blocks of 20 launches: 73-77 us, 73-82).
constexpr int kDualQuadShift = 2;  // log2 of the tiles per unit

// units.rows > 0: band groups over those units. Else each XCD takes a
// contiguous M-fastest range of units.per_xcd tiles. Measured (graph
// replays): 8192 x 7168 37.1 us against 38.3, 4096 x 7168 20.7 against 21.1;
// with fewer than six tiles per CU the ranges are ahead (7168 x 2048 11.7
// against 12.0, 2048 x 2048 5.5 against 5.9).
template <bool FULL, bool LINES>
__global__ __launch_bounds__(kDualThreads) void quant_dual_kernel(const uint16_t* __restrict__ x, uint32_t* __restrict__ row_q,
                                                         uint8_t* __restrict__ row_s, uint8_t* __restrict__ col_q,
                                                         uint8_t* __restrict__ col_s, int64_t M, int64_t K,
                                                         int tiles_m, int tiles, BandUnits units, float eps,
                                                         int c_eps) {
  __shared__ __attribute__((aligned(16))) uint8_t tile[kDualRows * kDualPitch];
  __shared__ __attribute__((aligned(8))) uint8_t rs_tile[kDualRows * 8];
  const int xcd = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
  int ms, kb;
  if (units.rows > 0) {
    if (!band_group_tile<false>(xcd, j, units, &ms, &kb)) return;
  } else {
    const int logical = xcd * units.per_xcd + j;
    if (logical >= tiles) return;
    ms = logical % tiles_m;
    kb = logical / tiles_m;
  }
  dual_tile<FULL, LINES>(x, row_q, row_s, col_q, col_s, M, K, ms, kb, eps, c_eps, tile, rs_tile);
}

// Grouped form: one launch over up to kDualGroupMax tensors (e.g. the weights
// of all local experts). Every XCD takes its band-group share of each item,
// item after item, so the XCDs sweep the items one after another together.
// The descriptor table travels by value in the kernel arguments.
struct DualItem {
  const uint16_t* x;
  uint32_t* row_q;
  uint8_t* row_s;
  uint8_t* col_q;
  uint8_t* col_s;
  int64_t M, K;
  BandUnits units;  // of its 64-row tiles
};

struct DualGroup {
  DualItem item[kDualGroupMax];
  int count, c_eps;
  float eps;
};

// With items walked in fours: each XCD's tiles of each item, counted by the
// host (with two divisions per item in every workgroup 24 expert weights took
// 330 us against 201).
struct DualGroupFours : DualGroup {
  int share[kXcds][kDualGroupMax];
};

// Each XCD takes its band-group share of each item, item after item, over
// the items' 64-row tiles. cfg5's 24 expert weights (16 of 7168 x 2048, 8 of
// 2048 x 7168): 208.8 us against 214.4 us with contiguous ranges of all
// items' 64-row tiles and 223-226 us with whole items per XCD. Smaller items
// as well: 8 of 2048 x 2048 24.1 against 25.3 us with the contiguous ranges,
// 16 of 1024 x 4096 43 against 45, 32 of 2048 x 768 35.5-38.4 against
// 39.6-41.2. Each XCD a run of row tiles of each item (all its bands, so the
// items of 8 bands write whole row-scale halves from one XCD) took 215-218 us
// for those items and 224-226 us for all items, against 206-211 us. Items of
// more than 64 bands (eight per XCD) are walked in units of four tiles, as
// single tensors are; on narrower ones that order and tile by tile differ by
// at most 1.4% either way (16 expert weights of hidden size 7168, ffn 2048:
// 201.9 us tile by tile, 201.5 in fours; ffn 4096: 401.5 and 405.5).
constexpr int kDualWideBands = 64;

// Group: DualGroup where no item is walked in fours (8 of 2048 x 2048 with the
// general walk and its table 22.1 us against 21.8).
template <bool FULL, bool LINES, typename Group>
__global__ __launch_bounds__(kDualThreads) void quant_dual_grouped_kernel(const Group g) {
  constexpr bool TILES = std::is_same_v<Group, DualGroup>;
  __shared__ __attribute__((aligned(16))) uint8_t tile[kDualRows * kDualPitch];
  __shared__ __attribute__((aligned(8))) uint8_t rs_tile[kDualRows * 8];
  const int b = blockIdx.x, xcd = b % kXcds;
  int j = b / kXcds, i = 0;
  for (; i < g.count; i++) {
    const BandUnits& u = g.item[i].units;
    int n;
    if constexpr (TILES) n = min(max(u.count - xcd * u.per_xcd, 0), u.per_xcd);
    else n = g.share[xcd][i];
    if (j < n) break;
    j -= n;
  }
  if (i == g.count) return;
  const DualItem& it = g.item[i];
  int ms, kb;
  if (!band_group_tile<TILES>(xcd, j, it.units, &ms, &kb)) return;
  dual_tile<FULL, LINES>(it.x, it.row_q, it.row_s, it.col_q, it.col_s, it.M, it.K, ms, kb, g.eps, g.c_eps, tile,
                         rs_tile);
}

// The largest XCD's share of a tensor's tiles: the grid's positions per XCD.
static int band_group_slots(const BandUnits& u) {
  int n = 0;
  for (int x = 0; x < kXcds; x++) n = std::max(n, band_group_tiles(x, u));
  return n;
}

// Tensors of whole 64 x 256 tiles.
static bool dual_full(int64_t M, int64_t K) { return M % kDualRows == 0 && K % kDualCols == 0; }

hipError_t launch_quant_dual(const void* x, void* row_q, void* row_s, void* col_q, void* col_s, int64_t M, int64_t K,
                             float eps, hipStream_t stream) {
  if (M == 0 || K == 0) return hipSuccess;
  const int64_t tiles_m = (M + kDualRows - 1) / kDualRows;
  const int64_t tiles_k = (K + kDualCols - 1) / kDualCols;
  const int64_t tiles = tiles_m * tiles_k;
  const bool band_group = tiles >= 6 * (int64_t)current_device_caps().cus;
  BandUnits units = {0, 0, (int)((tiles + kXcds - 1) / kXcds), 0, 1};
  int64_t slots = units.per_xcd;  // of each XCD
  if (band_group) {
    units = band_units(tiles_m, tiles_k, kDualQuadShift);
    slots = band_group_slots(units);
  }
  auto kernel = dual_full(M, K)        ? quant_dual_kernel<true, true>
                : K % kDualCols == 0 ? quant_dual_kernel<false, true>
                                     : quant_dual_kernel<false, false>;
  return launch(kernel, dim3((unsigned)(slots * kXcds)), dim3(kDualThreads), 0, stream, static_cast<const uint16_t*>(x),
                static_cast<uint32_t*>(row_q), static_cast<uint8_t*>(row_s), static_cast<uint8_t*>(col_q),
                static_cast<uint8_t*>(col_s), M, K, (int)tiles_m, (int)tiles, units, eps,
                host_c_eps(eps, 6.0f));
}

hipError_t launch_quant_dual_grouped(const DualSpec* items, int count, float eps, hipStream_t stream) {
  for (int base = 0; base < count; base += kDualGroupMax) {
    DualGroupFours g;
    memset(&g, 0, sizeof(g));
    g.count = count - base < kDualGroupMax ? count - base : kDualGroupMax;
    bool full = true, lines = true, single = true;
    int tiles = 0, slots[kXcds] = {};  // of the items so far: tiles, and each XCD's share
    for (int j = 0; j < g.count; j++) {
      const DualSpec& d = items[base + j];
      DualItem& it = g.item[j];
      it.x = static_cast<const uint16_t*>(d.x);
      it.row_q = static_cast<uint32_t*>(d.row_q);
      it.row_s = static_cast<uint8_t*>(d.row_s);
      it.col_q = static_cast<uint8_t*>(d.col_q);
      it.col_s = static_cast<uint8_t*>(d.col_s);
      it.M = d.M;
      it.K = d.K;
      const int64_t tiles_m = (d.M + kDualRows - 1) / kDualRows;
      const int bands = d.M == 0 ? 0 : (int)((d.K + kDualCols - 1) / kDualCols);
      it.units = band_units(tiles_m, bands, bands > kDualWideBands ? kDualQuadShift : 0);
      tiles += (int)tiles_m * bands;
      for (int x = 0; x < kXcds; x++) slots[x] += g.share[x][j] = band_group_tiles(x, it.units);
      full = full && dual_full(d.M, d.K);
      lines = lines && d.K % kDualCols == 0;
      single = single && it.units.shift == 0;
    }
    if (tiles == 0) continue;
    g.eps = eps;
    g.c_eps = host_c_eps(eps, 6.0f);
    const dim3 grid((unsigned)(*std::max_element(slots, slots + kXcds) * kXcds));
    const hipError_t e =
        single ? launch(full    ? quant_dual_grouped_kernel<true, true, DualGroup>
                        : lines ? quant_dual_grouped_kernel<false, true, DualGroup>
                                : quant_dual_grouped_kernel<false, false, DualGroup>,
                        grid, dim3(kDualThreads), 0, stream, static_cast<const DualGroup&>(g))
               : launch(full    ? quant_dual_grouped_kernel<true, true, DualGroupFours>
                        : lines ? quant_dual_grouped_kernel<false, true, DualGroupFours>
                                : quant_dual_grouped_kernel<false, false, DualGroupFours>,
                        grid, dim3(kDualThreads), 0, stream, g);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace omo_hip

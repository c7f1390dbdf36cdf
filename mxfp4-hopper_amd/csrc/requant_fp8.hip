// MXFP4 -> FP8 E4M3 requant, rowwise (1x128 power-of-two scales stored
// transposed) and the transposed-output variant.
//
// Rowwise semantics follow omo_per_token_Mxfp4ToFp8_kernel
// (code/kernel/per_token_Mxfp4ToFp8.cu:92-235). Per 128-element group G
// (64 code bytes, 4 E8M0 bytes s[4G..4G+3]):
//   g   = (uint16)(max(s) - 6)                                 :162-165
//   y_s = fp32 with bits ((uint8)g) << 23, stored at [col*M + row] :172-180
//   per element: bf16(code) - ((uint16)(g - s_i) << 7) (mod 2^16), as fp32,
//   clamped by fmaxf(-448, fminf(448, .)), then E4M3 RNE.       :192-229
// The modular subtraction is kept exactly, including its wrap for zero
// codes (-448 when s_i <= max(s) - 7) and for max(s) < 6.
//
// Transposed semantics follow omo_per_token_Mxfp4ToFp8_col_kernel
// (code/kernel/per_token_Mxfp4ToFp8_col.cu:110-301) on 128-row x 128-byte
// tiles: per MX column c of the tile g_c = (uint8)(max(eps8, max_rows s) - 6),
// y_s(g_c) replicated over the column's 32 outputs of scale row by (:183-212),
// element value (bf16(code) - ((uint8)(g_c - s) << 7)) & 0x7FFF (sign
// dropped, :244-274), clamped by fminf(fmaxf(., -448), 448), E4M3 RNE, and
// written to [element_column * M + row] (:282-290).
#include "omo_device.cuh"
#include "omo_internal.h"

namespace omo_hip {

// ---------------------------------------------------------------- rowwise
// A code dword (8 elements) becomes 8 FP8 bytes; a lane converts two of them.
//
// The reference subtracts off = 128 * (adjust mod 512) from the bf16 pattern
// of each code, adjust = (uint16)(g - s_i). Write d for the signed value of
// adjust mod 512. Subtracting a multiple of 128 never touches the low 7 bits
// and flips bit 15 exactly when the code is negative, so the result for a
// negative code is the result for its magnitude with the sign flipped; after
// the symmetric clamp and E4M3 rounding that is a flip of bit 7, except
// where the pattern is a NaN (both signs clamp to +448).
//
// Fast path, d in [-6, 5]: code * 2^-d is a normal E4M3 value for every
// nonzero magnitude (0.5 * 2^-5 = 2^-6 at the bottom, 6 * 2^6 = 384 at the
// top), so its byte is the E4M3 pattern of the code with -d added to the
// exponent field: {0x30, 0x38, 0x3C, 0x40, 0x44, 0x48, 0x4C} - 8d. A zero
// code gives 0 for d <= 0 and the wrapped -inf -> -448 (0xFE) for d >= 1.
// No NaN pattern arises in this range. The eight bytes form a per-lane
// table (t_hi:t_lo); v_perm_b32 looks up four elements per instruction.
//
// d = x - 6 with x = max(s) - s_i: the reference's adjust (uint16)(g - s_i)
// is x - 6 modulo 2^16, and x lies in [0, 255], so d in [-6, 5] is x <= 11.
__device__ __forceinline__ void fp8_table(uint32_t x, uint32_t& t_lo, uint32_t& t_hi) {
  // 8x (at most 88) in every byte. With 48 added to each base byte no byte
  // of the difference borrows, so the dword subtraction is per byte:
  // byte = base + 48 - 8x = base - 8d.
  const uint32_t x8 = x << 3;
  const uint32_t rep = __builtin_amdgcn_perm(x8, x8, 0u);
  t_hi = 0x7C787470u - rep;
  const uint32_t lo = 0x6C686058u - rep;  // byte 0 (0x58 - 8x) is replaced below
  t_lo = __builtin_amdgcn_perm(x >= 7u ? 0xFEu : 0u, lo, 0x03020104u);
}

// 8 elements of the code dword c under table (t_hi:t_lo). The low and high
// nibbles of the four code bytes are looked up separately (3-bit magnitude),
// their sign bits (bits 3 and 7 of each code byte) moved to bit 7 of the
// looked-up bytes by one bitop3 each (x ^ (y & 0x80808080)), and the two
// lookups interleaved into element order.
__device__ __forceinline__ u32x2 to_fp8_dword_fast(uint32_t c, uint32_t t_lo, uint32_t t_hi) {
  uint32_t lo = __builtin_amdgcn_perm(t_hi, t_lo, c & 0x07070707u);         // elements 0, 2, 4, 6
  uint32_t hi = __builtin_amdgcn_perm(t_hi, t_lo, (c >> 4) & 0x07070707u);  // elements 1, 3, 5, 7
  lo = __builtin_amdgcn_bitop3_b32(lo, c << 4, 0x80808080u, 0x78);
  hi = __builtin_amdgcn_bitop3_b32(hi, c, 0x80808080u, 0x78);
  u32x2 o;
  o[0] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
  o[1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
  return o;
}

// Reference restatement for one code dword under the 16-bit offset `offset`.
__device__ __forceinline__ u32x2 to_fp8_dword_ref(uint32_t c, uint32_t offset) {
  uint32_t lo = 0, hi = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t byte = (c >> (8 * k)) & 0xFFu;
    const uint32_t a0 = (e2m1_to_bf16_bits(byte & 0xFu) - offset) & 0xFFFFu;
    const uint32_t a1 = (e2m1_to_bf16_bits(byte >> 4) - offset) & 0xFFFFu;
    const float f0 = fmaxf(-448.0f, fminf(448.0f, bf16_to_f32(a0)));
    const float f1 = fmaxf(-448.0f, fminf(448.0f, bf16_to_f32(a1)));
    const uint32_t pr = fp8x2_from_f32(f0, f1);
    if (k < 2) lo |= pr << (16 * k); else hi |= pr << (16 * (k - 2));
  }
  u32x2 o;
  o[0] = lo;
  o[1] = hi;
  return o;
}

// Block tile: ROWS rows x kRqGroups groups of 128 elements (256 code bytes
// per row). Lane e of the tile (e = u * 256 + t) converts code pair
// c = e % (8 kRqGroups) of tile row e / (8 kRqGroups): 16 B stores,
// contiguous over 16-lane row pieces. The fp32 scales of a tile land in
// kRqGroups runs of ROWS consecutive floats of the transposed scale tensor
// [K/128, M]: a whole 128 B line with 32-row tiles, half of one with 16-row
// tiles, whose other half comes from the next row tile, placed on the same
// XCD by the contiguous renumbering below, so no line is assembled from
// partial writes on different XCDs. FP8 bytes are written non-temporally
// (the fp32 scales, 64 B pieces of lines, ordinarily: non-temporal they
// took 4096 x 7168 from 7.8 to 9.4 us); codes are read with ordinary
// loads (non-temporal code loads made this kernel and the transposed one
// 15-16% slower). The tile height (ROWS) is 16 rows without a gather and 32
// with one (the launcher says why); inputs of few rows take 8-row tiles, so
// that a launch still spreads over the CUs: 128 x 7168 ran 3.2 us in 56 tiles
// of 32 rows; its scale runs are then 32 B pieces of lines that four
// workgroups share.
constexpr int kRqGroups = 4;
constexpr int kRqRows = 32;
constexpr int kRqRowsPlain = 16;
constexpr int kRqRowsSmall = 8;
// Codes of row r start at q + r * q_stride and its scale bytes at
// s + r * s_stride (bytes): contiguous [M, Kb] + [M, Kb/16] tensors, or the
// expert-parallel payload rows [codes | scales] read in place. ALIGN8: the
// code rows are 8-byte aligned (one 8 B load per lane, else two 4 B loads).
// src (optional): output row r reads input row src[r] (a gather, e.g. the
// expert-major token order of a MoE permutation); an index outside
// [0, n_src) reads zero codes and zero scale bytes, i.e. the row a permutation
// pads with zeros, requantized. src_out (optional): a copy of src, so that a
// row order built in a larger buffer needs no copy launch of its own.
// ROWS64: rows addressed with 64-bit products (a gather, or strides or
// output rows of 2^24 bytes and more); otherwise addresses are a
// workgroup-uniform tile base plus 32-bit lane offsets (24-bit products).
// TAIL: the input rows end inside the last group: kb code bytes (a multiple
// of 16) and ks = kb / 16 scale bytes a row. The output is that of rows
// padded with zero codes and zero scale bytes to whole groups: pairs past the
// row read its last pair and are zeroed, and a group's four scale bytes, at
// any byte alignment, are read as one dword that ends at the row's end at the
// latest, shifted down. Padding by torch first (two fills, two copies, then
// this kernel) took 23 us of kernels at 4096 x 2880, this form 6.
template <int ROWS, bool ALIGN8, bool ROWS64, bool TAIL>
__global__ __launch_bounds__(256) void mxfp4_to_fp8_kernel(const uint8_t* __restrict__ q, int64_t q_stride,
                                                           const uint8_t* __restrict__ s, int64_t s_stride,
                                                           const int32_t* __restrict__ src, int64_t n_src,
                                                           u32x4* __restrict__ out, float* __restrict__ out_s,
                                                           uint32_t M, uint32_t gpr, uint32_t gx, uint32_t kb,
                                                           uint32_t ks, int32_t* __restrict__ src_out) {
  constexpr int PPR = 8 * kRqGroups;  // pairs per tile row
  constexpr int UNROLL = ROWS * PPR / 256;
  constexpr int RSTEP = 256 / PPR;    // rows between one lane's pairs
  const uint32_t L = xcd_contiguous(blockIdx.x, gridDim.x);
  const uint32_t bx = L % gx, by = L / gx;
  const uint32_t t = threadIdx.x;
  const uint32_t row0 = by * ROWS;                 // first row of the tile
  const uint32_t cp = bx * PPR + t % PPR;          // the lane's pair column, the same in each of its rows
  const uint32_t cpc = min(cp, (TAIL ? kb / 8 : 8 * gpr) - 1);
  // the lane's scale dword: byte offset in the row, and how far down its bytes move
  const uint32_t so = TAIL ? min(4 * (cpc >> 3), max(ks, 4u) - 4) : 4 * (cpc >> 3);
  const uint32_t sdown = TAIL ? 8 * (4 * (cpc >> 3) - so) : 0;
  const uint32_t lr0 = t / PPR;                    // the lane's first row within the tile
  // Every load is issued at clamped in-bounds indices (and zeroed afterwards
  // for a padding row): loads under a per-lane branch made the compiler wait
  // for each pair's codes at the branch's join before issuing the next
  // pair's loads, so a lane had one pair in flight instead of all.
  const uint8_t* qp[UNROLL];
  const uint8_t* sp[UNROLL];
  bool pad[UNROLL];
  if (ROWS64) {
    int64_t sr[UNROLL];
    if (src) {
#pragma unroll
      for (int u = 0; u < UNROLL; u++) sr[u] = src[min(row0 + lr0 + u * RSTEP, M - 1)];
      if (src_out && bx == 0 && t % PPR == 0) {
#pragma unroll
        for (int u = 0; u < UNROLL; u++)
          if (row0 + lr0 + u * RSTEP < M) src_out[row0 + lr0 + u * RSTEP] = (int32_t)sr[u];
      }
    } else {
#pragma unroll
      for (int u = 0; u < UNROLL; u++) sr[u] = min(row0 + lr0 + u * RSTEP, M - 1);
    }
#pragma unroll
    for (int u = 0; u < UNROLL; u++) {
      pad[u] = sr[u] < 0 || sr[u] >= n_src;
      const int64_t row = pad[u] ? 0 : sr[u];
      qp[u] = q + row * q_stride + 8 * cpc;
      sp[u] = s + row * s_stride + so;
    }
  } else {
    const uint8_t* qt = q + (int64_t)row0 * q_stride;
    const uint8_t* st = s + (int64_t)row0 * s_stride;
#pragma unroll
    for (int u = 0; u < UNROLL; u++) {
      const uint32_t lr = min(row0 + lr0 + u * RSTEP, M - 1) - row0;
      qp[u] = qt + (__umul24(lr, (uint32_t)q_stride) + 8 * cpc);
      sp[u] = st + (__umul24(lr, (uint32_t)s_stride) + so);
      pad[u] = false;
    }
  }
  u32x2 c[UNROLL];
  uint32_t sd[UNROLL];
  if (n_src > 0) {
#pragma unroll
    for (int u = 0; u < UNROLL; u++) {
      if (ALIGN8) {
        c[u] = *reinterpret_cast<const u32x2*>(qp[u]);
      } else {
        c[u][0] = *reinterpret_cast<const uint32_t*>(qp[u]);
        c[u][1] = *reinterpret_cast<const uint32_t*>(qp[u] + 4);
      }
      if (!TAIL) {
        sd[u] = *reinterpret_cast<const uint32_t*>(sp[u]);
      } else if (ks >= 4) {
        __builtin_memcpy(&sd[u], sp[u], 4);
      } else {  // rows of one to three blocks
        sd[u] = sp[u][0];
        if (ks > 1) sd[u] |= (uint32_t)sp[u][1] << 8;
        if (ks > 2) sd[u] |= (uint32_t)sp[u][2] << 16;
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < UNROLL; u++) c[u][0] = c[u][1] = sd[u] = 0u;
  }
#pragma unroll
  for (int u = 0; u < UNROLL; u++) {
    if (pad[u]) c[u][0] = c[u][1] = sd[u] = 0u;
    if (TAIL) {
      sd[u] >>= sdown;
      if (8 * cp >= kb) c[u][0] = c[u][1] = 0u;
    }
  }
  const uint32_t sh = 8 * ((t & 7u) >> 1);  // byte of s_i in the group's scale dword (cp & 7 == t & 7)
  u32x4* ot = out + (int64_t)row0 * (8 * (int64_t)gpr) + bx * PPR;
  float* os = out_s + (int64_t)(bx * kRqGroups) * M + row0;
  // Every pair is converted before the first store: a store ahead of the
  // next pair's conversion made the wait for that pair's loads wait for the
  // store as well (loads and stores share one counter).
  u32x4 ov[UNROLL];
  uint32_t gs[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; u++) {
    const uint32_t sw = sd[u];
    const uint32_t smax = max(max(sw & 0xFFu, (sw >> 8) & 0xFFu), max((sw >> 16) & 0xFFu, sw >> 24));
    const uint32_t s_i = (sw >> sh) & 0xFFu;
    const uint32_t x = smax - s_i;
    u32x2 o0, o1;
    if (x <= 11u) {
      uint32_t t_lo, t_hi;
      fp8_table(x, t_lo, t_hi);
      o0 = to_fp8_dword_fast(c[u][0], t_lo, t_hi);
      o1 = to_fp8_dword_fast(c[u][1], t_lo, t_hi);
    } else {
      const uint32_t offset = ((smax - 6u - s_i) << 7) & 0xFFFFu;  // (uint16)(g - s_i) << 7
      o0 = to_fp8_dword_ref(c[u][0], offset);
      o1 = to_fp8_dword_ref(c[u][1], offset);
    }
    ov[u][0] = o0[0];
    ov[u][1] = o0[1];
    ov[u][2] = o1[0];
    ov[u][3] = o1[1];
    gs[u] = ((smax - 6u) & 0xFFu) << 23;
  }
#pragma unroll
  for (int u = 0; u < UNROLL; u++) {
    const uint32_t lr = lr0 + u * RSTEP;
    if (row0 + lr >= M || cp >= 8 * gpr) continue;
    if (ROWS64) {
      __builtin_nontemporal_store(ov[u], ot + ((int64_t)lr * (8 * gpr) + t % PPR));
    } else {
      const uint32_t ob = (__umul24(lr, 8 * gpr) + t % PPR) * 16u;  // byte offset in the tile, below 2^29
      __builtin_nontemporal_store(ov[u], reinterpret_cast<u32x4*>(reinterpret_cast<uint8_t*>(ot) + ob));
    }
    if ((t & 7u) == 0) os[((t % PPR) >> 3) * M + lr] = __uint_as_float(gs[u]);
  }
}

hipError_t launch_mxfp4_to_fp8_rows(const void* q, int64_t q_stride, const void* s, int64_t s_stride,
                                    const int32_t* src, int64_t n_src, int32_t* src_out, void* out, float* out_s,
                                    int64_t M, int64_t Kb, hipStream_t stream) {
  if (M == 0 || Kb == 0) return hipSuccess;
  const int64_t gpr = (Kb + 63) / 64;
  const bool tail = Kb % 64 != 0;
  const int64_t gx = (gpr + kRqGroups - 1) / kRqGroups;
  const bool small = gx * ((M + kRqRows - 1) / kRqRows) < 2 * (int64_t)current_device_caps().cus;
  // Without a gather, 16-row tiles (two pairs per lane, twice the workgroups)
  // hide more of the conversion: 4096 x 7168 7.99 against 8.15 us (7.80
  // against 7.95 with every store after all conversions). With one,
  // the 32-row tiles keep four gathered rows' loads in flight per lane: the
  // gathered requant of 32868 rows 50.4 against 53.1 us with 16-row tiles.
  const int rows = small ? kRqRowsSmall : (src ? kRqRows : kRqRowsPlain);
  const int64_t gy = (M + rows - 1) / rows;
  const bool a8 = (q_stride % 8 == 0) && ((reinterpret_cast<uintptr_t>(q) & 7) == 0);
  const bool r64 = src || q_stride >= (1 << 24) || s_stride >= (1 << 24) || 128 * gpr >= (1 << 24);
  using Kernel = void (*)(const uint8_t*, int64_t, const uint8_t*, int64_t, const int32_t*, int64_t, u32x4*, float*,
                          uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, int32_t*);
  // [rows: 8, 16, 32][a8][r64]
  static const Kernel table[3][2][2] = {
      {{mxfp4_to_fp8_kernel<kRqRowsSmall, false, false, false>, mxfp4_to_fp8_kernel<kRqRowsSmall, false, true, false>},
       {mxfp4_to_fp8_kernel<kRqRowsSmall, true, false, false>, mxfp4_to_fp8_kernel<kRqRowsSmall, true, true, false>}},
      {{mxfp4_to_fp8_kernel<kRqRowsPlain, false, false, false>, mxfp4_to_fp8_kernel<kRqRowsPlain, false, true, false>},
       {mxfp4_to_fp8_kernel<kRqRowsPlain, true, false, false>, mxfp4_to_fp8_kernel<kRqRowsPlain, true, true, false>}},
      {{mxfp4_to_fp8_kernel<kRqRows, false, false, false>, mxfp4_to_fp8_kernel<kRqRows, false, true, false>},
       {mxfp4_to_fp8_kernel<kRqRows, true, false, false>, mxfp4_to_fp8_kernel<kRqRows, true, true, false>}}};
  // rows ending inside a group (no gather, 8 B aligned rows): [rows: 8, 16][r64]
  static const Kernel tails[2][2] = {
      {mxfp4_to_fp8_kernel<kRqRowsSmall, true, false, true>, mxfp4_to_fp8_kernel<kRqRowsSmall, true, true, true>},
      {mxfp4_to_fp8_kernel<kRqRowsPlain, true, false, true>, mxfp4_to_fp8_kernel<kRqRowsPlain, true, true, true>}};
  if (tail && (src || !a8)) return hipErrorInvalidValue;
  const int ri = rows == kRqRowsSmall ? 0 : rows == kRqRowsPlain ? 1 : 2;
  return launch(tail ? tails[ri][r64] : table[ri][a8][r64], dim3((unsigned)(gx * gy)), dim3(256), 0, stream,
                static_cast<const uint8_t*>(q), q_stride, static_cast<const uint8_t*>(s), s_stride, src, n_src,
                static_cast<u32x4*>(out), out_s, (uint32_t)M, (uint32_t)gpr, (uint32_t)gx, (uint32_t)Kb,
                (uint32_t)(Kb / 16), src_out);
}

hipError_t launch_mxfp4_to_fp8(const void* q, const void* s, void* out, float* out_s, int64_t M, int64_t Kb,
                               hipStream_t stream) {
  return launch_mxfp4_to_fp8_rows(q, Kb, s, Kb / 16, nullptr, M, nullptr, out, out_s, M, Kb, stream);
}

// ------------------------------------------------------------ transposed
// One 256-thread block per 128-row x 128-byte tile (256 element columns).
//
// The per-element rule of the reference (:244-290) is
//   byte = E4M3(clamp(bf16((bits(code) - (adj << 7)) mod 2^16 & 0x7FFF)))
// with adj = (uint8)(g - s_row). Subtracting a multiple of 128 never touches
// the low 7 bits, and for a negative code the subtraction and the final
// & 0x7FFF give the same pattern as for its magnitude (the sign bit only
// changes where the borrow lands above bit 14, which the mask removes). So
// the byte is a function of (adj, |code|) alone: a 256 x 8 table, built per
// block in LDS by restating the reference rule for every entry. Each lane
// then needs one 8-byte table row per tile row and v_perm_b32 lookups.
//
// Lane mapping: lane t owns code bytes 4c .. 4c+3 (element columns 8c ..
// 8c+7, one MX column), c = t / 8, and rows 16q .. 16q+15, q = t % 8; the 8
// lanes of a code dword write its 8 element columns' 128 output rows as one
// full 128 B line each per store instruction. Per row a lane reads one code
// dword and one 8-byte table row; the magnitudes of the four low nibbles
// (cw & 0x07070707) and of the four high nibbles ((cw >> 4) & 0x07070707)
// are the v_perm_b32 selectors that look up the four even and the four odd
// element columns' bytes, and 4x4 byte transposes (eight v_perm_b32 each)
// turn four rows of those into 4-row pieces of the output columns.
constexpr int kColTile = 128;
constexpr int kColPitch = kColTile + 32;  // 16 B aligned LDS rows; 40 dwords keep a wave's row reads on distinct banks

struct ColSmem {
  uint8_t codes[kColTile * kColPitch];
  uint8_t scales[8][kColTile];   // [MX column of the tile][row]
  uint32_t table[256][2];        // fp8 byte of |code| = 0..7 under adj (bytes 0..7)
  uint32_t gpart[8][4];          // per MX column, per wave partial maxima
};

// LDS row of tile row r: rows 16q + j (q = 0..7) are read together, so they
// are stored in consecutive LDS rows (distinct banks for pitch 144).
__device__ __forceinline__ int col_lds_row(int r) { return ((r & 15) << 3) | (r >> 4); }

// fp8 bytes of magnitudes 0..7 under adj, by the reference rule.
__device__ __forceinline__ void col_table_row(uint32_t adj, uint32_t* lo, uint32_t* hi) {
  uint32_t w[2] = {0u, 0u};
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const uint32_t a = ((e2m1_to_bf16_bits((uint32_t)c) - (adj << 7)) & 0xFFFFu) & 0x7FFFu;
    const float f = fminf(fmaxf(bf16_to_f32(a), -448.0f), 448.0f);
    w[c >> 2] |= (fp8x2_from_f32(f, f) & 0xFFu) << (8 * (c & 3));
  }
  *lo = w[0];
  *hi = w[1];
}

__global__ __launch_bounds__(256) void mxfp4_to_fp8_col_kernel(const uint8_t* __restrict__ q,
                                                               const uint8_t* __restrict__ s,
                                                               uint8_t* __restrict__ out, float* __restrict__ out_s,
                                                               int64_t M, int64_t Kb, uint32_t eps8) {
  __shared__ ColSmem sm;
  const int t = threadIdx.x;
  const uint32_t L = xcd_contiguous(blockIdx.x, gridDim.x), gx = (uint32_t)(Kb / kColTile);
  const int64_t bx = L % gx, by = L / gx;
  const int64_t row0 = by * kColTile;
  // ---- stage codes (1024 chunks of 16 B: 8 rows x 128 B per wave load) and scales
  u32x4 cv[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int id = t + 256 * k, r = id >> 3, c16 = id & 7;
    cv[k] = *reinterpret_cast<const u32x4*>(q + (row0 + r) * Kb + bx * kColTile + c16 * 16);
  }
  u32x2 sv = {0u, 0u};
  if (t < kColTile) sv = *reinterpret_cast<const u32x2*>(s + (row0 + t) * (Kb / 16) + bx * 8);
  {
    uint32_t lo, hi;
    col_table_row((uint32_t)t, &lo, &hi);
    sm.table[t][0] = lo;
    sm.table[t][1] = hi;
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int id = t + 256 * k, r = id >> 3, c16 = id & 7;
    *reinterpret_cast<u32x4*>(sm.codes + col_lds_row(r) * kColPitch + c16 * 16) = cv[k];
  }
  if (t < kColTile) {
#pragma unroll
    for (int c = 0; c < 8; c++) sm.scales[c][t] = (uint8_t)(sv[c >> 2] >> (8 * (c & 3)));
  }
  __syncthreads();
  // ---- g per MX column: (uint8)(max(eps8, max over 128 rows) - 6)
  {
    const int c = t >> 5, r4 = (t & 31) * 4;  // a wave covers two MX columns
    const uint32_t w = *reinterpret_cast<const uint32_t*>(&sm.scales[c][r4]);
    uint32_t m = max(max(w & 0xFFu, (w >> 8) & 0xFFu), max((w >> 16) & 0xFFu, w >> 24));
#pragma unroll
    for (int x = 1; x < 32; x <<= 1) m = max(m, (uint32_t)__shfl_xor((int)m, x));
    if ((t & 31) == 0) sm.gpart[c][0] = (max(m, eps8) - 6u) & 0xFFu;
  }
  __syncthreads();
  // scale row of the tile: 256 floats, entry e holds MX column e / 32 (:210-212)
  __builtin_nontemporal_store(__uint_as_float(sm.gpart[t >> 5][0] << 23), out_s + by * (Kb * 2) + bx * 256 + t);
  const int qq = t & 7, cg = t >> 3, mx = cg >> 2;
  const uint32_t g = sm.gpart[mx][0];
  const u32x4 sw = *reinterpret_cast<const u32x4*>(&sm.scales[mx][16 * qq]);
  u32x4 col[8];  // element column 8cg + k: rows 16qq + 4a .. 16qq + 4a + 3 in dword a
#pragma unroll
  for (int a = 0; a < 4; a++) {
    uint32_t ev[4], od[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t cw = *reinterpret_cast<const uint32_t*>(sm.codes + col_lds_row(16 * qq + 4 * a + i) * kColPitch + 4 * cg);
      const uint32_t adj = (g - ((sw[a] >> (8 * i)) & 0xFFu)) & 0xFFu;
      const u32x2 tr = *reinterpret_cast<const u32x2*>(&sm.table[adj][0]);
      ev[i] = __builtin_amdgcn_perm(tr[1], tr[0], cw & 0x07070707u);
      od[i] = __builtin_amdgcn_perm(tr[1], tr[0], (cw >> 4) & 0x07070707u);
    }
    // byte m of ev[i] / od[i] is element column 8cg + 2m / 2m + 1 of row 4a + i
    const uint32_t e0 = __builtin_amdgcn_perm(ev[1], ev[0], 0x05010400u), e1 = __builtin_amdgcn_perm(ev[1], ev[0], 0x07030602u);
    const uint32_t e2 = __builtin_amdgcn_perm(ev[3], ev[2], 0x05010400u), e3 = __builtin_amdgcn_perm(ev[3], ev[2], 0x07030602u);
    const uint32_t o0 = __builtin_amdgcn_perm(od[1], od[0], 0x05010400u), o1 = __builtin_amdgcn_perm(od[1], od[0], 0x07030602u);
    const uint32_t o2 = __builtin_amdgcn_perm(od[3], od[2], 0x05010400u), o3 = __builtin_amdgcn_perm(od[3], od[2], 0x07030602u);
    col[0][a] = __builtin_amdgcn_perm(e2, e0, 0x05040100u);
    col[2][a] = __builtin_amdgcn_perm(e2, e0, 0x07060302u);
    col[4][a] = __builtin_amdgcn_perm(e3, e1, 0x05040100u);
    col[6][a] = __builtin_amdgcn_perm(e3, e1, 0x07060302u);
    col[1][a] = __builtin_amdgcn_perm(o2, o0, 0x05040100u);
    col[3][a] = __builtin_amdgcn_perm(o2, o0, 0x07060302u);
    col[5][a] = __builtin_amdgcn_perm(o3, o1, 0x05040100u);
    col[7][a] = __builtin_amdgcn_perm(o3, o1, 0x07060302u);
  }
  uint8_t* o = out + (bx * 256 + 8 * cg) * M + row0 + 16 * qq;
#pragma unroll
  for (int k = 0; k < 8; k++) __builtin_nontemporal_store(col[k], reinterpret_cast<u32x4*>(o + k * M));
}

hipError_t launch_mxfp4_to_fp8_col(const void* q, const void* s, void* out, float* out_s, int64_t M, int64_t Kb,
                                   float eps, hipStream_t stream) {
  if (M == 0 || Kb == 0) return hipSuccess;
  uint32_t eps8 = 0;
  if (eps > 0.0f) eps8 = eps >= 255.0f ? 255u : (uint32_t)eps;  // (uint8_t)eps, truncating
  // 1-D grid, tile index bx fastest, renumbered per XCD in the kernel
  const dim3 grid((unsigned)((Kb / kColTile) * (M / kColTile)));
  return launch(mxfp4_to_fp8_col_kernel, grid, dim3(256), 0, stream, static_cast<const uint8_t*>(q),
                     static_cast<const uint8_t*>(s), static_cast<uint8_t*>(out), out_s, M, Kb, eps8);
}

}  // namespace omo_hip

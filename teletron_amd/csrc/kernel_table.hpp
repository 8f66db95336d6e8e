// Table of compiled kernel variants and the host-side lookup that maps a row
// width to one of them.  Each of the four kernel families (AdaLN / RMSNorm x
// forward / backward) is instantiated in its own translation unit through the
// lookup templates below, so the families compile in parallel.
#pragma once
#include "gate_kernels.hpp"
#include "norm_kernels.hpp"
#include "resnorm_kernels.hpp"

namespace tt {

struct KernelInfo {
  const void* fn;   // __global__ function taking one FwdArgs / BwdArgs by value
  int threads;      // workgroup size
  int tile_rows;    // rows one workgroup consumes per loop iteration
  int lane_loads;   // 128-bit loads per lane and streamed tensor in one tile
};

// Wide variants: (index, W waves per row, P packs per lane).  A row of `packs`
// 128-bit packs runs on the variant with the fewest lane slots 64*W*P >= packs.
#define TT_WIDE_LIST(X) \
  X(0, 1, 1) X(1, 2, 1) X(2, 3, 1) X(3, 4, 1) X(4, 3, 2) X(5, 4, 2) X(6, 5, 2) \
  X(7, 6, 2) X(8, 8, 2) X(9, 12, 2) X(10, 16, 2) X(11, 16, 4)
constexpr int kNumWide = 12;
constexpr int kWideW[kNumWide] = {1, 2, 3, 4, 3, 4, 5, 6, 8, 12, 16, 16};
constexpr int kWideP[kNumWide] = {1, 1, 1, 1, 2, 2, 2, 2, 2, 2, 2, 4};

// Narrow variants: (index, L lanes per row).
#define TT_NARROW_LIST(X) X(0, 1) X(1, 2) X(2, 4) X(3, 8) X(4, 16) X(5, 32)
constexpr int kNumNarrow = 6;
constexpr int kNarrowL[kNumNarrow] = {1, 2, 4, 8, 16, 32};
constexpr int kNarrowMaxPacks = 32;
constexpr int kMaxPacks = 64 * 16 * 4;

// ---- tuning constants, from sweeps on MI355X (see make_plan in capi.hip for the grid rule)
// R: rows in flight per row group;  Q: row groups per workgroup.  HBM throughput peaks with
// roughly 18 (forward) / 12 (backward, two input tensors) outstanding 128-bit loads per lane
// column of a CU and tensor, and barrier-coupled row groups in ONE workgroup per CU stream
// better than independent workgroups; Q is chosen so that one workgroup carries that load.
constexpr int kNarrowR = 2;    // loads per lane and tensor in flight, narrow kernels
// RMSNorm backward on narrow rows streams better with six loads per lane in ONE four-wave workgroup
// per CU than with two loads in two workgroups: 2,851,200 x 128 backward 362 -> 354 us between
// forward launches (reference contract 371 -> 358 us), 1-1.5 % at 32, 64 and 256 columns.  Forward
// and the AdaLN kernels lose with six (128 columns forward 242 -> 269 us, AdaLN backward 359 -> 363 us).
constexpr int kNarrowRmsBwdR = 6;
// RMSNorm forward on narrow rows with every lane slot in use: six loads per lane as well.  As fast as
// two (2,851,200 x 128: 242 us either way; 16 ... 256 columns within 1 %), but with two the time depends
// on where the output lies relative to the input (period 128 MiB: 243 us over three quarters of it,
// up to 279 us over the rest), with six it does not (240-244 us at every offset).  Masked widths keep
// two (96 columns 282 -> 285 us, 200 columns 369 -> 382 us with six).
constexpr int kNarrowRmsFwdFullR = 6;
constexpr int kNarrowNW = 4;   // independent waves per workgroup, narrow kernels
constexpr int kFwdLoadsPerCu = 18;   // target waves x loads-per-lane per CU, forward
constexpr int kBwdLoadsPerCu = 12;   // same, backward (per input tensor)
constexpr int kFwdXnLoadsPerCu = 12; // same, AdaLN forward that also stores x_norm (see fwd_xn_wide_Q)

constexpr int fwd_wide_R(int W, int P) { return 1; }   // two rows per tile: 1-3 % slower at every width
constexpr int bwd_wide_R(int W, int P) { return 1; }
// AdaLN backward has two barrier-coupled reductions per row; on the variants below two rows per
// row group and tile (both rows share each exchange) hide that latency better.  Measured,
// us at R = 1 -> R = 2: 32760 x 1536: 53.8 -> 51.9; 4 x 32760 x 1536: 200.8 -> 198.0;
// 150000 x 2048: 300.9 -> 290.0; 118800 x 3072: 358.4 -> 348.9; 60000 x 6144: 381.2 -> 355.4;
// 300000 x 1024: 290.7 -> 288.5.  Worse with R = 2: 512 columns (156.9 -> 169.0), 4096
// (356.6 -> 368.8), 8192 (358.0 -> 399.5), and 5120 (ten waves: spills).  RMSNorm (one reduction
// per row) is 2-3 % slower with R = 2 everywhere.  Ragged rows lose with two as well (60000 x 2200:
// 162 -> 184 us, 1000: 71 -> 77 us).
constexpr int adaln_bwd_wide_R(int W, int P, int rows) {
  if (row_mode(rows) == kRagged || row_mode(rows) == kOdd) return bwd_wide_R(W, P);
  return ((P == 1 && W >= 2 && W <= 4) || (P == 2 && (W == 3 || W == 6))) ? 2 : bwd_wide_R(W, P);
}
constexpr int fwd_wide_Q(int W, int P) {
  return W >= 7 ? 1 : (10 + W / 2) / W;          // about 10 waves per workgroup
}
constexpr int bwd_wide_Q(int W, int P) {
  int q = (2 * kBwdLoadsPerCu + W * P) / (2 * W * P);   // round(12 / (W*P))
  if (q < 1) q = 1;
  if (W * q < 6) q = (6 + W - 1) / W;                   // at least 6 waves to keep up with the arithmetic
  while (q > 1 && W * q > 12) --q;                      // at most 12 waves: 170 VGPRs per lane
  return q;
}

// Ragged rows (kRagged): their stores and the lines that they share are slower, and more row groups a workgroup
// hide it on these variants.  us at the groups of whole-line rows -> with these, 400 MB tensors unless stated:
//   AdaLN forward      520 columns 211 -> 195,  776: 152 -> 148,  904: 138 -> 138,  1016: 146 -> 135 (eight groups of two waves);
//                      4104: 152 -> 124,  4616: 142 -> 126,  5112: 133 -> 125 (three of five)
//   RMSNorm forward    1016: 147 -> 136, and in the caches 520 (20 MB) 11.5 -> 9.3, 904 8.8 -> 8.0; beyond them shorter rows lose
//                      (520: 167 -> 191, 776: 142 -> 145, 968: 136 -> 138)
//   AdaLN and RMSNorm forward, four groups of four waves: 1928 columns 149 / 142 -> 136 / 133,  2040: 153 / 150 -> 138 / 135; with more
//                      lanes idle they lose, most at 80 MB (1544: 29.3 / 28.6 -> 32.8 / 31.6, 1800: 29.7 / 28.8 -> 31.2 / 29.9)
//                      Neither of the last with batches that leave CUs idle when each has whole workgroups of this size: 150 MB, 86 / 140
//                      batches, 600 columns 82 / 85 -> 97 / 115, 1992: 64 / 60 -> 69 / 77 (residual + norm 1992 125 / 124 -> 132 / 130)
//   and backward       3080: 226 / 201 -> 193 / 191,  3536: 204 / 200 -> 188 / 189,  4088: 197 / 195 -> 190 / 187
//   RMSNorm backward   520 (200 MB) 131 -> 115,  648: 114 -> 103,  776: 104 -> 99,  1016: 99 -> 100,  968 (12 MB) 9.0 -> 8.2; in the caches
//                      with over a quarter of the lanes idle two smaller workgroups a CU are better (520, 31 MB: 18.6 -> 20.6)
//   gate, either way   2200: 210 -> 190,  2600: 200 -> 188,  3080: 198 -> 189,  3536: 198 -> 189,  4088: 193 -> 188
//   residual + norm forward beyond the caches: 1544 columns, ungated / gated 272 / 261 -> 278 / 265,  1736: 279 -> 268,
//                      1928: 269 / 261 -> 260 / 251;  gated 1032: 328 -> 268,  1288: 281 -> 263,  1528: 269 -> 269; in the caches they
//                      lose (gated 1032, 6 / 20 MB 8.2 / 17.5 -> 8.9 / 18.3; 1864, 20 MB 15.4 -> 16.6)
// Not taken: forward and AdaLN backward of 2056 to 3064 columns (2200: 233 -> 217, but 2600: 205 -> 223); residual + norm forward
// with two packs a lane (4600: 187 -> 175, but 6 MB 6.4 -> 8.6); one pack a lane in the other backward kernels (no gain);
// residual backward (170 registers and more).
constexpr int ragged_fwd_Q(Kind kind, int W, int P, int rows) {
  if (row_mode(rows) != kRagged) return fwd_wide_Q(W, P);
  if (P == 1 && (W == 2 || W == 4) && (rows & kUneven)) return fwd_wide_Q(W, P);
  if (P == 1 && W == 2) return kind == kAdaLN || (rows & (kCached | kDense)) ? 8 : fwd_wide_Q(W, P);
  if (P == 1 && W == 4) return rows & kDense ? 4 : fwd_wide_Q(W, P);
  return kind == kAdaLN && P == 2 && W == 5 ? 3 : fwd_wide_Q(W, P);
}
constexpr int ragged_bwd_Q(Kind kind, int W, int P, int rows) {
  if (row_mode(rows) != kRagged) return bwd_wide_Q(W, P);
  if (kind == kRMS && P == 1 && W == 2) return (rows & kCached) && (rows & kIdle) ? bwd_wide_Q(W, P) : 8;
  return P == 2 && W == 4 ? 3 : bwd_wide_Q(W, P);
}
constexpr int ragged_gate_Q(int W, int P, int rows) {
  return row_mode(rows) == kRagged && P == 2 && (W == 3 || W == 4) ? 12 / W : bwd_wide_Q(W, P);
}

// Index of the wide variant for `packs` (> kNarrowMaxPacks), or -1.
inline int select_wide(int packs) {
  int best = -1, best_slots = 1 << 30;
  for (int i = 0; i < kNumWide; ++i) {
    const int slots = 64 * kWideW[i] * kWideP[i];
    // fewest slots wins; on a tie the later entry (more packs per lane, fewer waves) wins
    if (slots >= packs && slots <= best_slots) { best = i; best_slots = slots; }
  }
  return best;
}
inline int select_narrow(int packs) {
  for (int i = 0; i < kNumNarrow; ++i)
    if (kNarrowL[i] >= packs) return i;
  return -1;
}

template <int KIND, int W, int P, int ROWS>
KernelInfo info_fwd_wide() {
  constexpr int R = fwd_wide_R(W, P), Q = ragged_fwd_Q(static_cast<Kind>(KIND), W, P, ROWS);
  return {reinterpret_cast<const void*>(&norm_fwd_wide<KIND, W, P, R, Q, kernel_rows(W, P, ROWS, short_rows(W, P))>), 64 * W * Q, Q * R, P * R};
}
template <int KIND, int W, int P, int ROWS>
KernelInfo info_bwd_wide() {
  constexpr int R = KIND == kAdaLN ? adaln_bwd_wide_R(W, P, ROWS) : bwd_wide_R(W, P), Q = ragged_bwd_Q(static_cast<Kind>(KIND), W, P, ROWS);
  return {reinterpret_cast<const void*>(&norm_bwd_wide<KIND, W, P, R, Q, kernel_rows(W, P, ROWS, short_rows(W, P))>), 64 * W * Q, Q * R, P * R};
}
template <int KIND, int W, int P, int ROWS>
KernelInfo info_bwd_saved_wide() {
  constexpr int R = bwd_wide_R(W, P), Q = bwd_wide_Q(W, P);
  return {reinterpret_cast<const void*>(&norm_bwd_saved_wide<KIND, W, P, R, Q, kernel_rows(W, P, ROWS, false)>), 64 * W * Q, Q * R, P * R};
}
template <int KIND, int L, int ROWS>
KernelInfo info_bwd_saved_narrow() {
  constexpr int R = KIND == kRMS ? kNarrowRmsBwdR : kNarrowR, NW = kNarrowNW;
  return {reinterpret_cast<const void*>(&norm_bwd_saved_narrow<KIND, L, R, NW, ROWS>), 64 * NW, NW * R * (64 / L), R};
}
template <int KIND, int L, int ROWS>
KernelInfo info_fwd_narrow() {
  constexpr int R = (KIND == kRMS && row_mode(ROWS) == kFull) ? kNarrowRmsFwdFullR : kNarrowR, NW = kNarrowNW;
  return {reinterpret_cast<const void*>(&norm_fwd_narrow<KIND, L, R, NW, ROWS>), 64 * NW, NW * R * (64 / L), R};
}
template <int KIND, int L, int ROWS>
KernelInfo info_bwd_narrow() {
  constexpr int R = KIND == kRMS ? kNarrowRmsBwdR : kNarrowR, NW = kNarrowNW;
  return {reinterpret_cast<const void*>(&norm_bwd_narrow<KIND, L, R, NW, ROWS>), 64 * NW, NW * R * (64 / L), R};
}

// Return the instantiation for `rows` (enum Rows): of kernels for whole-line rows (CALL: the arguments), of all but odd
// rows, of all.
#define TT_LINES(INFO, CALL, ...)                                             \
  return rows == kFull             ? INFO<__VA_ARGS__, kFull> CALL            \
         : rows == (kFull | kKeep) ? INFO<__VA_ARGS__, kFull | kKeep> CALL    \
         : keeps(rows)             ? INFO<__VA_ARGS__, kMasked | kKeep> CALL  \
                                   : INFO<__VA_ARGS__, kMasked> CALL;
#define TT_LANES(INFO, ROWS, ...)                           \
  (rows & kIdle    ? INFO<__VA_ARGS__, (ROWS) | kIdle>()    \
   : rows & kDense ? INFO<__VA_ARGS__, (ROWS) | kDense>()   \
                   : INFO<__VA_ARGS__, (ROWS)>())
#define TT_ROWS(INFO, ...)                                                             \
  if (row_mode(rows) == kRagged)                                                       \
    return keeps(rows)      ? TT_LANES(INFO, kRagged | kKeep | kCached, __VA_ARGS__)   \
           : rows & kCached ? TT_LANES(INFO, kRagged | kCached, __VA_ARGS__)           \
           : rows & kUneven ? TT_LANES(INFO, kRagged | kUneven, __VA_ARGS__)           \
                            : TT_LANES(INFO, kRagged, __VA_ARGS__);                    \
  TT_LINES(INFO, (), __VA_ARGS__)
#define TT_ROWS_ODD(INFO, ...)                                      \
  if (row_mode(rows) == kOdd) return INFO<__VA_ARGS__, kOdd>();     \
  TT_ROWS(INFO, __VA_ARGS__)

// AdaLN forward that also stores x_norm (the reference's forward contract): one read and two
// write streams.  Bare streams of that mix (no arithmetic) reach 5.7-5.9 TB/s on MI355X (370-385 us
// for the 2.19 GB of 118800 x 3072), and like writes on their own they go fastest with FEW requests
// in flight: about 12 loads per lane column of a CU (kFwdXnLoadsPerCu), not the 18-20 of the
// one-output forward.  One row group per workgroup and several independent workgroups per CU:
// barrier-coupled row groups are 1 % faster at best (118800 x 3072: 379-383 us against 384-390) but
// 5-8 % slower (400-413 us) over a quarter of the possible placements of the two outputs relative to
// the input (period 128 MiB); independent workgroups stay at 384-393 us at every placement.
// Measured with this rule: 75600 x 5120 416 us, 131040 x 1536 213 us, 150000 x 2048 323 us.
constexpr int fwd_xn_wide_Q(int W, int P) { return 1; }
template <int W, int P, int ROWS>
KernelInfo info_fwd_xn_wide() {
  constexpr int R = fwd_wide_R(W, P), Q = fwd_xn_wide_Q(W, P);
  return {reinterpret_cast<const void*>(&norm_fwd_wide<kAdaLN, W, P, R, Q, kernel_rows(W, P, ROWS, false), false, true>), 64 * W * Q, Q * R, P * R};
}
template <int L, int ROWS>
KernelInfo info_fwd_xn_narrow() {
  constexpr int R = kNarrowR, NW = kNarrowNW;
  return {reinterpret_cast<const void*>(&norm_fwd_narrow<kAdaLN, L, R, NW, ROWS, 0, true>), 64 * NW, NW * R * (64 / L), R};
}
inline KernelInfo lookup_fwd_xn(bool narrow, int idx, int rows) {
  if (narrow) {
    switch (idx) {
#define X(i, L) case i: TT_LINES(info_fwd_xn_narrow, (), L)
      TT_NARROW_LIST(X)
#undef X
    }
  } else {
    switch (idx) {
#define X(i, W, P)                                                                  \
  case i:                                                                           \
    if (row_mode(rows) == kOdd) return info_fwd_xn_wide<W, P, kOdd>();              \
    TT_LINES(info_fwd_xn_wide, (), W, P)
      TT_WIDE_LIST(X)
#undef X
    }
  }
  return {nullptr, 0, 0, 0};
}

template <int KIND>
KernelInfo lookup_fwd(bool narrow, int idx, int rows) {
  if (narrow) {
    switch (idx) {
#define X(i, L) case i: TT_LINES(info_fwd_narrow, (), KIND, L)
      TT_NARROW_LIST(X)
#undef X
    }
  } else {
    switch (idx) {
#define X(i, W, P) case i: TT_ROWS_ODD(info_fwd_wide, KIND, W, P)
      TT_WIDE_LIST(X)
#undef X
    }
  }
  return {nullptr, 0, 0, 0};
}
template <int KIND>
KernelInfo lookup_bwd(bool narrow, int idx, int rows) {
  if (narrow) {
    switch (idx) {
#define X(i, L) case i: TT_LINES(info_bwd_narrow, (), KIND, L)
      TT_NARROW_LIST(X)
#undef X
    }
  } else {
    switch (idx) {
#define X(i, W, P) case i: TT_ROWS_ODD(info_bwd_wide, KIND, W, P)
      TT_WIDE_LIST(X)
#undef X
    }
  }
  return {nullptr, 0, 0, 0};
}

// RMSNorm with the rotary embedding fused behind it (wide rows only).
template <int W, int P, int ROWS>
KernelInfo info_fwd_rope_wide() {
  constexpr int R = fwd_wide_R(W, P), Q = fwd_wide_Q(W, P);
  return {reinterpret_cast<const void*>(&norm_fwd_wide<kRMS, W, P, R, Q, kernel_rows(W, P, ROWS, false), true>), 64 * W * Q, Q * R, P * R};
}
// Twelve waves where a lane holds two packs: the table's 64 bytes a pack make a lane's loads slower to come back than
// those of the plain backward, whose six to eight waves stream its x and dy (3072 columns 355 us with six, 372 with
// twelve).  us, bwd_wide_Q -> this: 60000 x 3072 191.6 -> 177.4, 86646 x 3072 273.8 -> 258.3, 40000 x 4096 163.5 ->
// 158.7, 40000 x 6144 252.7 -> 239.2; 5120 columns have ten either way.  One pack a lane is as fast or slower with other counts.
constexpr int bwd_rope_wide_Q(int W, int P) { return P == 2 && W <= 12 ? 12 / W : bwd_wide_Q(W, P); }
template <int W, int P, int ROWS>
KernelInfo info_bwd_rope_wide() {
  constexpr int R = bwd_wide_R(W, P), Q = bwd_rope_wide_Q(W, P);
  return {reinterpret_cast<const void*>(&norm_bwd_wide<kRMS, W, P, R, Q, kernel_rows(W, P, ROWS, false), true>), 64 * W * Q, Q * R, P * R};
}
template <int L, int ROWS>
KernelInfo info_fwd_rope_narrow() {
  constexpr int R = kNarrowR, NW = kNarrowNW;
  return {reinterpret_cast<const void*>(&norm_fwd_narrow<kRMS, L, R, NW, ROWS, 1>), 64 * NW, NW * R * (64 / L), R};
}
template <int L, int ROWS>
KernelInfo info_bwd_rope_narrow() {
  constexpr int R = kNarrowR, NW = kNarrowNW;
  return {reinterpret_cast<const void*>(&norm_bwd_narrow<kRMS, L, R, NW, ROWS, 1>), 64 * NW, NW * R * (64 / L), R};
}
// Token mode of the narrow ROPE kernels (ROPE = 2: the rows a wave takes per tile are heads of one
// token, so the (cos, sin) entries are loaded once per tile and lane).  R loads of 64 / L rows each have to
// divide a token's heads: instantiated for rows of 8 and 16 lanes (head_dim 40 ... 128), the largest of
// R = 6, 4, 3 that divides (24 heads of 128: 6, 16: 4, 12: 3; 24 heads of 64: 3).  Other head counts
// look every row up (ROPE = 1, two loads), and so do most tensors that fit the caches (make_plan).
// us forward / backward + reduction, per row -> per token: 2 x 60000 x 12 x 128 137 / 190 -> 127 / 184, 60000 x 16 x 128 92 / 128 -> 89 / 127, 2 x 60000 x 24 x 64
// 133 / 189 -> 127 / 183.  R = 5 is slower (60000 x 40 x 128 221 / 318 -> 227 / 321).
// One workgroup per CU with about 24 loads per lane column and tensor in flight measured best (24
// heads of 128, four waves of six: forward 245 us, backward + reduction 356 us at 118800 tokens; 5 / 6 / 8
// waves: 277 / 265 / 267 us forward, 378 / 368 / 380 us backward; 2 and 3 waves need 2-3 workgroups per
// CU and reach 259-265 us).
constexpr int kRopeTokenMinL = 8, kRopeTokenMaxL = 16;
constexpr int rope_token_NW(int R) { return R > 0 ? (24 + R / 2) / R : 0; }
template <int L, int R, int ROWS>
KernelInfo info_rope_token(bool backward) {
  constexpr int NW = rope_token_NW(R);
  if (backward)
    return {reinterpret_cast<const void*>(&norm_bwd_narrow<kRMS, L, R, NW, ROWS, 2>), 64 * NW, NW * R * (64 / L), R};
  return {reinterpret_cast<const void*>(&norm_fwd_narrow<kRMS, L, R, NW, ROWS, 2>), 64 * NW, NW * R * (64 / L), R};
}
// Loads per wave and tile in token mode, or 0 where `heads` rows per token do not allow it.
inline int rope_token_R(int L, int64_t heads) {
  if (L < kRopeTokenMinL || L > kRopeTokenMaxL || heads <= 0) return 0;
  for (int r : {6, 4, 3})
    if (heads % (r * (64 / L)) == 0) return r;
  return 0;
}
template <int L, int ROWS>
KernelInfo lookup_rope_token(int R, bool backward) {
  return R == 6   ? info_rope_token<L, 6, ROWS>(backward)
         : R == 4 ? info_rope_token<L, 4, ROWS>(backward)
                  : info_rope_token<L, 3, ROWS>(backward);
}
inline KernelInfo lookup_rope(bool narrow, bool backward, int idx, int rows, int64_t heads) {
  if (const int r = narrow ? rope_token_R(kNarrowL[idx], heads) : 0) {
    if (kNarrowL[idx] == 16) TT_LINES(lookup_rope_token, (r, backward), 16)
    TT_LINES(lookup_rope_token, (r, backward), 8)
  }
  if (narrow) {
    switch (idx) {
#define X(i, L)                                         \
  case i:                                               \
    if (backward) TT_LINES(info_bwd_rope_narrow, (), L) \
    TT_LINES(info_fwd_rope_narrow, (), L)
      TT_NARROW_LIST(X)
#undef X
    }
    return {nullptr, 0, 0, 0};
  }
  switch (idx) {
#define X(i, W, P)                                       \
  case i:                                                \
    if (backward) TT_LINES(info_bwd_rope_wide, (), W, P) \
    TT_LINES(info_fwd_rope_wide, (), W, P)
    TT_WIDE_LIST(X)
#undef X
  }
  return {nullptr, 0, 0, 0};
}

template <int MODE, int W, int P, int ROWS>
KernelInfo info_gate_wide() {
  constexpr int R = bwd_wide_R(W, P), Q = ragged_gate_Q(W, P, ROWS);
  return {reinterpret_cast<const void*>(&gate_wide<MODE, W, P, R, Q, kernel_rows(W, P, ROWS, false)>), 64 * W * Q, Q * R, P * R};
}
template <int MODE, int L, int ROWS>
KernelInfo info_gate_narrow() {
  constexpr int R = kNarrowR, NW = kNarrowNW;
  return {reinterpret_cast<const void*>(&gate_narrow<MODE, L, R, NW, ROWS>), 64 * NW, NW * R * (64 / L), R};
}
template <int MODE>
KernelInfo lookup_gate(bool narrow, int idx, int rows) {
  if (narrow) {
    switch (idx) {
#define X(i, L) case i: TT_LINES(info_gate_narrow, (), MODE, L)
      TT_NARROW_LIST(X)
#undef X
    }
  } else {
    switch (idx) {
#define X(i, W, P) case i: TT_ROWS(info_gate_wide, MODE, W, P)
      TT_WIDE_LIST(X)
#undef X
    }
  }
  return {nullptr, 0, 0, 0};
}

// Residual update fused with the following LayerNorm (wide rows only): forward streams two
// inputs, backward three (four with a gate).
// Row groups per workgroup for the kernels with two to four streamed inputs, from sweeps on
// MI355X: about ten waves where a lane holds one pack per tensor; with two packs per lane as many
// row groups as fit in eight waves, which leaves the backward kernels their 170-235 VGPRs
// (ten waves cap them at 168 and they spill).  Measured (forward / backward / gated backward, us):
// 1536 columns 281 / 271 / 418 with 9 waves against 302 / 287 / 459 with 3; 2048: 207 / 203 / 326
// with 12 waves against 221 / 212 / 362 with 4; 3072 x 118800 rows: 492 / 477 / 746 with 6 waves;
// 4096 x 90000: 502 / 478 / 763 with 8 waves against 522 / 523 / 888 with 4; 5120: 519 / 525 / 786
// with 5 waves against 533 / 595 / 2437 with 10.
constexpr int res_waves_Q(int W, int P) {
  const int q = P == 1 ? (10 + W / 2) / W : 8 / W;
  return q < 1 ? 1 : q;
}
constexpr int res_fwd_Q(int W, int P) {
  return res_waves_Q(W, P);
}
constexpr int res_bwd_Q(int W, int P, bool gated) {
  return res_waves_Q(W, P);
}
constexpr int ragged_res_fwd_Q(int W, int P, int rows, bool gated) {   // see ragged_fwd_Q
  if (row_mode(rows) != kRagged || P != 1 || (rows & kCached)) return res_fwd_Q(W, P);
  if (!gated) return W == 4 && !(rows & kUneven) ? 4 : res_fwd_Q(W, P);
  return W == 4 ? 4 : W == 3 ? 5 : res_fwd_Q(W, P);
}
template <bool GATED, int W, int P, int ROWS>
KernelInfo info_res_fwd() {
  constexpr int R = 1, Q = ragged_res_fwd_Q(W, P, ROWS, GATED);
  return {reinterpret_cast<const void*>(&resnorm_fwd_wide<W, P, R, Q, GATED ? row_mode(ROWS) : kernel_rows(W, P, ROWS, short_rows(W, P)), GATED>), 64 * W * Q, Q * R, P * R};
}
template <bool GATED, int W, int P, int ROWS>
KernelInfo info_res_bwd() {
  constexpr int R = 1, Q = res_bwd_Q(W, P, GATED);
  return {reinterpret_cast<const void*>(&resnorm_bwd_wide<W, P, R, Q, GATED ? row_mode(ROWS) : kernel_rows(W, P, ROWS, short_rows(W, P)), GATED>), 64 * W * Q, Q * R, P * R};
}
template <bool GATED>
KernelInfo lookup_res(bool backward, int idx, int rows) {
  switch (idx) {
#define X(i, W, P)                                          \
  case i:                                                   \
    if (backward) { TT_ROWS(info_res_bwd, GATED, W, P) }    \
    TT_ROWS(info_res_fwd, GATED, W, P)
    TT_WIDE_LIST(X)
#undef X
  }
  return {nullptr, 0, 0, 0};
}

template <int KIND>
KernelInfo lookup_bwd_saved(bool narrow, int idx, int rows) {
  if (narrow) {
    switch (idx) {
#define X(i, L) case i: TT_LINES(info_bwd_saved_narrow, (), KIND, L)
      TT_NARROW_LIST(X)
#undef X
    }
  } else {
    switch (idx) {
#define X(i, W, P) case i: TT_LINES(info_bwd_saved_wide, (), KIND, W, P)
      TT_WIDE_LIST(X)
#undef X
    }
  }
  return {nullptr, 0, 0, 0};
}

// Defined one per translation unit (adaln_fwd.hip, adaln_fwd_xnorm.hip, adaln_bwd.hip, adaln_bwd_saved.hip, rms_fwd.hip, rms_bwd.hip, rms_bwd_saved.hip, rms_rope.hip, gate.hip,
// resnorm_plain.hip, resnorm_gated.hip).
KernelInfo adaln_fwd_kernel(bool narrow, int idx, int rows);
KernelInfo adaln_fwd_xnorm_kernel(bool narrow, int idx, int rows);
KernelInfo adaln_bwd_kernel(bool narrow, int idx, int rows);
KernelInfo rms_fwd_kernel(bool narrow, int idx, int rows);
KernelInfo rms_bwd_kernel(bool narrow, int idx, int rows);
KernelInfo adaln_bwd_saved_kernel(bool narrow, int idx, int rows);
KernelInfo rms_bwd_saved_kernel(bool narrow, int idx, int rows);
KernelInfo rms_rope_kernel(bool narrow, bool backward, int idx, int rows, int64_t heads);
KernelInfo gate_fwd_kernel(bool narrow, int idx, int rows);
KernelInfo gate_bwd_kernel(bool narrow, int idx, int rows);
KernelInfo resnorm_plain_kernel(bool backward, int idx, int rows);
KernelInfo resnorm_gated_kernel(bool backward, int idx, int rows);

}  // namespace tt

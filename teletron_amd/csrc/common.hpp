// Shared device helpers for the gfx950 fused-normalisation kernels:
// 128-bit bf16 pack load/store, bf16<->fp32 conversion, wave64 DPP reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tt {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;   // CDNA wavefront width
constexpr int kPack = 8;    // bf16 elements per 128-bit pack

// ---------------------------------------------------------------- memory
// A kernel touches each value of a streaming tensor once, so tensors beyond the caches bypass their retention: "nt" global
// loads, and stores with system scope on top ("sc0 sc1 nt": written through instead of being
// kept in L2), which measured 1-2 % faster than plain "nt" stores under the 2-reads-1-write mix
// of the backward kernels.  The compiler's builtin only offers "nt", hence the asm for stores;
// it is an ordinary vector store.  Parameters use ordinary cached loads.
// KEEP: ordinary loads, see kKeep.
template <bool KEEP = false>
__device__ __forceinline__ u32x4 load_stream(const void* base, size_t elem_off) {
  const u32x4* p = reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(base) + elem_off);
  if constexpr (KEEP) return *p;
  else return __builtin_nontemporal_load(p);
}
__device__ __forceinline__ void store_stream(void* base, size_t elem_off, u32x4 v) {
  u32x4* p = reinterpret_cast<u32x4*>(static_cast<uint16_t*>(base) + elem_off);
  // The compiler pads its own stores wider than 64 bits against two hazards of this target but
  // cannot see inside the asm, so the padding is spelled out: two wait states between a VALU
  // write of the data registers and the store, and two between the store and the next VALU
  // write of those registers (the data is read after issue).  Four are spent on each side.
  asm volatile("s_nop 3\n\tglobal_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 3" ::"v"(p), "v"(v) : "memory");
}
// Two stores of one lane to the same element offset of two tensors (an output and a second
// saved copy): one asm block, so the pair pays the hazard padding once.
__device__ __forceinline__ void store_stream2(void* base0, void* base1, size_t elem_off, u32x4 v0, u32x4 v1) {
  u32x4* p0 = reinterpret_cast<u32x4*>(static_cast<uint16_t*>(base0) + elem_off);
  u32x4* p1 = reinterpret_cast<u32x4*>(static_cast<uint16_t*>(base1) + elem_off);
  asm volatile("s_nop 3\n\tglobal_store_dwordx4 %0, %2, off sc0 sc1 nt\n\t"
               "global_store_dwordx4 %1, %3, off sc0 sc1 nt\n\ts_nop 3" ::"v"(p0), "v"(p1), "v"(v0), "v"(v1) : "memory");
}
// Values that the next kernel reads, perhaps on another XCD: written through to where all XCDs see them
// (device scope), but cached there.
__device__ __forceinline__ void store_agent(float* p, f32x4 v) {
  asm volatile("s_nop 3\n\tglobal_store_dwordx4 %0, %1, off sc1\n\ts_nop 3" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ u32x4 load_cached(const void* base, size_t elem_off) {
  return *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(base) + elem_off);
}

// How the rows of a wide kernel lie on its lane slots and in memory.
enum Rows : int {
  kMasked = 0,   // fewer packs than lane slots; a row is a whole number of 128-byte lines (x_norm forward: any)
  kFull = 1,     // every lane slot holds a pack
  kRagged = 2,   // as kMasked, but rows start anywhere inside a line (cols % 64 != 0)
  kOdd = 3,      // any row length and 2-byte aligned tensors; the last pack may be short
  // Added to the others (and to kFull / kMasked of the narrow kernels): the activations are read with ordinary loads,
  // so that tensors which fit the caches stay there for the next kernel that reads them.
  kKeep = 4,
  // Added to kRagged, for the row groups a workgroup (ragged_fwd_Q and the rules after it): the tensor fits the caches;
  // over a quarter, or at most a sixteenth, of the lane slots hold no pack; it is beyond the caches, and one workgroup
  // a CU is not to be had in whole workgroups a batch.
  kCached = 8,
  kIdle = 16,
  kDense = 32,
  kUneven = 64,
};
constexpr int row_mode(int rows) { return rows & 3; }
constexpr bool keeps(int rows) { return (rows & kKeep) != 0; }
// Where rows are not whole lines, the segments of neighbouring waves and rows share the lines at
// their ends.  A written-through store sends its part of such a line to memory on its own, and
// memory turns a part of a 64-byte sector into a read and a write; those lines have to meet in
// the L2 first.  Two ways (SHORT of the kernels):
//   short rows (at most 6 segments of 64 packs, norm and ungated residual + norm kernels): every
//     store is a plain "nt" store that the L2 writes back, and the loads, which share lines in the
//     same way, are cached ones.
//   otherwise: only the lanes whose line is shared do that, the others write through (written back
//     whole, the backward kernels lose 20 %: 80000 x 4416, 352 -> 419 us); nt loads.
// us forward / backward of 60000 rows, everything written through | all written back | shared lines only:
//   AdaLN 1000 columns 52 / 79 | 45 / 62 | 44 / 71;  2200: 154 / 198 | 98 / 162 | 117 / 184
//         3688: 185 / 290 | 162 / 233 | 139 / 226;  4424: 264 / 337 | 181 / 334 | 185 / 263
//   RMS   1544: 88 / 151 | 66 / 103 | 64 / 102;  2200: 139 / 226 | 97 / 147 | 97 / 155;  4600: 257 / 349 | 191 / 299 | 185 / 277
//   gate  1000: 73 / 75 | 66 / 58 | 61 / 64;  3000: 246 / 247 | 188 / 192 | 179 / 182
//   residual + norm 1544: 179 / 187 | 133 / 137 | 128 / 142;  gated: 179 / 232 | 134 / 207 | 129 / 192
constexpr bool short_rows(int W, int P) { return W * P <= 6; }
// The instantiation that stands for `rows`: kKeep goes where the loads are ordinary ones anyway, and above 6144 columns.
constexpr int kernel_rows(int W, int P, int rows, bool is_short) {
  return W * P > 12 || (row_mode(rows) == kRagged && is_short) || row_mode(rows) == kOdd ? row_mode(rows)
                                                                                          : row_mode(rows) | (rows & kKeep);
}

template <int ROWS, bool SHORT, bool KEEP>
__device__ __forceinline__ u32x4 load_row(const void* base, size_t elem_off) {
  if constexpr (ROWS == kRagged && SHORT) return load_cached(base, elem_off);
  else return load_stream<KEEP>(base, elem_off);
}
// Element offset of a lane's pack, from the column that its loads use (no further register) or from its slot.
// The kernels of 16 waves a row have 128 registers a lane and spill: with every slot in use they are
// the faster with the latter (32768 columns, AdaLN forward 133 -> 116, gate backward 338 -> 245 us; 16384,
// AdaLN backward 648 -> 571), where the others lose up to 16 % (ungated residual + norm backward,
// 8192 x 1536 24.5 -> 29.3: fewer registers let a second workgroup onto the CU, whose partial sums cost more
// than it gives).
template <int ROWS, int W>
__device__ __forceinline__ size_t pack_offset(int64_t row, int C, int col, int packs, int slot) {
  if constexpr (ROWS == kFull && W >= 16) return (size_t)(row * packs + slot) * kPack;
  else return (size_t)(row * C + col);
}
// Stores a lane's pack (act: the row has it); `left`: packs of the row from the wave's segment of 64 on.
template <int ROWS, bool SHORT>
__device__ __forceinline__ void store_row(void* base, size_t elem_off, bool act, int left, int lane, u32x4 v) {
  if (!act) return;
  if constexpr (ROWS == kRagged) {
    u32x4* p = reinterpret_cast<u32x4*>(static_cast<uint16_t*>(base) + elem_off);
    bool shared = true;
    if constexpr (!SHORT) {
      // position of the pack inside its 128-byte line, and whether the segment holds that whole line
      const int at = (static_cast<int>(reinterpret_cast<uintptr_t>(p) >> 4)) & 7;
      const int last = left < 64 ? left - 1 : 63;
      shared = lane < at || lane + 7 - at > last;
    }
    if (shared) {
      if constexpr (SHORT) __builtin_nontemporal_store(v, p);
      else *p = v;
      return;
    }
  }
  store_stream(base, elem_off, v);
}

// ---- kOdd rows: packs at any 2-byte address (this target's vector memory instructions take them)
typedef u32x4 u32x4_any __attribute__((aligned(2)));
__device__ __forceinline__ u32x4 load_any(const void* base, size_t elem_off) {
  return *reinterpret_cast<const u32x4_any*>(static_cast<const uint16_t*>(base) + elem_off);
}
// Stores the first n values of a pack (n <= 0: none).
__device__ __forceinline__ void store_any(void* base, size_t elem_off, u32x4 v, int n) {
  uint16_t* p = static_cast<uint16_t*>(base) + elem_off;
  if (n >= kPack) {
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4_any*>(p));
  } else {
#pragma unroll
    for (int j = 0; j < kPack - 1; ++j)
      if (j < n) p[j] = static_cast<uint16_t>(v[j / 2] >> (16 * (j & 1)));
  }
}
// A short last pack is loaded as the last eight values of its row, which is always inside the
// tensor; this moves its own values to the front and zeros in behind them.
__device__ __forceinline__ u32x4 drop_values(u32x4 v, int drop) {
  if (drop & 1) v = u32x4{v[0] >> 16 | v[1] << 16, v[1] >> 16 | v[2] << 16, v[2] >> 16 | v[3] << 16, v[3] >> 16};
  if (drop & 2) v = u32x4{v[1], v[2], v[3], 0};
  if (drop & 4) v = u32x4{v[2], v[3], 0, 0};
  return v;
}

// ---------------------------------------------------------------- bf16 <-> fp32
__device__ __forceinline__ void unpack8(u32x4 raw, float (&f)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f[2 * j]     = __builtin_bit_cast(float, raw[j] << 16);
    f[2 * j + 1] = __builtin_bit_cast(float, raw[j] & 0xffff0000u);
  }
}
// Round-to-nearest-even fp32 -> bf16, two at a time (v_cvt_pk_bf16_f32 on gfx950).
__device__ __forceinline__ unsigned pack2(float lo, float hi) {
  f32x2 v = {lo, hi};
  bf16x2 r = __builtin_convertvector(v, bf16x2);
  return __builtin_bit_cast(unsigned, r);
}
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
  u32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = pack2(f[2 * j], f[2 * j + 1]);
  return o;
}
__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __builtin_bit_cast(float, static_cast<unsigned>(h) << 16);
}
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  return static_cast<uint16_t>(pack2(f, 0.f) & 0xffffu);
}

// ---------------------------------------------------------------- wave64 reductions
// DPP controls: quad_perm[1,0,3,2]=0xB1, quad_perm[2,3,0,1]=0x4E,
// row_half_mirror=0x141, row_mirror=0x140.  Each step adds a lane's partner, so
// after k steps every lane of an aligned 2^k group holds that group's sum.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  int t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false);
  return v + __builtin_bit_cast(float, t);
}
__device__ __forceinline__ float readlane(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Sum over aligned groups of L lanes (L in 1,2,4,8,16,32,64); every lane of a
// group receives the group's total.  The summation order is fixed, so results
// are bitwise reproducible.
template <int L>
__device__ __forceinline__ float group_allsum(float v) {
  if constexpr (L >= 2) v = dpp_add<0xB1>(v);
  if constexpr (L >= 4) v = dpp_add<0x4E>(v);
  if constexpr (L >= 8) v = dpp_add<0x141>(v);
  if constexpr (L >= 16) v = dpp_add<0x140>(v);
  if constexpr (L == 32) {
    // partner row inside the 32-lane half: lane ^ 16
    int t = __builtin_amdgcn_ds_bpermute(((int)(threadIdx.x & 63) ^ 16) << 2, __builtin_bit_cast(int, v));
    v += __builtin_bit_cast(float, t);
  }
  if constexpr (L == 64) {
    float a = readlane(v, 0), b = readlane(v, 16), c = readlane(v, 32), d = readlane(v, 48);
    v = (a + b) + (c + d);
  }
  return v;
}
__device__ __forceinline__ float wave_allsum(float v) { return group_allsum<64>(v); }

}  // namespace tt

// Slab unpack kernels for gfx950: SquareQ INT8→bf16 dequant and fp32→bf16
// cast, scattering a packed device-resident source slab into a block's
// contiguous parameter buffer. Device code only: built into a code object that
// the library embeds and loads with the module API (sh_kernels.cpp); the plans
// and launches are host code in sh_unpack.cpp.
//
// Replaces the host-side staging arithmetic of the reference:
//   SquareQ dequant   src/stagehand/scheduler.py:290-300
//   bias / param cast src/stagehand/scheduler.py:181, 224-230, 302-306, 1066-1071
//   zero-fill         src/stagehand/scheduler.py:240, 276-297, 325
//
// Work decomposition. Every descriptor covers rows*cols elements, cut into
// tiles of kThreads * unroll * chunk elements; a host-built tile map gives
// each workgroup its descriptor in O(1) (one scalar load), and the descriptor
// itself is a 64-byte scalar load, so all per-region state lives in SGPRs.
// Each thread moves `unroll` chunks; all loads of a thread are issued before
// the first conversion. Loads and stores are up to 128-bit (an int8 chunk is
// one 128-bit store: 8 values to bf16 from a 64-bit load, 4 to fp32 from a
// 32-bit load; the cast reads 128 and writes 64 bits); the hardware's
// unaligned-access mode lets them start at any byte offset, which the reference
// layout needs (it has no padding, so int8 regions start at arbitrary offsets).
// A chunk inside one row needs one row scale; a chunk across two rows takes a
// second one and, from a padded source, a second load. Only rows shorter than a
// chunk and chunks cut by a region's ends go element by element. This is pure
// streaming: no LDS (the scale is one load per chunk) and no MFMA.
//
// Numerics. The dequant is computed exactly as the reference's torch CPU ops:
// f32(q) exactly, then an IEEE fp32 subtract of the zero point (skipped when
// no zero points are given: q - 0.0f == q bit for bit), then an IEEE fp32
// multiply by the row scale, each rounded to nearest even; fp32 denormals are
// kept (no flush flags). Contraction is disabled so nothing becomes an FMA.
// fp32→bf16 is round-to-nearest-even on the bit pattern,
//   bf16 = (u + 0x7FFF + ((u >> 16) & 1)) >> 16,
// which equals torch's CPU conversion for every non-NaN input; every NaN
// becomes 0xFFFF, as torch's CPU conversion does.

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

#include "sh_internal.h"
#include "sh_unpack_shape.h"
#include "stagehand_native.h"

#pragma clang fp contract(off)

namespace {

// NB bytes as 32-bit words; loaded and stored with unaligned-capable 128-bit
// (or 64-bit) vector memory operations.
template <uint32_t NB>
struct Words {
  uint32_t w[NB / 4];
};

template <uint32_t NB>
__device__ __forceinline__ Words<NB> ldw(const uint8_t* p) {
  Words<NB> v;
  __builtin_memcpy(&v, p, NB);
  return v;
}

template <uint32_t NB>
__device__ __forceinline__ void stw(uint8_t* p, const Words<NB>& v) {
  __builtin_memcpy(p, &v, NB);
}

// Non-temporal forms (the `nt` bit on the load / store): 8 or 16 bytes, any byte alignment.
typedef uint32_t u32x2_a1 __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32x4_a1 __attribute__((ext_vector_type(4), aligned(1)));

template <uint32_t NB>
__device__ __forceinline__ Words<NB> ldw_nt(const uint8_t* p) {
  static_assert(NB == 8 || NB == 16, "8- or 16-byte non-temporal loads");
  Words<NB> v;
  if constexpr (NB == 8) {
    const u32x2_a1 x = __builtin_nontemporal_load(reinterpret_cast<const u32x2_a1*>(p));
    v.w[0] = x.x;
    v.w[1] = x.y;
  } else {
    const u32x4_a1 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4_a1*>(p));
    v.w[0] = x.x;
    v.w[1] = x.y;
    v.w[2] = x.z;
    v.w[3] = x.w;
  }
  return v;
}

template <uint32_t NB>
__device__ __forceinline__ void stw_nt(uint8_t* p, const Words<NB>& v) {
  static_assert(NB == 8 || NB == 16, "8- or 16-byte non-temporal stores");
  if constexpr (NB == 8) {
    u32x2_a1 x;
    x.x = v.w[0];
    x.y = v.w[1];
    __builtin_nontemporal_store(x, reinterpret_cast<u32x2_a1*>(p));
  } else {
    u32x4_a1 x;
    x.x = v.w[0];
    x.y = v.w[1];
    x.z = v.w[2];
    x.w = v.w[3];
    __builtin_nontemporal_store(x, reinterpret_cast<u32x4_a1*>(p));
  }
}

// Rounded bf16 in bits 31..16 (low half is garbage): u + 0x7FFF + lsb.
__device__ __forceinline__ uint32_t rne_hi(float x) {
  const uint32_t u = __float_as_uint(x);
  return u + 0x7FFFu + ((u >> 16) & 1u);
}

__device__ __forceinline__ uint32_t rne_hi_nan(float x) {
  return (x != x) ? 0xFFFFFFFFu : rne_hi(x);
}

// Packs the upper halves of two rne_hi words: lo element in bits 15..0.
__device__ __forceinline__ uint32_t pack_hi(uint32_t lo, uint32_t hi) {
  return __builtin_amdgcn_perm(hi, lo, 0x07060302u);
}

__device__ __forceinline__ uint16_t bf16_bits(float x) { return (uint16_t)(rne_hi_nan(x) >> 16); }

__device__ __forceinline__ float i8_at(uint32_t word, uint32_t byte) {
  return (float)(int32_t)(int8_t)(uint8_t)(word >> (8 * byte));
}

template <bool HAS_ZP>
__device__ __forceinline__ float dq(float q, float s, float z) {
  if (HAS_ZP) q = q - z;
  return q * s;
}

// ── INT8 row-scale dequant ────────────────────────────────────────────────

// One chunk of C int8 values of a single row with a finite scale and zero point (they cannot turn
// a finite q into NaN) → C outputs.
template <uint32_t C, bool OUT_BF16, bool HAS_ZP>
__device__ __forceinline__ Words<C * (OUT_BF16 ? 2 : 4)> dq_chunk(const Words<C>& q, float s, float z) {
  Words<C * (OUT_BF16 ? 2 : 4)> o;
  if constexpr (OUT_BF16) {
#pragma unroll
    for (uint32_t w = 0; w < C / 2; ++w) {
      const uint32_t word = q.w[w / 2];
      o.w[w] = pack_hi(rne_hi(dq<HAS_ZP>(i8_at(word, (2 * w) % 4), s, z)),
                       rne_hi(dq<HAS_ZP>(i8_at(word, (2 * w + 1) % 4), s, z)));
    }
  } else {
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) o.w[j] = __float_as_uint(dq<HAS_ZP>(i8_at(q.w[j / 4], j % 4), s, z));
  }
  return o;
}

template <bool OUT_BF16>
__device__ __forceinline__ void store_elem(uint8_t* o, uint32_t idx, float v) {
  if constexpr (OUT_BF16) {
    const uint16_t b = bf16_bits(v);
    __builtin_memcpy(o + 2 * (size_t)idx, &b, 2);
  } else {
    __builtin_memcpy(o + 4 * (size_t)idx, &v, 4);
  }
}

// Chunk [e, e + C) of a region, element by element: a chunk cut by the region's start (e wrapped
// below 0, so its first elements are above every numel) or end.
template <uint32_t C, bool OUT_BF16, bool HAS_ZP>
__device__ __forceinline__ void dq_edge(const sh_unpack_desc& d, uint32_t e, uint32_t numel, uint32_t pad,
                                        const uint8_t* s, const float* sc, const float* zp, uint8_t* o) {
#pragma unroll 1
  for (uint32_t j = 0; j < C; ++j) {
    const uint32_t i = e + j;
    if (i >= numel) continue;
    const uint32_t r = sh::udiv(i, d.div_magic);
    const float q = (float)(int32_t)(int8_t)s[i + (uint64_t)r * pad];
    store_elem<OUT_BF16>(o, i, dq<HAS_ZP>(q, sc[r], HAS_ZP ? zp[r] : 0.0f));
  }
}

// C outputs from the bytes of q, each with its own scale and zero point.
template <uint32_t C, bool OUT_BF16, bool HAS_ZP>
__device__ __forceinline__ void dq_each_store(const Words<C>& q, const float (&sv)[C], const float (&zv)[C],
                                              uint8_t* out) {
  if constexpr (OUT_BF16) {
    Words<2 * C> ow;
#pragma unroll
    for (uint32_t w = 0; w < C / 2; ++w) {
      const float lo = dq<HAS_ZP>(i8_at(q.w[w / 2], (2 * w) % 4), sv[2 * w], zv[2 * w]);
      const float hi = dq<HAS_ZP>(i8_at(q.w[w / 2], (2 * w + 1) % 4), sv[2 * w + 1], zv[2 * w + 1]);
      ow.w[w] = pack_hi(rne_hi_nan(lo), rne_hi_nan(hi));
    }
    stw_nt<2 * C>(out, ow);
  } else {
    Words<4 * C> ow;
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) ow.w[j] = __float_as_uint(dq<HAS_ZP>(i8_at(q.w[j / 4], j % 4), sv[j], zv[j]));
    stw_nt<4 * C>(out, ow);
  }
}

// Whether the chunk of C elements at e lies inside the region. e wraps below 0 where a lead precedes
// element 0: to an index >= 2^32 - 4096, above every numel.
template <uint32_t C>
__device__ __forceinline__ bool whole_chunk(uint32_t e, uint32_t numel) {
  return e < numel && numel - e >= C;
}

// s_waitcnt operand: every vector memory operation done, no wait for the other counters.
constexpr int kWaitVmcnt0 = 0x0F70;

// Rows of at least a chunk, of any length and stride: a chunk lies in one row, or in the last `left`
// elements of one row and the first C - left of the next. Narrow unpadded rows whose chunks cross
// often take i8_narrow_rows instead.
//
// All chunks of a thread go through straight-line code as if each lay in one row with a finite
// scale: the loads first, then the conversions and the stores. Only then are the exceptions seen
// to, which few wavefronts have: a chunk across two rows, or under a scale or zero point that can
// make NaNs, is written once more (one wavefront's stores to one address land in program order),
// and a chunk cut by the region's start or end is written element by element. A lane without a
// whole chunk loads the region's first one, so that no load needs a branch; with the loads in
// branches of their own, the compiler put waits between them for registers that other paths of the
// kernel might have had in flight (the mixed kernel then took 172 us for a double-stream block of
// the 12B model, and 159 after an unrelated change).
//
// A chunk across rows takes the second row's bytes from the same load, or in a padded source from
// a load `pad` bytes later, whose bytes from `left` on are the next row's. Every load stays inside
// the region: the second row exists, as the whole chunk lies below numel.
//
// HBM bounds this. Measured (MI355X; before, rows that were not back to back or not whole chunks
// went element by element): a padded single-stream block of the 12B model with zero points 263 ->
// 68 us (6.2 TB/s); 2999-wide rows 75 -> 65 us (6.2 TB/s) and a slab of 128 such tensors 1376 ->
// 974 (1064 with its tiles off destination boundaries); the aligned double-stream block 159 -> 155
// us (6.6 TB/s) and slab of 128 tensors 1010 -> 993 (6.7 TB/s; 999 before its ragged regions took the
// first tiles).
//
// Once a thread has all its loads, its stores go out back to back, except (PACED) for aligned rows in
// the kernel that holds no other kind and in the one for long tables of sh_unpack_noalloc: there each
// store waits for the one before it. Measured, not paced against paced: double-stream block (mixed
// kernel) 154.9 against 157.5 us, padded block 68.1 against 70.3; but slab of 128 aligned tensors 1030-1060
// against 998-1007 us (6.6 GB, and 3% from 3 GB on; up to 2 GB the same), and a mixed table in the scratch
// array of 74K tiles 300.8 against 296.3, of 166K 660.9 against 631.2. Pacing holds back writes in a stream
// that is two thirds writes; why only these gain from it is not known.
template <bool OUT_BF16, bool HAS_ZP, bool PACED, uint32_t C, uint32_t U>
__device__ __forceinline__ void i8_rows(const sh_unpack_desc& d, uint32_t e0, uint32_t numel, uint32_t pad,
                                        const uint8_t* __restrict__ s, const float* __restrict__ sc,
                                        const float* __restrict__ zp, uint8_t* __restrict__ o) {
  constexpr uint32_t kOutBytes = OUT_BF16 ? 2 : 4;
  Words<C> q[U];
  float sv[U], zv[U];
  uint32_t row[U];
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    const uint32_t i = whole_chunk<C>(e, numel) ? e : 0u;
    row[k] = sh::udiv(i, d.div_magic);
    q[k] = ldw<C>(s + i + (uint64_t)row[k] * pad);
  }
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    sv[k] = sc[row[k]];
    zv[k] = HAS_ZP ? zp[row[k]] : 0.0f;
  }
  if (PACED && pad == 0 && (d.cols % C) == 0 && (d.lead % C) == 0) {
#pragma unroll
    for (uint32_t k = 0; k < U; ++k) {
      const uint32_t e = e0 + k * (kThreads * C);
      const auto out = dq_chunk<C, OUT_BF16, HAS_ZP>(q[k], sv[k], zv[k]);
      if (whole_chunk<C>(e, numel)) stw_nt<C * kOutBytes>(o + (size_t)e * kOutBytes, out);
      if (k + 1 < U) __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    }
  } else {
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
#pragma unroll
    for (uint32_t k = 0; k < U; ++k) {
      const uint32_t e = e0 + k * (kThreads * C);
      const auto out = dq_chunk<C, OUT_BF16, HAS_ZP>(q[k], sv[k], zv[k]);
      if (whole_chunk<C>(e, numel)) stw_nt<C * kOutBytes>(o + (size_t)e * kOutBytes, out);
    }
    asm volatile("; not paced");  // keeps this tail apart from the other's, which waits in between
  }
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    if (!whole_chunk<C>(e, numel)) {
      dq_edge<C, OUT_BF16, HAS_ZP>(d, e, numel, pad, s, sc, zp, o);
      continue;
    }
    const uint32_t left = (row[k] + 1) * d.cols - e;  // modulo 2^32; the difference fits
    const bool finite = !OUT_BF16 || (__builtin_isfinite(sv[k]) && (!HAS_ZP || __builtin_isfinite(zv[k])));
    if (left >= C && finite) continue;
    float s1 = sv[k], z1 = zv[k];
    Words<C> qq = q[k];
    if (left < C) {
      s1 = sc[row[k] + 1];
      z1 = HAS_ZP ? zp[row[k] + 1] : 0.0f;
      if (pad != 0) {
        const Words<C> q1 = ldw<C>(s + e + (uint64_t)row[k] * pad + pad);
#pragma unroll
        for (uint32_t w = 0; w < C / 4; ++w) {
          const uint32_t own = left > 4 * w ? left - 4 * w : 0u;  // bytes of this word in the first row
          const uint32_t m = own >= 4 ? 0xFFFFFFFFu : (1u << (8 * own)) - 1u;
          qq.w[w] = (qq.w[w] & m) | (q1.w[w] & ~m);
        }
      }
    }
    float se[C], ze[C];
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) {
      se[j] = j < left ? sv[k] : s1;
      ze[j] = j < left ? zv[k] : z1;
    }
    dq_each_store<C, OUT_BF16, HAS_ZP>(qq, se, ze, o + (size_t)e * kOutBytes);
  }
}

// Unpadded rows of at least a chunk and below kNarrowRowBytes of output, where chunks cross rows: every
// chunk takes its row's scale and the next one's (its own again where it ends inside the row) and is
// written once. In such rows most wavefronts have a chunk across rows, and i8_rows' second pass over
// them costs more than the second scale and the choice per element. As there, the loads go first,
// without a branch, and the stores back to back once all of them are there.
//
// Measured (MI355X, one region; in brackets i8_rows, and the path before both, which tracked the row
// element by element): 64 M elements to bf16, 9-wide rows 34.7 us [75, 34.6], 77 31.1 [47, 31.0], 255 30.7
// [35.4, 30.6]; 1 G elements, 77 519 [934, 569], 513 510 [604, 560], 1023 509 [550, 559]; to fp32, 1 G elements, 9 995
// [2163, 1352], 255 893 [904, 1340].
template <bool OUT_BF16, bool HAS_ZP, uint32_t C, uint32_t U>
__device__ __forceinline__ void i8_narrow_rows(const sh_unpack_desc& d, uint32_t e0, uint32_t numel,
                                               const uint8_t* __restrict__ s, const float* __restrict__ sc,
                                               const float* __restrict__ zp, uint8_t* __restrict__ o) {
  Words<C> q[U];
  uint32_t row[U], left[U];
  float s0[U], s1[U], z0[U], z1[U];
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    const uint32_t i = whole_chunk<C>(e, numel) ? e : 0u;
    row[k] = sh::udiv(i, d.div_magic);
    left[k] = (row[k] + 1) * d.cols - i;  // modulo 2^32; the difference fits
    q[k] = ldw<C>(s + i);
  }
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t next = left[k] < C ? row[k] + 1 : row[k];  // exists: the chunk lies below numel
    s0[k] = sc[row[k]];
    s1[k] = sc[next];
    z0[k] = HAS_ZP ? zp[row[k]] : 0.0f;
    z1[k] = HAS_ZP ? zp[next] : 0.0f;
  }
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    if (whole_chunk<C>(e, numel)) {
      float se[C], ze[C];
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        se[j] = j < left[k] ? s0[k] : s1[k];
        ze[j] = j < left[k] ? z0[k] : z1[k];
      }
      dq_each_store<C, OUT_BF16, HAS_ZP>(q[k], se, ze, o + (size_t)e * (OUT_BF16 ? 2 : 4));
    } else {
      dq_edge<C, OUT_BF16, HAS_ZP>(d, e, numel, 0, s, sc, zp, o);
    }
  }
}

// Rows shorter than a chunk: the row is tracked element by element inside each chunk.
template <bool OUT_BF16, bool HAS_ZP, uint32_t C, uint32_t U>
__device__ __forceinline__ void i8_short_rows(const sh_unpack_desc& d, uint32_t e0, uint32_t numel, uint32_t pad,
                                              const uint8_t* __restrict__ s, const float* __restrict__ sc,
                                              const float* __restrict__ zp, uint8_t* __restrict__ o) {
#pragma unroll 1
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    if (whole_chunk<C>(e, numel)) {
      uint32_t r = sh::udiv(e, d.div_magic);
      uint32_t c = e - r * d.cols;
      Words<C> q{};
      if (pad == 0) {
        q = ldw<C>(s + e);
      } else {
        uint32_t rq = r, cq = c;
#pragma unroll
        for (uint32_t j = 0; j < C; ++j) {
          q.w[j / 4] |= (uint32_t)s[e + j + (uint64_t)rq * pad] << (8 * (j % 4));
          if (++cq == d.cols) {
            cq = 0;
            ++rq;
          }
        }
      }
      float se[C], ze[C];
#pragma unroll
      for (uint32_t j = 0; j < C; ++j) {
        se[j] = sc[r];
        ze[j] = HAS_ZP ? zp[r] : 0.0f;
        if (++c == d.cols) {
          c = 0;
          ++r;
        }
      }
      dq_each_store<C, OUT_BF16, HAS_ZP>(q, se, ze, o + (size_t)e * (OUT_BF16 ? 2 : 4));
    } else {
      dq_edge<C, OUT_BF16, HAS_ZP>(d, e, numel, pad, s, sc, zp, o);
    }
  }
}

// Output rows below this size take i8_narrow_rows where chunks cross rows. Above, fewer chunks cross, and
// i8_rows is as fast or faster: rows of 1155 bf16 (64 M elements) 30.8 us against 30.4, (1 G) 518 and 509,
// 3001 493 and 509, a slab of 128 tensors of 2999 to 11996 elements a row 966 and 1009; fp32, 700 822 and 833, a
// double-stream block of hidden 3001 272 and 285.
constexpr uint32_t kNarrowRowBytes = 2048;

template <bool OUT_BF16, bool HAS_ZP, bool PACED>
__device__ __forceinline__ void tile_i8(const sh_unpack_desc& d, uint32_t local,
                                        const uint8_t* __restrict__ src,
                                        const float* __restrict__ scales,
                                        const float* __restrict__ zps, uint8_t* __restrict__ dst) {
  // A chunk is one 16-byte store, 8 bf16 or 4 fp32 outputs, so a wavefront's store instruction
  // covers one contiguous 1 KiB span. With 8 fp32 per chunk each lane wrote two 16-byte halves at a
  // 32-byte stride: a float32 double-stream block (hidden 1536) 84 us, now 61 (7.0 TB/s); plain
  // instead of non-temporal fp32 stores 75 us.
  constexpr uint32_t C = OUT_BF16 ? kChunkI8 : kStepF32;
  constexpr uint32_t U = OUT_BF16 ? kUnrollI8 : kPerThreadF32 / C;
  constexpr uint32_t T = kThreads * U * C;
  const uint32_t cols = d.cols;
  const uint32_t numel = d.rows * cols;
  const uint32_t pad = d.src_ld - cols;  // src_ld is never 0 in a launch table
  const uint8_t* s = src + d.src_off;
  uint8_t* o = dst + d.dst_off;
  const float* sc = scales + d.scale_off;
  const float* zp = HAS_ZP ? zps + d.scale_off : nullptr;
  const bool crossing = ((cols | d.lead) % C) != 0;  // chunks may lie across rows
  const bool narrow = pad == 0 && crossing && cols >= C && cols < kNarrowRowBytes / (OUT_BF16 ? 2u : 4u);
  // A workgroup takes one tile, or two of an fp32 output where the table is near the launch limit.
  const uint32_t last = OUT_BF16 ? 0u : d.reserved;
  uint32_t e0 = (local << last) * T + threadIdx.x * C - d.lead;
#pragma unroll 1
  for (uint32_t sub = 0; sub <= last; ++sub, e0 += T) {
    if (narrow)
      i8_narrow_rows<OUT_BF16, HAS_ZP, C, U>(d, e0, numel, s, sc, zp, o);
    else if (cols >= C)
      i8_rows<OUT_BF16, HAS_ZP, PACED, C, U>(d, e0, numel, pad, s, sc, zp, o);
    else
      i8_short_rows<OUT_BF16, HAS_ZP, C, U>(d, e0, numel, pad, s, sc, zp, o);
  }
}

// ── fp32 → bf16 cast ──────────────────────────────────────────────────────

// Plain stores: the next kernel reads the output, and finds what the L2s still hold of it. Non-temporal
// stores make a cast of up to 400 MB 4-10% faster by itself and the pair slower (MI355X, cast and a
// matrix product that reads it, 64 rows: 2048x512 9.9 us with plain and 11.6 with nt stores, 3072x3072
// 27.2 and 32.4, 8192x2048 30.2 and 39.1, 12288x3072 56.9 and 62.0).
__device__ __forceinline__ void tile_f32_bf16(const sh_unpack_desc& d, uint32_t local,
                                              const uint8_t* __restrict__ src,
                                              uint8_t* __restrict__ dst) {
  constexpr uint32_t C = kChunkF32;
  constexpr uint32_t U = kUnrollF32;
  const uint32_t numel = d.rows * d.cols;
  const uint8_t* s = src + d.src_off;
  uint8_t* o = dst + d.dst_off;
  const uint32_t e0 = local * (kThreads * U * C) + threadIdx.x * C - d.lead;
  Words<4 * C> v[U];
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    if (whole_chunk<C>(e, numel)) v[k] = ldw_nt<4 * C>(s + (size_t)e * 4);  // read once
  }
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    if (whole_chunk<C>(e, numel)) {
      Words<2 * C> ow;
#pragma unroll
      for (uint32_t w = 0; w < C / 2; ++w)
        ow.w[w] = pack_hi(rne_hi_nan(__uint_as_float(v[k].w[2 * w])), rne_hi_nan(__uint_as_float(v[k].w[2 * w + 1])));
      stw<2 * C>(o + (size_t)e * 2, ow);
    } else {
#pragma unroll 1
      for (uint32_t j = e; j != e + C; ++j) {  // cut by the region's start or end
        if (j >= numel) continue;
        float x;
        __builtin_memcpy(&x, s + (size_t)j * 4, 4);
        const uint16_t b = bf16_bits(x);
        __builtin_memcpy(o + (size_t)j * 2, &b, 2);
      }
    }
  }
}

// ── bf16 → fp32 widen ─────────────────────────────────────────────────────

// A tile is kThreads * kPerThreadF32 elements, moved kStepF32 at a time (one 16-byte store) with
// consecutive lanes on consecutive steps, so each store instruction of a wavefront covers one
// contiguous 1 KiB span.
__device__ __forceinline__ void bf16_f32_steps(uint32_t e0, uint32_t numel, const uint8_t* __restrict__ s,
                                               uint8_t* __restrict__ o) {
  constexpr uint32_t C = kStepF32;
  constexpr uint32_t U = kPerThreadF32 / C;
  Words<2 * C> v[U];
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    if (whole_chunk<C>(e, numel)) v[k] = ldw<2 * C>(s + (size_t)e * 2);
  }
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) {
    const uint32_t e = e0 + k * (kThreads * C);
    if (whole_chunk<C>(e, numel)) {
      Words<4 * C> ow;
#pragma unroll
      for (uint32_t w = 0; w < C / 2; ++w) {
        ow.w[2 * w] = v[k].w[w] << 16;
        ow.w[2 * w + 1] = v[k].w[w] & 0xFFFF0000u;
      }
      stw_nt<4 * C>(o + (size_t)e * 4, ow);
    } else {
#pragma unroll 1
      for (uint32_t j = e; j != e + C; ++j) {  // cut by the region's start or end
        if (j >= numel) continue;
        uint16_t b;
        __builtin_memcpy(&b, s + (size_t)j * 2, 2);
        const uint32_t w = (uint32_t)b << 16;
        __builtin_memcpy(o + (size_t)j * 4, &w, 4);
      }
    }
  }
}

__device__ __forceinline__ void tile_bf16_f32(const sh_unpack_desc& d, uint32_t local,
                                              const uint8_t* __restrict__ src,
                                              uint8_t* __restrict__ dst) {
  constexpr uint32_t T = kThreads * kPerThreadF32;
  const uint32_t numel = d.rows * d.cols;
  uint32_t e0 = (local << d.reserved) * T + threadIdx.x * kStepF32 - d.lead;
#pragma unroll 1
  for (uint32_t sub = 0; sub <= d.reserved; ++sub, e0 += T)  // one tile, or two as in tile_i8
    bf16_f32_steps(e0, numel, src + d.src_off, dst + d.dst_off);
}

// ── byte copy / zero fill ─────────────────────────────────────────────────

// A tile is kThreads * C bytes, moved as 16-byte words with consecutive lanes on consecutive words
// (each load / store instruction of a wavefront covers one contiguous 1 KiB span).
template <bool ZERO>
__device__ __forceinline__ void tile_bytes(const sh_unpack_desc& d, uint32_t local,
                                           const uint8_t* __restrict__ src,
                                           uint8_t* __restrict__ dst) {
  constexpr uint32_t W = 16;
  constexpr uint32_t kWords = (ZERO ? kChunkZero : kChunkCopy) / W;
  const uint32_t nbytes = d.rows * d.cols;
  const uint8_t* s = src + d.src_off;
  uint8_t* o = dst + d.dst_off;
  const uint32_t b0 = local * (kThreads * kWords * W) + threadIdx.x * W - d.lead;
  Words<W> v[kWords];
#pragma unroll
  for (uint32_t k = 0; k < kWords; ++k) {
    const uint32_t b = b0 + k * (kThreads * W);
    if (whole_chunk<W>(b, nbytes)) {
      if (ZERO) {
#pragma unroll
        for (uint32_t w = 0; w < W / 4; ++w) v[k].w[w] = 0;
      } else {
        v[k] = ldw<W>(s + b);
      }
    }
  }
#pragma unroll
  for (uint32_t k = 0; k < kWords; ++k) {
    const uint32_t b = b0 + k * (kThreads * W);
    if (whole_chunk<W>(b, nbytes)) {
      stw<W>(o + b, v[k]);
    } else {
#pragma unroll 1
      for (uint32_t j = b; j != b + W; ++j)  // cut by the region's start or end
        if (j < nbytes) o[j] = ZERO ? (uint8_t)0 : s[j];
    }
  }
}

// ── kernels ───────────────────────────────────────────────────────────────

// Reads a whole descriptor before any of its fields is tested. Left to itself the compiler
// loads the kind, branches on it and only then loads the fields the branch uses: one more round
// of dependent scalar loads at the start of every workgroup (tile map entry, kind, fields).
__device__ __forceinline__ sh_unpack_desc load_desc(const sh_unpack_desc* __restrict__ p) {
  static_assert(sizeof(sh_unpack_desc) == 64, "descriptor is 16 dwords");
  uint32_t w[16];
  __builtin_memcpy(w, p, sizeof w);
#pragma unroll
  for (int i = 0; i < 16; ++i) asm volatile("" : "+s"(w[i]));  // every dword in an SGPR here
  sh_unpack_desc d;
  __builtin_memcpy(&d, w, sizeof d);
  return d;
}

template <uint32_t MASK, bool HAS_ZP, bool PACED>
__device__ __forceinline__ void unpack_tile(const sh_unpack_desc& d, uint32_t tile,
                                            const uint8_t* __restrict__ src,
                                            const float* __restrict__ scales,
                                            const float* __restrict__ zps,
                                            uint8_t* __restrict__ dst) {
  const uint32_t local = tile - d.tile_begin;
  // The single-kind kernels are launched only for plans whose every descriptor has that kind
  // (launch_tiles), so they test no kind.
  if constexpr (MASK == kMaskDequantBf16) {
    tile_i8<true, HAS_ZP, true>(d, local, src, scales, zps, dst);
    return;
  }
  if constexpr (MASK == kMaskCastBf16) {
    tile_f32_bf16(d, local, src, dst);
    return;
  }
  switch (d.kind) {
    case SH_KIND_I8_ROWSCALE_BF16:
      if constexpr ((MASK & bit(SH_KIND_I8_ROWSCALE_BF16)) != 0)
        tile_i8<true, HAS_ZP, PACED>(d, local, src, scales, zps, dst);
      break;
    case SH_KIND_I8_ROWSCALE_F32:
      if constexpr ((MASK & bit(SH_KIND_I8_ROWSCALE_F32)) != 0)
        tile_i8<false, HAS_ZP, false>(d, local, src, scales, zps, dst);
      break;
    case SH_KIND_F32_BF16:
      if constexpr ((MASK & bit(SH_KIND_F32_BF16)) != 0) tile_f32_bf16(d, local, src, dst);
      break;
    case SH_KIND_BF16_F32:
      if constexpr ((MASK & bit(SH_KIND_BF16_F32)) != 0) tile_bf16_f32(d, local, src, dst);
      break;
    case SH_KIND_COPY_BYTES:
      if constexpr ((MASK & bit(SH_KIND_COPY_BYTES)) != 0) tile_bytes<false>(d, local, src, dst);
      break;
    case SH_KIND_ZERO_BYTES:
      if constexpr ((MASK & bit(SH_KIND_ZERO_BYTES)) != 0) tile_bytes<true>(d, local, src, dst);
      break;
    default:
      break;
  }
}

template <uint32_t MASK, bool HAS_ZP, bool PACED = false>
__device__ __forceinline__ void unpack_body(const sh_unpack_desc* __restrict__ descs,
                                            const uint32_t* __restrict__ tile_map,
                                            const uint8_t* __restrict__ src,
                                            const float* __restrict__ scales,
                                            const float* __restrict__ zps,
                                            uint8_t* __restrict__ dst) {
  const uint32_t tile = blockIdx.x;
  unpack_tile<MASK, HAS_ZP, PACED>(load_desc(descs + tile_map[tile]), tile, src, scales, zps, dst);
}

// The launch table in the kernel's arguments: the descriptor of a tile is the last one whose
// tile_begin is not above it. One launch in place of three: an MLP block of 6 MB 7.0-10.4 us instead of
// 12.6, bound by the host's call (the rule and both sides are at kMaxArgsTiles, sh_unpack.cpp).
template <bool HAS_ZP>
__device__ __forceinline__ void unpack_args_body(const DescArgs& a, const uint8_t* __restrict__ src,
                                                 const float* __restrict__ scales,
                                                 const float* __restrict__ zps,
                                                 uint8_t* __restrict__ dst) {
  const uint32_t tile = blockIdx.x;
  uint32_t i = 0;
#pragma unroll
  for (uint32_t step = kDescChunk / 2; step > 0; step /= 2)
    if (a.tile_begin[i + step] <= tile) i += step;
  unpack_tile<kMaskAll, HAS_ZP, false>(load_desc(a.d + i), tile, src, scales, zps, dst);
}

}  // namespace

#define SH_KERNEL_ARGS                                                                 \
  const sh_unpack_desc *__restrict__ descs, const uint32_t *__restrict__ tile_map,    \
      const uint8_t *__restrict__ src, const float *__restrict__ scales,              \
      const float *__restrict__ zps, uint8_t *__restrict__ dst

extern "C" __global__ __launch_bounds__(kThreads) void sh_dequant_i8_bf16_kernel(SH_KERNEL_ARGS) {
  unpack_body<kMaskDequantBf16, false>(descs, tile_map, src, scales, zps, dst);
}
extern "C" __global__ __launch_bounds__(kThreads) void sh_dequant_i8_bf16_zp_kernel(SH_KERNEL_ARGS) {
  unpack_body<kMaskDequantBf16, true>(descs, tile_map, src, scales, zps, dst);
}
extern "C" __global__ __launch_bounds__(kThreads) void sh_cast_f32_bf16_kernel(SH_KERNEL_ARGS) {
  unpack_body<kMaskCastBf16, false>(descs, tile_map, src, scales, zps, dst);
}
extern "C" __global__ __launch_bounds__(kThreads) void sh_unpack_mixed_kernel(SH_KERNEL_ARGS) {
  unpack_body<kMaskAll, false>(descs, tile_map, src, scales, zps, dst);
}
extern "C" __global__ __launch_bounds__(kThreads) void sh_unpack_mixed_zp_kernel(SH_KERNEL_ARGS) {
  unpack_body<kMaskAll, true>(descs, tile_map, src, scales, zps, dst);
}

extern "C" __global__ __launch_bounds__(kThreads) void sh_unpack_mixed_paced_kernel(SH_KERNEL_ARGS) {
  unpack_body<kMaskAll, false, true>(descs, tile_map, src, scales, zps, dst);
}
extern "C" __global__ __launch_bounds__(kThreads) void sh_unpack_mixed_paced_zp_kernel(SH_KERNEL_ARGS) {
  unpack_body<kMaskAll, true, true>(descs, tile_map, src, scales, zps, dst);
}

extern "C" __global__ __launch_bounds__(kThreads) void sh_unpack_args_kernel(
    const uint8_t* __restrict__ src, const float* __restrict__ scales, const float* __restrict__ zps,
    uint8_t* __restrict__ dst, DescArgs a) {
  unpack_args_body<false>(a, src, scales, zps, dst);
}
extern "C" __global__ __launch_bounds__(kThreads) void sh_unpack_args_zp_kernel(
    const uint8_t* __restrict__ src, const float* __restrict__ scales, const float* __restrict__ zps,
    uint8_t* __restrict__ dst, DescArgs a) {
  unpack_args_body<true>(a, src, scales, zps, dst);
}

// ── allocation-free launches (sh_unpack_noalloc) ─────────────────────────────
//
// A short table travels in the launch's arguments (DescArgs, above). The launch table and the tile
// map of any other call live in this file-scope array, one copy per
// GPU (each device's load of the code object holds its own), until the library unloads its
// kernels: descriptors at offset 0, the tile map after them. The host never names this
// array: it looks up the device address by name in the loaded module (hipModuleGetGlobal,
// sh_kernels.cpp), so the symbol has external C linkage.
static_assert(SH_UNPACK_NOALLOC_SCRATCH_BYTES ==
                  SH_UNPACK_NOALLOC_MAX_DESCS * sizeof(sh_unpack_desc) + SH_UNPACK_NOALLOC_MAX_TILES * 4ull,
              "scratch layout: descriptor table, then one uint32 per tile");
extern "C" {
__device__ __align__(256) uint8_t scratch[SH_UNPACK_NOALLOC_SCRATCH_BYTES];
}

extern "C" __global__ __launch_bounds__(kDescChunk) void sh_put_descs_kernel(DescChunk c, sh_unpack_desc* table) {
  if (threadIdx.x < c.count) table[c.first + threadIdx.x] = c.d[threadIdx.x];
}

// map[t] = the descriptor whose tiles [tile_begin, tile_begin + ntiles) hold t. Descriptors
// hold consecutive, non-empty tile ranges in table order, so a binary search over tile_begin
// finds it.
extern "C" __global__ __launch_bounds__(256) void sh_fill_tile_map_kernel(const sh_unpack_desc* __restrict__ table,
                                                                          uint32_t n, uint32_t* __restrict__ map,
                                                                          uint32_t n_tiles) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= n_tiles) return;
  uint32_t lo = 0, hi = n - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (table[mid].tile_begin <= t) lo = mid;
    else hi = mid - 1;
  }
  map[t] = lo;
}

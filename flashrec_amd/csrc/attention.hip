// Paged attention over the e4m3 KV pool (page size 1): every query token
// attends to its own ragged list of slots.
//
// Reference: python/flashrec/attention/flashinfer.py:380-431 (_sdpa, the
// fallback that defines the result: gather k/v rows by slot, cast to the
// query dtype, scaled_dot_product_attention with scale D^-0.5, grouped-query
// heads repeated) and :240-378 (paged KV view and the decode / prefill
// plans: kv_indptr / kv_indices, page size 1, kv heads in NHD layout).  A
// query token t sees the slots kv_indices[kv_start[t] .. + kv_len[t]) — one
// token per row in decode; in causal prefill, token j of a row with prefix P
// sees P + j + 1.
//
// The work of one call goes in whole groups of 32 / NREP consecutive query
// tokens (32 query rows), each group and kv head an item of its own on bf16
// MFMA (attend_segment).  The tokens of a group are taken in segments that
// read common keys: one segment where all of them see the same first 32 slots
// (beams of one request over their shared prompt, or a prompt's tokens at
// 32 keys and more), else runs of tokens that share a slot list (the first
// tokens of a prompt) or at least 32 leading slots (beams of two requests
// meeting in a group), down to single tokens.  An item's key blocks are split
// over NW waves of a workgroup when the items alone do not fill the chip.
// Arithmetic in fp32 (e4m3 and bf16 convert exactly); the probabilities of
// whole groups are rounded to bf16 (as the reference's bf16 SDPA does), those
// of groups in several segments keep their fp32 value, as three bf16 terms.
// Output bf16.
#include <type_traits>

#include "attn_plan.h"
#include "fr_common.h"

namespace fr {

struct AttnArgs {
  const uint16_t* q;  // [T, Hq, 128] bf16
  int64_t sqt, sqh;
  const uint8_t* kc;  // [slots, Hk, 128] e4m3
  const uint8_t* vc;
  int64_t skp, skh, svp, svh;
  const int32_t* kv_indices;
  const int32_t* kv_start;  // [T]
  const int32_t* kv_len;    // [T]
  uint16_t* out;            // [T, Hq, 128] bf16
  int64_t sot, soh;
  int64_t T, Hq, Hk, num_slots;
  uint32_t row16;  // slot stride of both caches in 16-byte units, 0 where they differ or offsets pass 2^32
  float qscale;  // softmax scale * log2(e)
  const int32_t* gp;  // the plan (attn_plan.h), or null
};

// Longest slot prefix shared by the `count` tokens from t0 on (count <= TOK).
// Lanes 0 .. count-1 fetch the tokens' (start, length) in one load; every
// comparison load of a 64-position chunk is issued before any is used.
template <int TOK>
__device__ __forceinline__ int32_t tokens_prefix(const AttnArgs& a, int64_t t0, int count, int lane) {
  int32_t my_start = 0, my_len = 0x7FFFFFFF;
  if (lane < count) {
    my_start = a.kv_start[t0 + lane];
    my_len = a.kv_len[t0 + lane];
  }
  int32_t lenmin = my_len;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) lenmin = min(lenmin, __shfl_xor(lenmin, o, 64));
  // unconditional loads (lists past the last token read the first token's,
  // positions past the shortest list its last one): under a branch each would
  // wait for the one before it
  int32_t starts[TOK];
#pragma unroll
  for (int tt = 0; tt < TOK; ++tt) starts[tt] = __builtin_amdgcn_readlane(my_start, tt < count ? tt : 0);
  int32_t P = 0;
  for (int32_t c = 0; c < lenmin; c += 64) {
    const bool in = c + lane < lenmin;
    const int32_t pos = in ? c + lane : lenmin - 1;
    int32_t sv[TOK];
#pragma unroll
    for (int tt = 0; tt < TOK; ++tt) sv[tt] = a.kv_indices[starts[tt] + pos];
    const int32_t s0 = sv[0];
    bool ok = in;
#pragma unroll
    for (int tt = 1; tt < TOK; ++tt) ok = ok && sv[tt] == s0;
    const uint64_t bad = __ballot(!ok);
    if (bad) {
      P = c + __builtin_ctzll(bad);
      break;
    }
    P = c + 64;
  }
  return min(P, lenmin);
}

// Bit tt (1 .. count-1): token t0 + tt reads the slot list of token t0 + tt -
// 1, or shares at least its first 32 slots.
template <int TOK>
__device__ __forceinline__ uint32_t linked_tokens(const AttnArgs& a, int64_t t0, int count, int lane) {
  int32_t my_start = -1, my_len = 0;
  if (lane < count) {
    my_start = a.kv_start[t0 + lane];
    my_len = a.kv_len[t0 + lane];
  }
  const int32_t prev = __shfl_up(my_start, 1, 64), plen = __shfl_up(my_len, 1, 64);
  const bool in = lane > 0 && lane < count;
  uint32_t linked = static_cast<uint32_t>(__ballot(in && my_start == prev));
  const uint32_t tryit = static_cast<uint32_t>(__ballot(in && my_start != prev && my_len >= 32 && plen >= 32));
  int32_t x[TOK], y[TOK];
  const int pos = lane & 31;
#pragma unroll
  for (int tt = 1; tt < TOK; ++tt) {
    // lists that are not to be looked at read a word that is there
    const bool t = (tryit >> tt) & 1u;
    const int32_t* const px = t ? a.kv_indices + __builtin_amdgcn_readlane(my_start, tt) + pos : a.kv_start + t0;
    const int32_t* const py = t ? a.kv_indices + __builtin_amdgcn_readlane(my_start, tt - 1) + pos : a.kv_start + t0;
    x[tt] = *px;
    y[tt] = *py;
  }
#pragma unroll
  for (int tt = 1; tt < TOK; ++tt)
    if (((tryit >> tt) & 1u) && __ballot(x[tt] != y[tt]) == 0) linked |= 1u << tt;
  return linked;
}

// ---------------------------------------------------------------------------
// One wave per (group of 32 / NREP consecutive query tokens, kv head[, share
// of the key blocks]), i.e. 32 query rows, on bf16 MFMA.
//
// Blocks of 32 keys are multiplied for all 32 queries at once:
//   K and V rows are gathered 8 whole rows per 16-byte load (8 lanes a row:
//       a gather in fragment order touches 32 lines per load, and the address
//       path, not the matrix work, then sets the block's time) and staged in
//       wave-private LDS, the next block's gathers in flight meanwhile
//   S^T[32 keys x 32 queries] = K . Q^T   (8 x mfma_f32_32x32x16_bf16; a lane
//       reads 64 bytes of one key row and converts them to bf16 with one op
//       per two bytes; dims are taken in the order 64h + 8s + t on both
//       operands, which leaves the dot products unchanged)
//   online softmax per query: a lane owns one query column and 16 key rows,
//       so the block max takes one cross-lane step
//   O^T[128 x 32] += V^T . P^T  (8 MFMAs; V is staged as bf16 [key][dim] and
//       read back transposed with ds_read_b64_tr_b16; the keys of each 16-key
//       chunk are taken in the order the score layout holds them, so P^T
//       feeds the B operand without a lane exchange)
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t* lds_s16x4_t;

// e4m3 x 8 (two dwords, little-endian) -> bf16 x 8, exact
__device__ __forceinline__ bf16x8_t e4m3x8_to_bf16(uint32_t w0, uint32_t w1) {
  const bf16x2_t a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, false);
  const bf16x2_t b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, true);
  const bf16x2_t c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, false);
  const bf16x2_t d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, true);
  // each pair is one dword: the vector is the four dwords as they are
  return __builtin_bit_cast(bf16x8_t, u32x4{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                            __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)});
}

constexpr int kVRow = 288;   // LDS bytes per staged bf16 V row: 256 + 32 (bank spread)
constexpr int kKRow = 144;   // LDS bytes per staged e4m3 K row: 128 + 16 (bank spread)
constexpr int kStage = 32 * (kVRow + kKRow);  // one wave's staging

// A run of consecutive tokens of a group that read common keys.
struct Segment {
  int32_t first, count;  // tokens of the group
  int32_t shared;        // leading list positions that hold the same slots for all of them
  bool one_list;         // the tokens read one slot list, each its own length of it
};

// What a lane knows about its query column n = lane % 32: token t0 + n / NREP,
// head kh * NREP + n % NREP, and 64 of its 128 dims.
struct Query {
  u32x4 q[8];
  int32_t start, len;  // the token's slot list (len 0 past the last token)
  bool ok;
};

template <int NREP>
__device__ __forceinline__ Query load_query(const AttnArgs& a, int64_t t0, int kh, int lane) {
  Query Q;
  const int n = lane & 31, h = lane >> 5;
  const int64_t t = t0 + n / NREP;
  Q.ok = t < a.T;
  Q.len = Q.ok ? a.kv_len[t] : 0;
  Q.start = a.kv_start[Q.ok ? t : t0];
  const uint16_t* qp = a.q + (Q.ok ? t : t0) * a.sqt + (kh * NREP + n % NREP) * a.sqh + 64 * h;
#pragma unroll
  for (int s = 0; s < 8; ++s) Q.q[s] = Q.ok ? *reinterpret_cast<const u32x4*>(qp + 8 * s) : u32x4{0, 0, 0, 0};
  return Q;
}

// Softmax state of a lane's query over the keys seen so far: both halves hold
// the same m; l and O are per half (O^T rows 32 mt + 8 (v / 4) + 4 h + v % 4).
struct Softmax {
  float m, l;
  f32x16_t O[4];
};

// Block range [part * blocks / parts, (part + 1) * blocks / parts) of a
// segment, for the queries of its tokens (the other columns' results mean
// nothing).  FINE: probabilities as three bf16 terms, and `nan` reports a NaN
// code in a V row that some of the segment's queries must not see (its product
// with their zero probability would still be NaN).  `stage`: kStage bytes of
// this wave's LDS.
template <int NREP, bool FINE>
__device__ __forceinline__ void attend_segment(const AttnArgs& a, uint8_t* stage, int kh, int lane, const Query& Q,
                                               const Segment& seg, int part, int parts, Softmax& X, bool& nan) {
  uint8_t* const vs = stage;
  uint8_t* const ks = stage + 32 * kVRow;
  const int n = lane & 31;  // query column, and key row when reading K
  const int h = lane >> 5;  // half: dims 64h .. 64h + 63
  const int tok = n / NREP;
  const bool inseg = tok >= seg.first && tok < seg.first + seg.count;
  const int32_t qlen = inseg ? Q.len : 0;
  X.m = -__builtin_inff();
  X.l = 0.0f;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int v = 0; v < 16; ++v) X.O[mt][v] = 0.0f;

  int32_t maxlen = qlen, minlen = inseg && Q.ok ? Q.len : 0x7FFFFFFF;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    maxlen = max(maxlen, __shfl_xor(maxlen, o, 64));
    minlen = min(minlen, __shfl_xor(minlen, o, 64));
  }
  // Blocks of 32 key rows.  Block b < nshared: row r is position 32 b + r of
  // the common list; after that, row r holds position shared + (b - nshared) *
  // NREP + r % NREP of token r / NREP's own list, and each query only sees its
  // own token's rows.  (No more common positions than the shortest list has,
  // whatever a plan made for other lists says.)
  const int32_t P = seg.one_list ? maxlen : max(min(seg.shared, minlen), 0);
  const int32_t rest = seg.one_list ? 0 : maxlen - P;
  const int32_t nshared = (P + 31) / 32;
  const int32_t nblocks = nshared + (rest > 0 ? (rest + NREP - 1) / NREP : 0);
  const int32_t b0 = part * nblocks / parts, b1 = (part + 1) * nblocks / parts;
  // blocks from here on hold rows that some query of the segment must not see
  const int32_t clean = min(nshared, seg.one_list ? minlen / 32 : nshared);
  const int32_t* const i0 = a.kv_indices + __builtin_amdgcn_readlane(Q.start, seg.first * NREP);
  const int32_t* const ik = a.kv_indices + Q.start;

  // Slot of key row n of block b (-1: none), fetched a block ahead of its
  // gathers.  Gathers are unconditional (an invalid row reads slot 0's
  // bytes); scores of invalid rows are masked and their V rows zeroed, so
  // nothing from them (not even a NaN pattern) reaches the sums.
  auto slot_of = [&](int32_t b) __attribute__((always_inline)) -> int32_t {
    if (b >= b1) return -1;
    if (b < nshared) {
      const int32_t pos = 32 * b + n;
      return pos < P ? i0[pos] : -1;
    }
    const int32_t pos = P + (b - nshared) * NREP + n % NREP;
    return pos < qlen ? ik[pos] : -1;
  };
  const int gr = lane >> 3;         // gathers: row 8 i + gr, bytes 16 (lane % 8) ..
  const int gc = (lane & 7) * 16;
  const uint8_t* const kbase = a.kc + kh * a.skh + gc;
  const uint8_t* const vbase = a.vc + kh * a.svh + gc;
  u32x4 kw[4], vw[4];
  uint32_t rows_ok = 0;  // bit r: key row r of the gathered block usable
  auto gather = [&](int32_t slot) __attribute__((always_inline)) {
    const bool ok = slot >= 0 && slot < a.num_slots;
    rows_ok = static_cast<uint32_t>(__ballot(ok));
    const int32_t sl = ok ? slot : 0;
    if (a.row16 != 0) {
      // one pool layout, offsets in 16-byte units below 2^32: one multiply per
      // block, made by the lane that holds the slot (quarter-rate: 64-bit
      // products per gathered row took a third of the block's issue time)
      const uint32_t off = static_cast<uint32_t>(sl) * a.row16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint64_t o = static_cast<uint64_t>(static_cast<uint32_t>(__shfl(static_cast<int>(off), 8 * i + gr, 64))) << 4;
        kw[i] = *reinterpret_cast<const u32x4*>(kbase + o);
        vw[i] = *reinterpret_cast<const u32x4*>(vbase + o);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t s = __shfl(sl, 8 * i + gr, 64);
      kw[i] = *reinterpret_cast<const u32x4*>(kbase + s * a.skp);
      vw[i] = *reinterpret_cast<const u32x4*>(vbase + s * a.svp);
    }
  };

  // kind 0: every query sees every valid row; 1: rows below its own length;
  // 2: its own token's rows
  auto compute = [&](int32_t b, uint32_t ok_rows, auto kind_c) __attribute__((always_inline)) {
    constexpr int KIND = decltype(kind_c)::value;
    // S^T = K . Q^T
    f32x16_t S;
#pragma unroll
    for (int v = 0; v < 16; ++v) S[v] = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(ks + n * kKRow + 64 * h + 16 * i);
      S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e4m3x8_to_bf16(w[0], w[1]),
                                                  __builtin_bit_cast(bf16x8_t, Q.q[2 * i]), S, 0, 0, 0);
      S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e4m3x8_to_bf16(w[2], w[3]),
                                                  __builtin_bit_cast(bf16x8_t, Q.q[2 * i + 1]), S, 0, 0, 0);
    }
    // scores of this lane's query against key rows r = 8(v/4) + 4h + v%4,
    // unscaled (the scale is positive: the block max scales with them, and
    // each probability takes the scale in one fma)
    float x[16];
    if (KIND == 0 && ok_rows == 0xFFFFFFFFu) {
#pragma unroll
      for (int v = 0; v < 16; ++v) x[v] = S[v];
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = 8 * (v / 4) + 4 * h + (v % 4);
        bool ok = (ok_rows >> r) & 1u;
        if (KIND == 1) ok = ok && 32 * b + r < qlen;
        if (KIND == 2) ok = ok && r / NREP == tok && P + (b - nshared) * NREP + r % NREP < qlen;
        x[v] = ok ? S[v] : -__builtin_inff();
      }
    }
    float mb = x[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) mb = __builtin_fmaxf(mb, x[v]);
    mb = __builtin_fmaxf(mb, __shfl_xor(mb, 32, 64)) * a.qscale;
    // Lazy rescale: probabilities are taken against the reference max m and
    // may reach 2^8; the accumulators are rescaled only when some query's
    // block max passes m + 8 (wave-uniform, so O is touched rarely).
    const bool grow = mb > X.m + 8.0f;
    if (__ballot(grow)) {
      const float mn = grow ? mb : X.m;
      const float alpha = (X.m == -__builtin_inff()) ? 0.0f : __builtin_amdgcn_exp2f(X.m - mn);
      X.m = mn;
      X.l *= alpha;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v) X.O[mt][v] *= alpha;
    }
    // m stays -inf only while every row this query saw was masked; then
    // every x is -inf and the probabilities must be 0, not exp2(NaN)
    const float mref = X.m == -__builtin_inff() ? 0.0f : X.m;
    float pr[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      pr[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(x[v], a.qscale, -mref));  // x = -inf gives 0
      X.l += pr[v];
    }
    // FINE: three terms of 8 significant bits hold all 24 of the fp32
    // probability (each difference is exact)
    constexpr int TERMS = FINE ? 3 : 1;
    bf16x8_t pb[2][TERMS];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int k = 0; k < TERMS; ++k) {
        u32x4 w;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          float& p0 = pr[8 * c + 2 * t];
          float& p1 = pr[8 * c + 2 * t + 1];
          w[t] = pack_bf16x2(p0, p1);
          p0 -= __uint_as_float(w[t] << 16);
          p1 -= __uint_as_float(w[t] & 0xFFFF0000u);
        }
        pb[c][k] = __builtin_bit_cast(bf16x8_t, w);
      }
    // O^T += V^T . P^T; A[dim][k] through the transposing LDS read
    const int g = lane >> 4, i16 = lane & 15;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int col = 32 * mt + 16 * (g & 1) + 4 * (i16 & 3);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int r0 = 16 * c + 4 * h + (i16 >> 2);
        const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(vs + r0 * kVRow + 2 * col));
        const s16x4_t hi =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(vs + (r0 + 8) * kVRow + 2 * col));
        const bf16x8_t av = __builtin_bit_cast(
            bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int k = 0; k < TERMS; ++k)
          X.O[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, pb[c][k], X.O[mt], 0, 0, 0);
      }
    }
  };

  if (b0 >= b1) return;
  // the next block's gathers are in flight while a block is multiplied; the
  // three-term form has no registers to spare for them
  constexpr bool AHEAD = !FINE;
  int32_t slot = slot_of(b0);
  if (AHEAD) {
    gather(slot);
    slot = slot_of(b0 + 1);
  }
  for (int32_t b = b0; b < b1; ++b) {
    if (!AHEAD) {
      gather(slot);
      slot = slot_of(b + 1);
    }
    const uint32_t ok_rows = rows_ok;
    if (ok_rows != 0xFFFFFFFFu) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int w = 0; w < 4; ++w) vw[i][w] = (ok_rows >> (8 * i + gr)) & 1u ? vw[i][w] : 0u;
    }
    if (FINE && b >= clean) {
      uint32_t bad = 0;  // some byte of magnitude 0x7F
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int w = 0; w < 4; ++w) bad |= ((vw[i][w] & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u;
      nan = nan || __ballot(bad != 0) != 0;
    }
    // rows -> LDS: K as it is, V as bf16 [key][dim]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 8 * i + gr;
      *reinterpret_cast<u32x4*>(ks + r * kKRow + gc) = kw[i];
      *reinterpret_cast<bf16x8_t*>(vs + r * kVRow + 2 * gc) = e4m3x8_to_bf16(vw[i][0], vw[i][1]);
      *reinterpret_cast<bf16x8_t*>(vs + r * kVRow + 2 * gc + 16) = e4m3x8_to_bf16(vw[i][2], vw[i][3]);
    }
    if (AHEAD && b + 1 < b1) {
      gather(slot);
      slot = slot_of(b + 2);
    }
    if (b < clean) compute(b, ok_rows, std::integral_constant<int, 0>{});
    else if (b < nshared) compute(b, ok_rows, std::integral_constant<int, 1>{});
    else compute(b, ok_rows, std::integral_constant<int, 2>{});
  }
}

// The whole group as one segment, from its shared prefix rounded down to 32:
// the up to 31 shared positions past that join the common blocks (as own rows
// they would take NREP keys a block: at 28 of them 14 blocks instead of one).
// Lane stride * tt holds token tt's list start and length in (start, len).
template <int TOK>
__device__ __forceinline__ Segment whole_group(const AttnArgs& a, int32_t p32, int32_t start, int32_t len, bool ok,
                                               int stride, int lane) {
  const int32_t st = __builtin_amdgcn_readfirstlane(start);
  if (__ballot(ok && start != st) == 0) return Segment{0, TOK, p32, true};
  int32_t minlen = ok ? len : 0x7FFFFFFF;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) minlen = min(minlen, __shfl_xor(minlen, o, 64));
  // (every list holds p32 positions and more; a token past the last one
  // repeats the first)
  const bool in = p32 + (lane & 31) < minlen;
  const int32_t pos = in ? p32 + (lane & 31) : 0;
  int32_t sv[TOK];
#pragma unroll
  for (int tt = 0; tt < TOK; ++tt) sv[tt] = a.kv_indices[__builtin_amdgcn_readlane(start, tt * stride) + pos];
  bool same = in;
#pragma unroll
  for (int tt = 1; tt < TOK; ++tt) same = same && sv[tt] == sv[0];
  const uint32_t bad = static_cast<uint32_t>(__ballot(!same));  // the two halves agree
  return Segment{0, TOK, p32 + (bad ? __builtin_ctz(bad) : 32), false};
}

// The segment of a group that starts at token `at`, for groups whose tokens do
// not all share 32 slots: the run of linked tokens from there on.  Lane layout
// of (tok, start) as above.
template <int TOK>
__device__ __forceinline__ Segment next_segment(const AttnArgs& a, int64_t t0, int ntok, uint32_t linked, int at,
                                                int tok, int32_t start, int stride, int lane) {
  Segment s{at, 1, 0, true};
  while (at + s.count < ntok && ((linked >> (at + s.count)) & 1u)) ++s.count;
  // one list for all of them?
  const int32_t st = __builtin_amdgcn_readlane(start, at * stride);
  if (__ballot(tok >= at && tok < at + s.count && start != st) == 0) return s;
  s.one_list = false;
  s.shared = tokens_prefix<TOK>(a, t0 + at, s.count, lane);
  return s;
}

// The plan, one wave per group, made once for every layer of a batch (record
// layout in attn_plan.h).
template <int TOK>
__global__ __launch_bounds__(256) void attn_group_plan(AttnArgs a, int32_t* gp, int64_t groups) {
  const int lane = threadIdx.x & 63;
  const int64_t group = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (group >= groups) return;
  const int64_t t0 = group * TOK;
  const int ntok = static_cast<int>(min<int64_t>(TOK, a.T - t0));
  const bool ok = lane < ntok;
  const int32_t start = a.kv_start[ok ? t0 + lane : t0];
  const int32_t p = tokens_prefix<TOK>(a, t0, ntok, lane);
  int32_t cnt = 0, sh = 0;  // lane i: token t0 + i's entries
  if (p >= 32) {
    cnt = lane == 0 ? ntok : 0;
    sh = lane == 0 ? p : 0;
  } else {
    const uint32_t linked = linked_tokens<TOK>(a, t0, ntok, lane);
    for (int at = 0; at < ntok;) {
      const Segment s = next_segment<TOK>(a, t0, ntok, linked, at, ok ? lane : TOK, start, 1, lane);
      if (lane == at) {
        cnt = s.count;
        sh = s.shared;
      }
      at += s.count;
    }
  }
  int32_t* const rec = gp + group * plan_stride(TOK);
  if (lane == 0) {
    rec[0] = p & ~31;
    rec[kPlanTag] = plan_tag(group);
  }
  if (lane < TOK) {
    rec[kPlanCount + lane] = cnt;
    rec[plan_shared_at(TOK) + lane] = sh;
  }
}

// A group's segments: from the plan's record, or found here (no plan, or a
// buffer that holds no record of this group).
template <int NREP>
struct Segments {
  static constexpr int TOK = 32 / NREP;
  int64_t t0;
  int ntok;
  int32_t whole;  // prefix shared by the whole group rounded down to 32 (0: several segments)
  bool planned = false;
  int32_t cnt = 0, sh = 0;  // lane i: the record's entries of token i
  uint32_t linked = 0;
  __device__ __forceinline__ Segments(const AttnArgs& a, int64_t t0_, int64_t group, int lane)
      : t0(t0_), ntok(static_cast<int>(min<int64_t>(TOK, a.T - t0_))) {
    if (a.gp) {
      const int32_t* const rec = a.gp + group * plan_stride(TOK);
      const int i = lane < TOK ? lane : 0;
      whole = rec[0];
      cnt = rec[kPlanCount + i];
      sh = rec[plan_shared_at(TOK) + i];
      planned = __builtin_amdgcn_readfirstlane(rec[kPlanTag]) == plan_tag(group);
    }
    if (!planned) {
      whole = tokens_prefix<TOK>(a, t0, ntok, lane) & ~31;
      if (whole == 0) linked = linked_tokens<TOK>(a, t0, ntok, lane);
    }
  }
  // Segments of the group (as far as the record knows its tokens).
  __device__ __forceinline__ int number(int lane) const {
    return planned ? __builtin_popcountll(__ballot(lane < ntok && cnt > 0)) : ntok - __builtin_popcount(linked);
  }
  __device__ __forceinline__ Segment at(const AttnArgs& a, int first, const Query& Q, bool single, int lane) const {
    if (single) return Segment{first, 1, 0, true};
    const int tok = (lane & 31) / NREP;
    if (planned) {
      const int count = plan_count(__builtin_amdgcn_readlane(cnt, first), first, ntok);
      const int32_t st = __builtin_amdgcn_readlane(Q.start, first * NREP);
      const bool one = __ballot(tok >= first && tok < first + count && Q.start != st) == 0;
      return Segment{first, count, __builtin_amdgcn_readlane(sh, first), one};
    }
    if (whole > 0) return whole_group<TOK>(a, whole, Q.start, Q.len, Q.ok, NREP, lane);
    return next_segment<TOK>(a, t0, ntok, linked, first, tok, Q.start, NREP, lane);
  }
};

// A lane's normalised output row piece: 4 consecutive dims 32 mt + 8 j + 4 h ..
// as bf16 (no visible key: zeros, the softmax of an empty row is undefined).
__device__ __forceinline__ u32x2 out4(const Softmax& X, float inv, int mt, int j) {
  return u32x2{pack_bf16x2(X.O[mt][4 * j] * inv, X.O[mt][4 * j + 1] * inv),
               pack_bf16x2(X.O[mt][4 * j + 2] * inv, X.O[mt][4 * j + 3] * inv)};
}

// One item on one wave: the lane's query's 64 dims as 32 packed bf16 pairs.
template <int NREP>
__device__ __forceinline__ void attend_item(const AttnArgs& a, uint8_t* stage, int64_t group, int kh, int lane,
                                            u32x2 (&o)[16]) {
  const int64_t t0 = group * (32 / NREP);
  const Query Q = load_query<NREP>(a, t0, kh, lane);
  const Segments<NREP> segs(a, t0, group, lane);
  Softmax X;
  bool nan = false;
  if (segs.whole > 0) {
    attend_segment<NREP, false>(a, stage, kh, lane, Q, segs.at(a, 0, Q, false, lane), 0, 1, X, nan);
    const float lt = X.l + __shfl_xor(X.l, 32, 64);
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) o[i] = out4(X, inv, i >> 2, i & 3);
    return;
  }
  const int tok = (lane & 31) / NREP;
  int single_until = 0;
  for (int at = 0; at < segs.ntok;) {
    const Segment s = segs.at(a, at, Q, at < single_until, lane);
    nan = false;
    attend_segment<NREP, true>(a, stage, kh, lane, Q, s, 0, 1, X, nan);
    if (nan && s.count > 1) {
      single_until = at + s.count;
      continue;
    }
    const float lt = X.l + __shfl_xor(X.l, 32, 64);
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    if (tok >= at && tok < at + s.count) {
#pragma unroll
      for (int i = 0; i < 16; ++i) o[i] = out4(X, inv, i >> 2, i & 3);
    }
    at += s.count;
  }
}

// Items on one wave each (launches with enough of them to fill the chip).
template <int NREP>
__global__ __launch_bounds__(64, 2) void paged_attn_d128(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kStage];
  const int lane = threadIdx.x;
  // last groups first: a causal prompt's longest items lead, the short ones
  // fill the tail
  const int64_t groups = (a.T + 32 / NREP - 1) / (32 / NREP);
  const int64_t group = groups - 1 - blockIdx.x / a.Hk;
  const int kh = static_cast<int>(blockIdx.x % a.Hk);
  u32x2 o[16];
  attend_item<NREP>(a, lds, group, kh, lane, o);
  const int n = lane & 31, h = lane >> 5;
  const int64_t t = group * (32 / NREP) + n / NREP;
  if (t >= a.T) return;
  uint16_t* const op = a.out + t * a.sot + (kh * NREP + n % NREP) * a.soh;
#pragma unroll
  for (int i = 0; i < 16; ++i) *reinterpret_cast<u32x2*>(op + 8 * i + 4 * h) = o[i];
}

// An item's key blocks split over NW waves: each wave's softmax state over its
// share, then the states merged through LDS (rescaled to the common max, added
// in wave order) and the rows written by all threads.
template <int NREP, int NW>
__global__ __launch_bounds__(64 * NW, 2) void paged_attn_split_d128(AttnArgs a) {
  constexpr int kMerge = NW * 16384;  // 32 queries x 128 dims fp32 per wave
  __shared__ __attribute__((aligned(16))) uint8_t lds[kMerge > NW * kStage ? kMerge : NW * kStage];
  __shared__ float ms[NW][32], ls[NW][32];
  __shared__ int saw_nan;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t groups = (a.T + 32 / NREP - 1) / (32 / NREP);
  const int64_t group = groups - 1 - blockIdx.x / a.Hk;
  const int kh = static_cast<int>(blockIdx.x % a.Hk);
  const int64_t t0 = group * (32 / NREP);
  const int n = lane & 31, h = lane >> 5;
  const Query Q = load_query<NREP>(a, t0, kh, lane);
  const Segments<NREP> segs(a, t0, group, lane);
  uint8_t* const stage = lds + wave * kStage;

  auto merge = [&](const Segment& s, const Softmax& X) __attribute__((always_inline)) {
    const float lt = X.l + __shfl_xor(X.l, 32, 64);
    if (lane < 32) {
      ms[wave][n] = X.m;
      ls[wave][n] = lt;
    }
    __syncthreads();  // the states' maxima are known, and no wave stages any more
    float M = ms[0][n];
#pragma unroll
    for (int w = 1; w < NW; ++w) M = __builtin_fmaxf(M, ms[w][n]);
    const float sc = X.m == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(X.m - M);
    // query n's 4 dims 4 u .. 4 u + 3 in 16-byte unit u ^ n of its 512 bytes
    // (the 32 lanes of a write, and of a read below, on distinct units)
    float4* const mine = reinterpret_cast<float4*>(lds) + wave * 1024 + n * 32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int mt = i >> 2, j = i & 3, u = 8 * mt + 2 * j + h;
      mine[u ^ n] = make_float4(X.O[mt][4 * j] * sc, X.O[mt][4 * j + 1] * sc, X.O[mt][4 * j + 2] * sc,
                                X.O[mt][4 * j + 3] * sc);
    }
    __syncthreads();
#pragma unroll
    for (int i = threadIdx.x; i < 1024; i += 64 * NW) {
      const int qn = i >> 5, u = i & 31, tok = qn / NREP;
      const int64_t t = t0 + tok;
      float mx = ms[0][qn];
#pragma unroll
      for (int w = 1; w < NW; ++w) mx = __builtin_fmaxf(mx, ms[w][qn]);
      float L = 0.0f;
      float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float4 x = reinterpret_cast<const float4*>(lds)[w * 1024 + qn * 32 + (u ^ qn)];
        const float m = ms[w][qn];
        L += m == -__builtin_inff() ? 0.0f : ls[w][qn] * __builtin_amdgcn_exp2f(m - mx);
        acc.x += x.x;
        acc.y += x.y;
        acc.z += x.z;
        acc.w += x.w;
      }
      const float inv = L > 0.0f ? 1.0f / L : 0.0f;
      if (t < a.T && tok >= s.first && tok < s.first + s.count) {
        uint16_t* const op = a.out + t * a.sot + (kh * NREP + qn % NREP) * a.soh + 4 * u;
        *reinterpret_cast<u32x2*>(op) =
            u32x2{pack_bf16x2(acc.x * inv, acc.y * inv), pack_bf16x2(acc.z * inv, acc.w * inv)};
      }
    }
  };

  Softmax X;
  bool nan = false;
  if (segs.whole > 0) {
    const Segment s = segs.at(a, 0, Q, false, lane);
    attend_segment<NREP, false>(a, stage, kh, lane, Q, s, wave, NW, X, nan);
    merge(Segment{0, 32 / NREP, 0, false}, X);  // tokens that the plan did not know: zeros
    return;
  }
  // Several segments.  As many as waves and more go to the waves in turn, each
  // on one wave and without a merge: rows with lists of their own else pay three
  // barriers and a merge for a block or two of each wave.  16/8 heads, us, split
  // / dealt: 64 rows x 40 keys 79.2 / 26.4 (66.7 token by token on the VALU),
  // 64 x 200 114 / 59.2, 64 x 1500 291 / 219.
  int single_until = 0;
  if (segs.number(lane) >= NW) {
    const int tok = n / NREP;
    int dealt = 0;
    bool mine = false;
    for (int at = 0; at < segs.ntok;) {
      const bool single = at < single_until;
      const Segment s = segs.at(a, at, Q, single, lane);
      if (!single) mine = dealt++ % NW == wave;  // (a segment taken again stays with its wave)
      if (mine) {
        nan = false;
        attend_segment<NREP, true>(a, stage, kh, lane, Q, s, 0, 1, X, nan);
        if (nan && s.count > 1) {
          single_until = at + s.count;
          continue;
        }
        const float lt = X.l + __shfl_xor(X.l, 32, 64);
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        if (tok >= at && tok < at + s.count) {
          uint16_t* const op = a.out + (t0 + tok) * a.sot + (kh * NREP + n % NREP) * a.soh;
#pragma unroll
          for (int i = 0; i < 16; ++i) *reinterpret_cast<u32x2*>(op + 8 * i + 4 * h) = out4(X, inv, i >> 2, i & 3);
        }
      }
      at += s.count;
    }
    return;
  }
  for (int at = 0; at < segs.ntok;) {
    if (threadIdx.x == 0) saw_nan = 0;
    __syncthreads();  // the last merge has been read, the flag is clear
    const Segment s = segs.at(a, at, Q, at < single_until, lane);
    nan = false;
    attend_segment<NREP, true>(a, stage, kh, lane, Q, s, wave, NW, X, nan);
    if (nan && lane == 0) saw_nan = 1;
    __syncthreads();
    if (saw_nan && s.count > 1) {
      single_until = at + s.count;
      __syncthreads();  // every wave has read the flag
      continue;
    }
    merge(s, X);
    at += s.count;
  }
}

// Attention fused with the per-token e4m3 quant of its output (the o_proj
// input, linear.py:118-151 -> sglops.py:84-96): one workgroup per group of
// 32 / NREP tokens, wave w on kv head w (Hk <= 8, NREP < 8).  Each wave
// stages its 32 bf16 output rows in its LDS region; after a barrier, wave w
// takes tokens w, w + 8, ...: the token's Hq x 128 bf16 values (4 heads per
// pass, 8 dims per lane), row amax, scale = amax / 448 and the codes, in the
// row kernels' arithmetic (quant8_e4m3).  The codes are bit-for-bit what
// paged_attn_d128 followed by the per-token quant writes.
template <int NREP>
__global__ __launch_bounds__(512, 1) void paged_attn_grouped_quant_d128(AttnArgs a, uint8_t* qout, int64_t ldq,
                                                                        float* qscale) {
  constexpr int TOK = 32 / NREP;
  __shared__ __attribute__((aligned(16))) uint8_t lds[8 * kStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t group = blockIdx.x;
  const int64_t t0 = group * TOK;
  if (t0 >= a.T) return;
  if (wave < a.Hk) {
    u32x2 o[16];
    attend_item<NREP>(a, lds + wave * kStage, group, wave, lane, o);
    uint8_t* const op = lds + wave * kStage + (lane & 31) * kVRow;
#pragma unroll
    for (int i = 0; i < 16; ++i) *reinterpret_cast<u32x2*>(op + 16 * i + 8 * (lane >> 5)) = o[i];
  }
  __syncthreads();
  const int ntok = static_cast<int>(min<int64_t>(TOK, a.T - t0));
  const int hq = static_cast<int>(a.Hq);
  const int hl = lane >> 4;       // head inside a pass of 4
  const int dl = (lane & 15) * 8;  // first of this lane's 8 dims
  for (int tt = wave; tt < ntok; tt += 8) {
    u32x4 w[8];
    float amax = 0.0f;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      const int head = 4 * p + hl;
      w[p] = u32x4{0, 0, 0, 0};
      if (head < hq) {
        const uint8_t* src = lds + (head / NREP) * kStage + (tt * NREP + head % NREP) * kVRow + 2 * dl;
        w[p] = *reinterpret_cast<const u32x4*>(src);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        amax = maxnan(amax, __builtin_fabsf(__uint_as_float(w[p][i] << 16)));
        amax = maxnan(amax, __builtin_fabsf(__uint_as_float(w[p][i] & 0xFFFF0000u)));
      }
    }
    amax = maxnan(wave_maxnan(amax), kAmaxFloor);
    const float scale = amax / kFp8Max;
    const int64_t t = t0 + tt;
    if (lane == 0) qscale[t] = scale;
    const bool finite = amax < 3.0e38f;
    const float r = 1.0f / scale;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      const int head = 4 * p + hl;
      if (head < hq) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[2 * i] = __uint_as_float(w[p][i] << 16);
          v[2 * i + 1] = __uint_as_float(w[p][i] & 0xFFFF0000u);
        }
        *reinterpret_cast<u32x2*>(qout + t * ldq + head * 128 + dl) = quant8_e4m3(v, scale, r, finite);
      }
    }
  }
}

// Waves per item for a launch of `items` whose slot lists hold `entries`
// slots.  Items alone leave SIMDs idle below about 2048 (two waves on each of
// 1024); splitting costs a merge and, in decode, the quant as a launch of its
// own.  A prompt's tokens share one list (few entries a token); decode rows
// each bring their own, so entries per token is their length.  Measured, us,
// waves 1 / 2 / 4 / 8 (attention; the fused quant or the split plus quant for
// decode; rows x keys, 16 query and 8 kv heads):
//   50 x 202 (32 items)     22.6 /    - / 12.0 / 12.4
//   512 x 130 (256)         17.9 / 13.8 / 12.6 / 12.9    512 x 1503   89.1 / - / 27.8 / 24.6
//   1024 x 130 (512)        18.2 / 16.0 / 15.9 / 21.9    1024 x 1002  64.5 / 38.3 / 30.1 / 36.1
//   1248 x 1133 (624)        180 / 98.9 / 73.4 / 75.4
//   2048 x 130 (1024)       19.6 / 21.5 / 26.7 / 39.1    2048 x 1002  65.8 / 46.1 / 51.1 / 67.9
//   4096 x 130 (2048)       21.9 /    - / 46.4 / 74.3    4096 x 1002  72.7 / 85.3 / 91.1 / 127
//   prefill 1999 (1000)     76.9 / 47.9 / 44.5 / 60.3    4 x 500 (1000)  33.1 / 30.3 / 30.4 / 41.5
//   prefill 4000 (2000)      159 /  122 /  125 /  159
// A kv head per query head makes groups of 32 tokens, whose segments gain most
// from being dealt to waves (attention alone): 1024 rows x 200, a list each, 32/32
// heads 542 / 398 / 393 / 415; 8 requests x 512 beams x 132, 8/8 heads 18.5 / 18.7.
static int attn_waves(int64_t T, int64_t items, int64_t entries, int64_t nrep) {
  const int64_t simds = 4 * num_cus();
  const bool prompt = entries < 8 * T;
  const int64_t keys = entries / T;
  if (4 * items <= simds) return prompt || keys > 600 ? 8 : 4;
  if (2 * items <= simds) return 4;
  if (items <= simds) return prompt ? 4 : (keys < 300 ? (nrep == 1 ? 2 : 1) : (4 * items <= 3 * simds ? 4 : 2));
  return prompt && items <= 2 * simds ? 2 : 1;
}

template <int NREP>
static hipError_t launch_attn(const AttnArgs& a, int waves, hipStream_t st) {
  const int64_t items = (a.T + 32 / NREP - 1) / (32 / NREP) * a.Hk;
  const dim3 grid(static_cast<unsigned>(items));
  switch (waves) {
    case 8: hipLaunchKernelGGL((paged_attn_split_d128<NREP, 8>), grid, dim3(512), 0, st, a); break;
    case 4: hipLaunchKernelGGL((paged_attn_split_d128<NREP, 4>), grid, dim3(256), 0, st, a); break;
    case 2: hipLaunchKernelGGL((paged_attn_split_d128<NREP, 2>), grid, dim3(128), 0, st, a); break;
    default: hipLaunchKernelGGL((paged_attn_d128<NREP>), grid, dim3(64), 0, st, a); break;
  }
  return hipGetLastError();
}

}  // namespace fr

using namespace fr;

template <int NREP>
static hipError_t launch_grouped_quant(const AttnArgs& a, uint8_t* qout, int64_t ldq, float* qs, hipStream_t st) {
  const int64_t groups = (a.T + 32 / NREP - 1) / (32 / NREP);
  hipLaunchKernelGGL((paged_attn_grouped_quant_d128<NREP>), dim3(static_cast<unsigned>(groups)), dim3(512), 0, st,
                     a, qout, ldq, qs);
  return hipGetLastError();
}

// Checks shared by both entry points; fills `a` (output fields left unset).
static int attn_args(AttnArgs& a, const void* q, int64_t sqt, int64_t sqh, const void* k_cache, int64_t skp,
                     int64_t skh, const void* v_cache, int64_t svp, int64_t svh, int64_t num_slots,
                     const int32_t* kv_indices, const int32_t* kv_start, const int32_t* kv_len, int64_t T,
                     int64_t Hq, int64_t Hk, int64_t D, float scale, const int32_t* group_prefix) {
  if (T < 0 || Hq <= 0 || Hk <= 0 || D <= 0) return FR_EINVAL;
  if (T > 0 && (!q || !k_cache || !v_cache || !kv_indices || !kv_start || !kv_len)) return FR_EINVAL;
  if (D != 128 || Hq % Hk != 0) return FR_EUNSUPPORTED;
  const int64_t nrep = Hq / Hk;
  if (nrep != 1 && nrep != 2 && nrep != 4 && nrep != 8) return FR_EUNSUPPORTED;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  // 16-byte vector access: row and head strides in whole 16-byte units
  if (!al16(q) || !al16(k_cache) || !al16(v_cache) || sqt % 8 || sqh % 8 || skp % 16 || skh % 16 || svp % 16 ||
      svh % 16)
    return FR_EUNSUPPORTED;
  a = AttnArgs{};
  a.q = static_cast<const uint16_t*>(q);
  a.sqt = sqt;
  a.sqh = sqh;
  a.kc = static_cast<const uint8_t*>(k_cache);
  a.vc = static_cast<const uint8_t*>(v_cache);
  a.skp = skp;
  a.skh = skh;
  a.svp = svp;
  a.svh = svh;
  a.kv_indices = kv_indices;
  a.kv_start = kv_start;
  a.kv_len = kv_len;
  a.T = T;
  a.Hq = Hq;
  a.Hk = Hk;
  a.num_slots = num_slots;
  a.row16 = skp == svp && skp > 0 && num_slots <= (int64_t(1) << 32) / (skp / 16) ? static_cast<uint32_t>(skp / 16) : 0;
  a.qscale = scale * 1.4426950408889634f;
  a.gp = group_prefix;
  return FR_OK;
}

extern "C" int fr_paged_attention_split_fp8(const void* q, int64_t sqt, int64_t sqh, const void* k_cache,
                                            int64_t skp, int64_t skh, const void* v_cache, int64_t svp,
                                            int64_t svh, int64_t num_slots, const int32_t* kv_indices,
                                            const int32_t* kv_start, const int32_t* kv_len, void* out,
                                            int64_t sot, int64_t soh, int64_t T, int64_t Hq, int64_t Hk,
                                            int64_t D, float scale, const int32_t* group_prefix, int waves,
                                            void* stream) {
  AttnArgs a;
  const int rc = attn_args(a, q, sqt, sqh, k_cache, skp, skh, v_cache, svp, svh, num_slots, kv_indices, kv_start,
                           kv_len, T, Hq, Hk, D, scale, group_prefix);
  if (rc != FR_OK) return rc;
  if (waves != 1 && waves != 2 && waves != 4 && waves != 8) return FR_EINVAL;
  if (T == 0) return FR_OK;
  if (!out) return FR_EINVAL;
  if ((reinterpret_cast<uintptr_t>(out) & 15u) || sot % 8 || soh % 8) return FR_EUNSUPPORTED;
  a.out = static_cast<uint16_t*>(out);
  a.sot = sot;
  a.soh = soh;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e;
  switch (Hq / Hk) {
    case 1: e = launch_attn<1>(a, waves, st); break;
    case 2: e = launch_attn<2>(a, waves, st); break;
    case 4: e = launch_attn<4>(a, waves, st); break;
    default: e = launch_attn<8>(a, waves, st); break;
  }
  return e == hipSuccess ? FR_OK : FR_ELAUNCH;
}

extern "C" int fr_paged_attention_fp8(const void* q, int64_t sqt, int64_t sqh, const void* k_cache,
                                      int64_t skp, int64_t skh, const void* v_cache, int64_t svp,
                                      int64_t svh, int64_t num_slots, const int32_t* kv_indices,
                                      const int32_t* kv_start, const int32_t* kv_len, void* out,
                                      int64_t sot, int64_t soh, int64_t T, int64_t Hq, int64_t Hk,
                                      int64_t D, float scale, const int32_t* group_prefix,
                                      void* stream) {
  return fr_paged_attention_split_fp8(q, sqt, sqh, k_cache, skp, skh, v_cache, svp, svh, num_slots, kv_indices,
                                      kv_start, kv_len, out, sot, soh, T, Hq, Hk, D, scale, group_prefix, 1, stream);
}

extern "C" int fr_paged_attention_quant_fp8(const void* q, int64_t sqt, int64_t sqh, const void* k_cache,
                                            int64_t skp, int64_t skh, const void* v_cache, int64_t svp,
                                            int64_t svh, int64_t num_slots, const int32_t* kv_indices,
                                            const int32_t* kv_start, const int32_t* kv_len, void* out_q,
                                            int64_t ldq, float* out_scale, int64_t T, int64_t Hq, int64_t Hk,
                                            int64_t D, float scale, const int32_t* group_prefix, void* stream) {
  AttnArgs a;
  const int rc = attn_args(a, q, sqt, sqh, k_cache, skp, skh, v_cache, svp, svh, num_slots, kv_indices, kv_start,
                           kv_len, T, Hq, Hk, D, scale, group_prefix);
  if (rc != FR_OK) return rc;
  // one wave per kv head in a workgroup of 8; the quantizing passes hold a token
  // of up to 32 heads, which 8 query heads for each of 8 kv heads would pass
  if (Hk > 8 || Hq / Hk == 8) return FR_EUNSUPPORTED;
  if (T == 0) return FR_OK;
  if (!out_q || !out_scale || ldq < Hq * D) return FR_EINVAL;
  if ((reinterpret_cast<uintptr_t>(out_q) & 7u) || ldq % 8) return FR_EUNSUPPORTED;  // 8-byte code stores
  uint8_t* qo = static_cast<uint8_t*>(out_q);
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e;
  switch (Hq / Hk) {
    case 1: e = launch_grouped_quant<1>(a, qo, ldq, out_scale, st); break;
    case 2: e = launch_grouped_quant<2>(a, qo, ldq, out_scale, st); break;
    default: e = launch_grouped_quant<4>(a, qo, ldq, out_scale, st); break;
  }
  return e == hipSuccess ? FR_OK : FR_ELAUNCH;
}

// Query groups of T tokens (-1: unsupported head ratio).
static int64_t attn_groups(int64_t T, int64_t Hq, int64_t Hk) {
  if (T < 0 || Hq <= 0 || Hk <= 0 || Hq % Hk != 0) return -1;
  const int64_t nrep = Hq / Hk;
  if (nrep != 1 && nrep != 2 && nrep != 4 && nrep != 8) return -1;
  const int64_t tok = 32 / nrep;
  return (T + tok - 1) / tok;
}

extern "C" int64_t fr_paged_attention_plan_size(int64_t T, int64_t Hq, int64_t Hk) {
  const int64_t groups = attn_groups(T, Hq, Hk);
  return groups < 0 ? -1 : groups * plan_stride(static_cast<int>(32 / (Hq / Hk)));
}

extern "C" int fr_paged_attention_waves(int64_t T, int64_t Hq, int64_t Hk, int64_t entries) {
  const int64_t groups = attn_groups(T, Hq, Hk);
  return groups <= 0 || entries < 0 ? 1 : attn_waves(T, groups * Hk, entries, Hq / Hk);
}

extern "C" int fr_paged_attention_plan(const int32_t* kv_indices, const int32_t* kv_start,
                                       const int32_t* kv_len, int64_t T, int64_t Hq, int64_t Hk,
                                       int32_t* group_prefix, void* stream) {
  const int64_t groups = attn_groups(T, Hq, Hk);
  if (groups < 0) return FR_EUNSUPPORTED;
  if (groups == 0) return FR_OK;
  if (!kv_indices || !kv_start || !kv_len || !group_prefix) return FR_EINVAL;
  AttnArgs a{};
  a.kv_indices = kv_indices;
  a.kv_start = kv_start;
  a.kv_len = kv_len;
  a.T = T;
  a.Hq = Hq;
  a.Hk = Hk;
  const dim3 grid(static_cast<unsigned>((groups + 3) / 4)), block(256);
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (Hq / Hk) {
    case 1: hipLaunchKernelGGL((attn_group_plan<32>), grid, block, 0, st, a, group_prefix, groups); break;
    case 2: hipLaunchKernelGGL((attn_group_plan<16>), grid, block, 0, st, a, group_prefix, groups); break;
    case 4: hipLaunchKernelGGL((attn_group_plan<8>), grid, block, 0, st, a, group_prefix, groups); break;
    default: hipLaunchKernelGGL((attn_group_plan<4>), grid, block, 0, st, a, group_prefix, groups); break;
  }
  return hipGetLastError() == hipSuccess ? FR_OK : FR_ELAUNCH;
}

// W8A8 fp8 GEMM for launches whose output has too few tiles to fill the chip
// (few activation rows, or a narrow output with a long K):
//   out[m, n] = (sum_k a[m, k] * w[n, k]) * sa[m] * sb[n] (+ bias[n])
// the same product and epilogue variants as gemm_fp8.hip and gemm_fp8_pre.hip
// (python/flashrec/kernel/sglops.py:99-140), for both weight layouts.
//
// What bounds those launches is not the matrix cores but how few bytes are in
// flight: at M = 20 the down projection (N 2048, K 6144) is 16 tiles of
// 128 x 128, so 16 of 256 CUs stream 12.6 MB through 96 dependent K steps.
// Here the output tile is small (32 or 64 columns x 32 .. 128 rows) and K is
// split over the NW waves of the workgroup: each wave multiplies the whole
// tile over its own K range with loads of its own (no barrier in the K
// loop), and the partial sums are added in wave order through LDS at the end,
// so the result does not depend on timing.
//  * Activations: a wave-private LDS ring of NS slots (128 bytes of K each),
//    filled by direct-to-LDS loads of whole 128-byte row pieces (fragment
//    loads straight from rows touch 32 lines per instruction), XOR-swizzled
//    as in the large kernels.
//  * Weights: prearranged blocks come as contiguous 1 KB runs straight into
//    registers, one register set per ring slot; [N, K] rows as 16-byte pieces
//    in the same fragment order, so both layouts give the same bits.
#include "gemm_common.h"

namespace fr {

constexpr uint32_t kOob = 0x80000000u;

// The four 16-byte fragment pieces of one 32-row block and ring slot (two K
// steps), waited for inside the statement.
template <int OFF>
__device__ __forceinline__ void read_block(const uint32_t (&ad)[4], u32x4 (&v)[4]) {
  asm volatile(
      "ds_read_b128 %0, %4 offset:%8\n\tds_read_b128 %1, %5 offset:%8\n\t"
      "ds_read_b128 %2, %6 offset:%8\n\tds_read_b128 %3, %7 offset:%8\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
      : "v"(ad[0]), "v"(ad[1]), "v"(ad[2]), "v"(ad[3]), "n"(OFF)
      : "memory");
}

template <int FN, int FM, int NW, int NS, bool PRE, bool SILU>
__global__ __launch_bounds__(64 * NW) void gemm_fp8_small(GemmArgs g, int out_dtype) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BN = 32 * FN, BM = 32 * FM;
  constexpr int SLOT = BM * 128;           // bytes of one activation slot
  constexpr int IA = SLOT / 1024;          // its 1 KB loads
  constexpr int IW = 4 * FN;               // weight loads per slot (two K steps, two halves)
  constexpr int OPS = IA + IW;             // vector-memory operations per slot
  constexpr int RING = NW * NS * SLOT;
  constexpr int RED = NW * FN * FM * 4096;  // partial sums
  static_assert((NS - 1) * OPS < 64, "vmcnt range");
  static_assert(NS * SLOT <= 65536, "ring offsets are instruction immediates");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[RING > RED ? RING : RED];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t tilesN = static_cast<uint32_t>((g.N + BN - 1) / BN);
  const uint32_t tilesM = static_cast<uint32_t>((g.M + BM - 1) / BM);
  // workgroup i runs on XCD i % 8: each XCD takes a contiguous run of tiles,
  // row tiles fastest, so the tiles that share weights share an L2
  const uint32_t nt = tilesN * tilesM, chunk = (nt + 7) / 8;
  const uint32_t id = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= chunk || id >= nt) return;
  const int64_t m0 = static_cast<int64_t>(id % tilesM) * BM;
  const int64_t n0 = static_cast<int64_t>(id / tilesM) * BN;

  // K in slots of 128 bytes (the prearranged layout's count: a multiple of
  // two), split over the waves
  const int KS = static_cast<int>((g.K + 255) / 256) * 2;
  const int s0 = wave * KS / NW, s1 = (wave + 1) * KS / NW;

  const __amdgpu_buffer_rsrc_t ra = make_rsrc(g.a, static_cast<uint32_t>((g.M - 1) * g.lda + g.K));
  const uint32_t wblk = static_cast<uint32_t>(g.ldb);  // PRE: bytes per 32-row block, else row stride
  const __amdgpu_buffer_rsrc_t rw =
      PRE ? make_rsrc(g.b, static_cast<uint32_t>((g.N + 31) / 32 * wblk))
          : make_rsrc(g.b, static_cast<uint32_t>((g.N - 1) * g.ldb + g.K));

  uint8_t* const ring = smem + wave * (NS * SLOT);
  // lane L of a 1 KB load: row L / 8 of its 8 rows, chunk slot L % 8 holding
  // the row's chunk (L % 8) ^ ((row / 2) % 8)
  const int lrow = lane >> 3;
  const int lchunk = (lane & 7) ^ (lrow >> 1);  // of even loads; odd ones hold chunk ^ 4
  const uint32_t la = static_cast<uint32_t>((m0 + lrow) * g.lda);
  const uint32_t a8 = static_cast<uint32_t>(8 * g.lda);
  uint32_t wv;
  if constexpr (PRE) wv = static_cast<uint32_t>(n0 / 32) * wblk + 16 * lane;
  else wv = static_cast<uint32_t>((n0 + (lane & 31)) * g.ldb) + 32 * (lane >> 5);

  u32x4 wr[NS][2][FN][2];
  auto issue = [&](int q, int s) __attribute__((always_inline)) {
    const bool live = s < s1;  // past the wave's range: zeros (keeps the counts of the waits)
    const int64_t krem = g.K - static_cast<int64_t>(s) * 128;  // bytes of K from this slot on
#pragma unroll
    for (int i = 0; i < IA; ++i) {
      const int c = lchunk ^ ((i & 1) * 4);
      const bool in = live && c * 16 < krem;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(ring + q * SLOT + i * 1024), 16,
                                               in ? la + i * a8 + c * 16 : kOob, s * 128, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          uint32_t vo;
          int so;
          if constexpr (PRE) {
            vo = live ? wv + i * wblk + h * 1024 : kOob;
            so = (2 * s + u) * 2048;
          } else {
            const bool in = live && 64 * u + 32 * (lane >> 5) + 16 * h < krem;
            vo = in ? wv + i * 32 * wblk + 16 * h : kOob;
            so = s * 128 + 64 * u;
          }
          wr[q][u][i][h] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, vo, so, 0));
        }
  };

  // The outputs this thread finishes are known from the start: column group
  // cg (4 columns; with SiLU the gate group, its up group two further) of rows
  // row0 + RS * u.  Their scales and residual are fetched behind the first K
  // loads, so the epilogue waits for no load of its own (about 1 us).
  constexpr int CG = BN / 4;             // column groups per row
  constexpr int T = 64 * NW;
  constexpr int UPT = BM * CG / T > 0 ? BM * CG / T : 1;  // outputs of 4 columns per thread
  const int cgs = SILU ? CG / 2 : CG;
  const int cx = tid % cgs, row0 = tid / cgs;
  constexpr int RS = T / (SILU ? CG / 2 : CG);
  const int cg = SILU ? (cx >> 1) * 4 + (cx & 1) : cx;
  const int64_t n = n0 + 4 * cg;
  constexpr int NU = SILU ? (UPT + 1) / 2 : UPT;
  float sbv[SILU ? 8 : 4], sav[NU];
  u32x2 resv[NU];
  // 8-byte output (and residual) pieces where the rows allow them
  const bool wide = n + 4 <= g.N && g.bias == nullptr && g.ldo % 4 == 0 &&
                    (reinterpret_cast<uintptr_t>(g.out) & 7) == 0 &&
                    (g.res == nullptr || (g.ldr % 4 == 0 && (reinterpret_cast<uintptr_t>(g.res) & 7) == 0));
  auto fetch_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      sbv[t] = g.sb[(n + t < g.N ? n + t : g.N - 1) * g.sb_stride];
      if constexpr (SILU) sbv[4 + t] = g.sb[(n + 8 + t < g.N ? n + 8 + t : g.N - 1) * g.sb_stride];
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int64_t m = m0 + row0 + RS * u;
      const int64_t mc = m < g.M ? m : g.M - 1;
      sav[u] = g.sa[mc * g.sa_stride];
      resv[u] = u32x2{0u, 0u};
      if (!SILU && g.res && wide)
        resv[u] = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(g.res) + mc * g.ldr + n);
    }
  };

  // fragment reads: lane l reads row l % 32, chunks 4 u + 2 (l / 32) + h
  const int fr = lane & 31;
  const uint32_t rbase = lds_addr(ring) + fr * 128;
  const int c0 = (lane >> 5) * 2, gx = swz_g8(fr);
  const uint32_t ad[4] = {rbase + ((c0 ^ gx) << 4), rbase + (((c0 ^ 1) ^ gx) << 4), rbase + (((c0 ^ 4) ^ gx) << 4),
                          rbase + (((c0 ^ 5) ^ gx) << 4)};
  v16f acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = v16f{};

  auto slot = [&](auto qc) __attribute__((always_inline)) {
    constexpr int q = decltype(qc)::value;
    waitcnt_vm<(NS - 1) * OPS>();
    __builtin_amdgcn_sched_barrier(0);
    auto block = [&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      u32x4 fa[4];
      read_block<q * SLOT + j * 4096>(ad, fa);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const v8i av = (v8i)__builtin_shufflevector(fa[2 * u], fa[2 * u + 1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int i = 0; i < FN; ++i) {
          const v8i wvv = (v8i)__builtin_shufflevector(wr[q][u][i][0], wr[q][u][i][1], 0, 1, 2, 3, 4, 5, 6, 7);
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wvv, av, acc[i][j], 0, 0, 0, 0, 0, 0);
        }
      }
    };
    block(std::integral_constant<int, 0>{});
    if constexpr (FM > 1) block(std::integral_constant<int, 1>{});
    if constexpr (FM > 2) {
      block(std::integral_constant<int, 2>{});
      block(std::integral_constant<int, 3>{});
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // one slot's loads, then the next one's: the counted waits name them by
  // their place in issue order
#pragma unroll
  for (int q = 0; q < NS; ++q) {
    issue(q, s0 + q);
    __builtin_amdgcn_sched_barrier(0);
  }
  fetch_scales();
  for (int s = s0; s < s1; s += NS) {
    slot(std::integral_constant<int, 0>{});
    issue(0, s + NS);
    if constexpr (NS > 1) {
      if (s + 1 >= s1) break;
      slot(std::integral_constant<int, 1>{});
      issue(1, s + 1 + NS);
    }
    if constexpr (NS > 2) {
      if (s + 2 >= s1) break;
      slot(std::integral_constant<int, 2>{});
      issue(2, s + 2 + NS);
    }
    if constexpr (NS > 3) {
      if (s + 3 >= s1) break;
      slot(std::integral_constant<int, 3>{});
      issue(3, s + 3 + NS);
    }
  }
  // every load has landed before the ring becomes the partial sums
  waitcnt_vm<0>();
  __syncthreads();

  // partial sums: block (i, j), quarter q of wave w at ((w * FN + i) * FM +
  // j) * 4 KB + q KB, lane (row r, half h) at slot (r ^ (2 q + h)) + 32 h, so
  // that the eight column groups of one row fall on eight bank groups below
  {
    float4* const red = reinterpret_cast<float4*>(smem) + wave * (FN * FM * 256);
    const int r = lane & 31, h = lane >> 5;
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          red[((i * FM + j) * 4 + q) * 64 + (r ^ (2 * q + h)) + 32 * h] =
              make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
  }
  __syncthreads();
  // sum over the waves of the 4 columns 4 c .. 4 c + 3 of row `row`
  auto total = [&](int row, int c, float* v) __attribute__((always_inline)) {
    const int i = c >> 3, p = c & 7, j = row >> 5, r = row & 31;
    const float4* src = reinterpret_cast<const float4*>(smem) +
                        ((i * FM + j) * 4 + (p >> 1)) * 64 + (r ^ p) + 32 * (p & 1);
    float4 t = src[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      const float4 x = src[w * (FN * FM * 256)];
      t.x += x.x;
      t.y += x.y;
      t.z += x.z;
      t.w += x.w;
    }
    v[0] = t.x;
    v[1] = t.y;
    v[2] = t.z;
    v[3] = t.w;
  };
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int row = row0 + RS * u;
    const int64_t m = m0 + row;
    if (row >= BM || m >= g.M || n >= g.N) continue;
    float v[4];
    total(row, cg, v);
    if constexpr (SILU) {
      // gate columns 16 k .. + 7 and their up columns + 8 give output
      // columns 8 k .. + 7 (N is a multiple of 16: a chunk is never cut)
      float up[4], y[4];
      total(row, cg + 2, up);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float gv = round_bf16((v[t] * sav[u]) * sbv[t]);
        const float uv = round_bf16((up[t] * sav[u]) * sbv[4 + t]);
        const float sg = __builtin_fabsf(gv) <= 80.0f ? silu_in_range(gv) : gv / (1.0f + expf(-gv));
        y[t] = round_bf16(sg) * uv;
      }
      uint16_t* const o = static_cast<uint16_t*>(g.out) + m * g.ldo + (n / 16) * 8 + (n % 16);
      const u32x2 w = {pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
      if ((reinterpret_cast<uintptr_t>(o) & 7) == 0) {
        *reinterpret_cast<u32x2*>(o) = w;
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] = static_cast<uint16_t>(w[t / 2] >> (16 * (t & 1)));
      }
      continue;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = (v[t] * sav[u]) * sbv[t];
    if (out_dtype == FR_DTYPE_FP32) {
      float* const o = static_cast<float*>(g.out) + m * g.ldo + n;
      if (n + 4 <= g.N && g.bias == nullptr && (reinterpret_cast<uintptr_t>(o) & 15) == 0) {
        *reinterpret_cast<f32x4*>(o) = f32x4{v[0], v[1], v[2], v[3]};
        continue;
      }
      store4<FR_DTYPE_FP32>(g.out, g.ldo, m, n, g.N, v, g.bias, nullptr, 0);
      continue;
    }
    if (!wide) {
      if (out_dtype == FR_DTYPE_BF16) store4<FR_DTYPE_BF16>(g.out, g.ldo, m, n, g.N, v, g.bias, g.res, g.ldr);
      else store4<FR_DTYPE_FP16>(g.out, g.ldo, m, n, g.N, v, g.bias, g.res, g.ldr);
      continue;
    }
    const bool bf = out_dtype == FR_DTYPE_BF16;
    u32x2 w = bf ? u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}
                 : u32x2{pack_fp16x2(v[0], v[1]), pack_fp16x2(v[2], v[3])};
    if (g.res) {
      const u32x2 r = resv[u];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (bf)
          w[t] = pack_bf16x2(__uint_as_float(w[t] << 16) + __uint_as_float(r[t] << 16),
                             __uint_as_float(w[t] & 0xFFFF0000u) + __uint_as_float(r[t] & 0xFFFF0000u));
        else
          w[t] = pack_fp16x2(fp16_to_f32(static_cast<uint16_t>(w[t] & 0xFFFFu)) +
                                 fp16_to_f32(static_cast<uint16_t>(r[t] & 0xFFFFu)),
                             fp16_to_f32(static_cast<uint16_t>(w[t] >> 16)) +
                                 fp16_to_f32(static_cast<uint16_t>(r[t] >> 16)));
      }
    }
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(g.out) + m * g.ldo + n) = w;
  }
#endif  // __HIP_DEVICE_COMPILE__
}

template <int FN, int FM, int NW, int NS, bool PRE>
static hipError_t launch_small(const GemmArgs& g, int out_dtype, hipStream_t st) {
  const int64_t nt = ((g.N + 32 * FN - 1) / (32 * FN)) * ((g.M + 32 * FM - 1) / (32 * FM));
  const unsigned grid = static_cast<unsigned>((nt + 7) / 8 * 8);
  if (g.silu)
    hipLaunchKernelGGL((gemm_fp8_small<FN, FM, NW, NS, PRE, true>), dim3(grid), dim3(64 * NW), 0, st, g, out_dtype);
  else
    hipLaunchKernelGGL((gemm_fp8_small<FN, FM, NW, NS, PRE, false>), dim3(grid), dim3(64 * NW), 0, st, g, out_dtype);
  return hipGetLastError();
}

// The rule.  Tile counts decide: each tile shape is taken as long as its
// launch is one round of workgroups, the smallest tile first (most CUs, least
// work per wave).  Measured in one process with the weights rotated through
// HBM, against the large tiles of gemm_fp8_pre.hip (us, prearranged weights):
//   32 x 32, 4 waves    20 x 2048 x 6144   25.0 -> 9.7    128 x 2048 x 2048  10.2 -> 5.1
//   32 x 64, 4 waves    20 x 12288 x 2048  12.9 -> 8.8    (384 32 x 32 tiles: 9.6)
//   64 x 32, 4 waves    128 x 4096 x 2048  10.3 -> 6.2    256 x 2048 x 6144  28.8 -> 12.3
//   64 x 64, 8 waves    512 x 2048 x 6144  28.3 -> 15.1   512 x 2048 x 2048  10.4 -> 7.5
//   128 x 64, 4 waves   1001 x 2048 x 6144 28.4 -> 23.6; at K = 2048 the large tiles are as fast (11.4, 11.6)
// (rows x columns).  Past one round the large tiles win (512 x 4096 x 2048
// 10.8 against 13.4 on 64 x 64), and so they do for wide outputs past 64
// rows (128 x 12288 x 2048 13.9 against 14.8).  [N, K] rows take the same
// route, so that both layouts add in the same order: 12.4 -> 6.1 .. 10.1 at
// K = 2048, 33.9 -> 14.1 .. 23.5 at 6144.
enum class Small { kNone, k32x32, k32x64, k64x32, k64x64, k128x64 };

static Small small_choice(const GemmArgs& g) {
  const int64_t cus = num_cus();
  auto tiles = [&](int64_t bm, int64_t bn) { return ((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn); };
  if (tiles(32, 32) <= cus) return Small::k32x32;
  if (g.M <= 32 && tiles(32, 64) <= 2 * cus) return Small::k32x64;
  if (tiles(64, 32) <= cus) return Small::k64x32;
  if (tiles(64, 64) <= cus) return Small::k64x64;
  if (g.K >= 4096 && tiles(128, 64) <= cus) return Small::k128x64;
  return Small::kNone;
}

template <bool PRE>
static hipError_t dispatch_small(const GemmArgs& g, int out_dtype, hipStream_t st, bool& taken) {
  taken = true;
  switch (small_choice(g)) {
    case Small::k32x32: return launch_small<1, 1, 4, 4, PRE>(g, out_dtype, st);
    case Small::k32x64: return launch_small<2, 1, 4, 2, PRE>(g, out_dtype, st);
    case Small::k64x32: return launch_small<1, 2, 4, 2, PRE>(g, out_dtype, st);
    case Small::k64x64: return launch_small<2, 2, 8, 1, PRE>(g, out_dtype, st);
    case Small::k128x64: return launch_small<2, 4, 4, 1, PRE>(g, out_dtype, st);
    default: taken = false; return hipSuccess;
  }
}

hipError_t gemm_small(const GemmArgs& g, int out_dtype, bool pre, hipStream_t st, bool& taken) {
  return pre ? dispatch_small<true>(g, out_dtype, st, taken) : dispatch_small<false>(g, out_dtype, st, taken);
}

}  // namespace fr

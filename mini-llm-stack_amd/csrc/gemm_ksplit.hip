// Weight-only INT8 / INT4 GEMMs whose output tiles would not fill the GPU, or whose K is no
// multiple of 64: LDS-tiled MFMA tiles of 64 to 256 rows, the reduction axis split over
// blocks, the fp32 partial products summed by a second kernel.
//
// The dense engine (gemm_mfma16.hip) gives every block all of K. A prompt chunk of 333 rows
// through a 11008 -> 4096 projection is then 64 blocks of 256 x 128 (or 176 of 32 x 256, a
// wavefront a SIMD) that each walk 172 stages of 64 k. Here the same tiles are cut into S
// ranges of K, so that about two rounds of 256 blocks share the walk.
//
// Measured (bf16 x, K-split against the kernel that took the shape before): INT4 g128 333 x
// 4096 x 11008 300 -> 47 us, INT8 170 -> 43; INT8 512 x 4096 x 4096 62 -> 31; INT8 1149 x 1336 x
// 2720 (K % 64 = 32: the register GEMV, 4 rows a pass) 379 -> 24; fp32 x, INT4 g32 200 x 4096 x
// 4096 (fp32 FMAs, 4 rows a pass) 411 -> 51. The prompt shapes stay bound by the widening and
// the LDS operand reads of their stages (0.6 - 0.9 us a stage of 128 - 256 rows, 3 to 4 times
// the MFMA time).
//
// Kernel. Block tile BM x BN x 64 (k), 8 wavefronts (two a SIMD). Schedule of a stage, as the
// engine's 256-row kernels: operand reads from LDS, the next stage's activation loads
// (LDS-direct), the MFMAs with the next stage's weights widened and stored between their
// groups, the weight loads of the stage after that, and a barrier that waits for everything
// but those. INT8 widens to exact integers, row scales apply to the sum; INT4 to exact
// 16 (v - 8); a group's products are scaled by s / 16 from a table of the block's own K range
// and added to the result, then cleared (so an infinite x reaches the outputs of its group's
// sum alone, as in fp32).
//
// Ragged K (a multiple of 32): in the last stage the lanes that hold k >= K load activations
// from past the operand's end, which read as zeros, so whatever finite weight those k see
// adds nothing. The descriptors end with the last row's K-th element.
//
// fp32 activations come as PARTS bf16 rows per row of x in 16 PARTS-row groups (row R of the
// split matrix: part (R / 16) % PARTS of row 16 (R / (16 PARTS)) + R % 16), so that a lane
// holds all parts of one output in PARTS consecutive accumulator tiles.
#include <algorithm>
#include <type_traits>

#include "mfma16.h"

namespace mls {

namespace {

typedef uint32_t lds16_t __attribute__((ext_vector_type(4)));

constexpr uint32_t kOutside = 0x80000000u;  // past every descriptor (they span < 2^31 bytes)

struct KsArgs {
  const void* a;
  const uint8_t* b;
  const void* s;
  void* c;        // direct: output rows; partial: fp32 [S][m_out][ldc]
  int lda, ldb;   // elements of 16-bit x; bytes
  int s_dt, group;
  int64_t ld_sn, ld_sg, ldc, c_sstride;
  int M, N, K, m_out;  // M: rows of a (PARTS rows per output row in groups of 16)
  int m_tiles, n_tiles, tile_gm;
  int splits, unit, units;  // K ranges in units of `unit` k
};

template <int WBITS, typename MT, typename OT, int BM, int BN, int WM, int WN, int PARTS, bool PARTIAL, int GK>
__global__ __launch_bounds__(64 * WM * WN) void ksplit_kernel(const KsArgs p) {
  constexpr bool I4 = WBITS == 4;
  constexpr int BK = 64, NW = WM * WN, NT = 64 * NW;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16;
  static_assert(NW == 8 && WTM % (16 * PARTS) == 0 && WTN % 16 == 0, "wave tiles of whole row groups");
  constexpr int A_INSTR = BM * 8 / 64, PW = (A_INSTR + NW - 1) / NW;  // LDS-direct loads a stage (one: 64 chunks)
  constexpr int B_ROWP = I4 ? 4 : 8;                                  // 8-byte weight pieces a row and stage
  constexpr int B_PT = BN * B_ROWP / NT;
  static_assert(BN * B_ROWP % NT == 0 && B_PT <= 15, "whole pieces per thread");
  constexpr int B_RSTEP = NT / B_ROWP;
  static_assert(B_RSTEP % 8 == 0, "swizzle");

  __shared__ __align__(16) uint4 As[2][BM * 8];
  __shared__ __align__(16) uint4 Bs[2][BN * 8];
  extern __shared__ __align__(16) float cT[];  // INT4: [groups of this range][BN]

  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int tiles = p.m_tiles * p.n_tiles;
  const int sp = L / tiles;
  int nt, mt;
  tile_order(L - sp * tiles, p.m_tiles, p.n_tiles, p.tile_gm, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN;
  const int M = p.M, N = p.N, K = p.K;
  const int k_lo = (int)((int64_t)p.units * sp / p.splits) * p.unit;
  const int k_hi = min((int)((int64_t)p.units * (sp + 1) / p.splits) * p.unit, K);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / WN) * WTM, wn0 = (wave % WN) * WTN;

  const int rows_a = min(BM, M - m0), rows_b = min(BN, N - n0);
  const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const uint8_t*)p.a + (int64_t)m0 * p.lda * 2), (short)0, ((rows_a - 1) * p.lda + K) * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.b + (int64_t)n0 * p.ldb), (short)0, (rows_b - 1) * p.ldb + (I4 ? K / 2 : K), 0x00020000);
  // activation slot s = (i NW + wave) 64 + lane: row s / 8, logical chunk (s % 8) ^ (row & 7),
  // which depends on the lane alone
  const int a_lc = (lane & 7) ^ ((lane >> 3) & 7);
  int a_off[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) a_off[i] = (((i * NW + wave) * 64 + lane) >> 3) * p.lda * 2 + a_lc * 16;
  // piece tid + NT i: row tid / B_ROWP + B_RSTEP i, piece tid % B_ROWP of it
  const int b_row0 = tid / B_ROWP, b_kc = tid % B_ROWP;
  const int b_off0 = b_row0 * p.ldb + b_kc * 8;
  const int b_lds0 = b_row0 * 8 + ((I4 ? 2 * b_kc : b_kc) ^ swz(b_row0));
  const int b_lds1 = b_row0 * 8 + ((2 * b_kc + 1) ^ swz(b_row0));  // INT4: a piece is two chunks

  uint2 rb[B_PT];
  auto load_b = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < B_PT; ++i)
      rb[i] = __builtin_bit_cast(
          uint2, __builtin_amdgcn_raw_buffer_load_b64(rsb, b_off0 + B_RSTEP * i * p.ldb, I4 ? k0 / 2 : k0, 0));
  };
  constexpr int UNITS = I4 ? 2 * B_PT : B_PT;  // 16-byte chunks a thread stores a stage
  auto store_unit = [&](uint4* bs, int u) __attribute__((always_inline)) {
    if constexpr (I4) {
      const int i = u >> 1, h = u & 1;
      const uint32_t x = (h == 0 ? rb[i].x : rb[i].y) ^ 0x88888888u;
      const uint32_t hi = x & 0xF0F0F0F0u;         // byte b: 16 (v - 8) of k = 2b + 1
      const uint32_t lo = (x << 4) & 0xF0F0F0F0u;  // byte b: k = 2b
      bs[(h == 0 ? b_lds0 : b_lds1) + B_RSTEP * 8 * i] = make_uint4(
          pack_exact2<MT>(sbyte_f32<0>(lo), sbyte_f32<0>(hi)), pack_exact2<MT>(sbyte_f32<1>(lo), sbyte_f32<1>(hi)),
          pack_exact2<MT>(sbyte_f32<2>(lo), sbyte_f32<2>(hi)), pack_exact2<MT>(sbyte_f32<3>(lo), sbyte_f32<3>(hi)));
    } else {
      const uint32_t d0 = rb[u].x, d1 = rb[u].y;
      bs[b_lds0 + B_RSTEP * 8 * u] = make_uint4(
          pack_exact2<MT>(sbyte_f32<0>(d0), sbyte_f32<1>(d0)), pack_exact2<MT>(sbyte_f32<2>(d0), sbyte_f32<3>(d0)),
          pack_exact2<MT>(sbyte_f32<0>(d1), sbyte_f32<1>(d1)), pack_exact2<MT>(sbyte_f32<2>(d1), sbyte_f32<3>(d1)));
    }
  };
  auto dma_a = [&](uint4* as, int k0) __attribute__((always_inline)) {
    const bool in = k0 + a_lc * 8 < K;  // (K % 8 == 0: a chunk lies on one side)
#pragma unroll
    for (int i = 0; i < PW; ++i)
      if (A_INSTR % NW == 0 || i * NW + wave < A_INSTR)
        lds_load16(rsa, as + (i * NW + wave) * 64, in ? a_off[i] : (int)kOutside, k0 * 2);
  };

  f32x4 acc[TN][TM], tot[I4 ? TN : 1][I4 ? TM : 1];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (I4) tot[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  const int lr = lane & 15, lk = lane >> 4;
  const int nk = (k_hi - k_lo + BK - 1) / BK;

  // prologue: stage 0 in buffers 0, stage 1's weights in registers; the barrier also publishes
  // the scale table
  dma_a(As[0], k_lo);
  load_b(k_lo);
  if constexpr (I4) {
    // NT / BN threads a row (rows past N repeat row N - 1, whose outputs are not stored)
    constexpr int TPR = NT / BN;
    const int G = (k_hi - k_lo) / p.group, g0 = k_lo / p.group, n = tid / TPR;
    const int64_t r = (int64_t)min(n0 + n, N - 1) * p.ld_sn + (int64_t)g0 * p.ld_sg;
    for (int g = tid % TPR; g < G; g += TPR) {
      cT[g * BN + n] = scale_at(p.s, p.s_dt, r + (int64_t)g * p.ld_sg) * 0.0625f;
    }
  }
#pragma unroll
  for (int u = 0; u < UNITS; ++u) store_unit(Bs[0], u);
  load_b(k_lo + BK);
  __syncthreads();
  int kend_g = p.group, g_idx = 0;  // INT4: where the running group ends (from k_lo), its index
  // one stage; FRESH: a group starts with it (INT4; with groups of 32 one starts at every
  // k-step), so its first MFMAs take a zero accumulator and nothing is cleared. Which stages
  // those are is known at compile time for groups of 32 (GK), 64 and 128 (stages in pairs;
  // ranges are whole groups); larger groups (GK = 0) clear their products instead, as a
  // branch between the two forms keeps the widening from being scheduled beside the MFMAs
  // (2048 x 11008 x 4096, groups of 128: 228 us clearing, 273 us branching).
  auto stage = [&](auto freshc, int kt) __attribute__((always_inline)) {
    constexpr bool FRESH = decltype(freshc)::value;
    const int r = kt & 1;
    // operand reads through an opaque base: otherwise the compiler may keep one address
    // register per tile read live across the loop
    uint32_t abase = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)As[r];
    uint32_t bbase = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)Bs[r];
    asm volatile("" : "+v"(abase), "+v"(bbase));
    const auto* as = reinterpret_cast<const __attribute__((address_space(3))) lds16_t*>(abase);
    const auto* bs = reinterpret_cast<const __attribute__((address_space(3))) lds16_t*>(bbase);
    uint4* as_next = As[r ^ 1];
    uint4* bs_next = Bs[r ^ 1];
    const int k0 = k_lo + kt * BK;
    uint4 aop[2][TM], bop[2][TN];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int ch = ks * 4 + lk;
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const int row = wn0 + i * 16 + lr;
        bop[ks][i] = __builtin_bit_cast(uint4, bs[row * 8 + (ch ^ swz(row))]);
      }
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int row = wm0 + j * 16 + lr;
        aop[ks][j] = __builtin_bit_cast(uint4, as[row * 8 + (ch ^ swz(row))]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    dma_a(as_next, k0 + BK);  // stage kt + 1 (past the range: unused)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      // k-step ks's MFMAs, with half of stage kt + 1's weights widened and stored beside them
      constexpr int U0 = (UNITS + 1) / 2;
      const int nu = ks == 0 ? U0 : UNITS - U0, ub = ks == 0 ? 0 : U0;
      static_assert(TN * TM % U0 == 0 && TN * TM % (UNITS - U0) == 0, "MFMA groups");
      const int per = TN * TM / nu;
#pragma unroll
      for (int gi = 0; gi < nu; ++gi) {
#pragma unroll
        for (int x = gi * per; x < (gi + 1) * per; ++x) {
          const int i = x / TM, j = x % TM;
          if constexpr (I4)
            tot[i][j] = Mfma16<MT>::mma(bop[ks][i], aop[ks][j],
                                        GK == 32 || (FRESH && ks == 0) ? f32x4{0.f, 0.f, 0.f, 0.f} : tot[i][j]);
          else acc[i][j] = Mfma16<MT>::mma(bop[ks][i], aop[ks][j], acc[i][j]);
        }
        store_unit(bs_next, ub + gi);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (I4) {
        const bool ends = GK == 32 ? k0 + 32 * (ks + 1) <= k_hi
                          : GK == 64 ? ks == 1
                          : GK == 128 ? ks == 1 && !FRESH
                                      : ks == 1 && (kt + 1) * BK == kend_g;
        if (ends) {  // group g_idx of the range ends: acc += s_g / 16 * its products
#pragma unroll
          for (int i = 0; i < TN; ++i) {
            const float4 c4 = *reinterpret_cast<const float4*>(&cT[g_idx * BN + wn0 + i * 16 + 4 * lk]);
            const float c[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
            for (int j = 0; j < TM; ++j) {
#pragma unroll
              for (int q = 0; q < 4; ++q) acc[i][j][q] = fmaf(c[q], tot[i][j][q], acc[i][j][q]);
              if constexpr (GK == 0) tot[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
          }
          ++g_idx;
          kend_g += p.group;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    load_b(k0 + 2 * BK);  // stage kt + 2 (past the end: harmless)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    // everything but the weight loads just issued (vector loads complete in order), and the
    // widened-weight stores
    __builtin_amdgcn_s_waitcnt(B_PT | 0x70);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if constexpr (GK == 128) {
    for (int kt = 0; kt < nk; kt += 2) {
      stage(std::true_type{}, kt);
      stage(std::false_type{}, kt + 1);
    }
  } else {
    for (int kt = 0; kt < nk; ++kt) stage(std::integral_constant<bool, GK == 64>{}, kt);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- epilogue: tiles PARTS jo + part hold the parts of output row (m0 + wm0) / PARTS + 16 jo + lr
  OT* c = static_cast<OT*>(p.c) + (PARTIAL ? (int64_t)sp * p.c_sstride : 0);
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int nb = n0 + wn0 + i * 16 + 4 * lk;
    if (nb >= N) continue;
    float sn[4] = {1.f, 1.f, 1.f, 1.f};
    if constexpr (!I4 && !PARTIAL) {
#pragma unroll
      for (int r = 0; r < 4; ++r) sn[r] = scale_at(p.s, p.s_dt, (int64_t)min(nb + r, N - 1) * p.ld_sn);
    }
#pragma unroll
    for (int jo = 0; jo < TM / PARTS; ++jo) {
      const int m = (m0 + wm0) / PARTS + jo * 16 + lr;
      if (m >= p.m_out) continue;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float t = acc[i][jo * PARTS + PARTS - 1][r];  // the smallest part first
#pragma unroll
        for (int part = PARTS - 2; part >= 0; --part)
          t = PARTS == 3 ? fmaf(t, 1.0f / 256.0f, acc[i][jo * PARTS + part][r])  // (part p is stored times 2^8p)
                         : t + acc[i][jo * PARTS + part][r];
        v[r] = t * sn[r];
      }
      OT* dst = c + (int64_t)m * p.ldc + nb;
      if (PARTIAL || (nb + 3 < N && (p.ldc % 4) == 0)) {  // (partial rows are padded to 4 columns)
        store4<OT>(dst, v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (nb + r < N) dst[r] = from_f32<OT>(v[r]);
      }
    }
  }
}

// c[m][n] = s[n] * sum_sp part[sp][m][n] (INT4: no scale), rounded once. One thread per 4
// columns; the partial products are still in the Infinity Cache.
template <typename OT, bool SCALE>
__global__ __launch_bounds__(256) void ksplit_sum_kernel(const float* __restrict__ part, int64_t sstride, int ldp,
                                                         int splits, const void* __restrict__ s, int s_dt,
                                                         OT* __restrict__ c, int64_t ldc, int M, int N) {
  const int q = ldp / 4;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (int64_t)M * q) return;
  const int m = (int)(t / q), n = (int)(t - (int64_t)m * q) * 4;
  const float* src = part + (int64_t)m * ldp + n;
  f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll 4
  for (int sp = 1; sp < splits; ++sp) v += *reinterpret_cast<const f32x4*>(src + sp * sstride);
  if constexpr (SCALE) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] *= scale_at(s, s_dt, min(n + r, N - 1));
  }
  OT* dst = c + (int64_t)m * ldc + n;
  if (n + 3 < N && ((uintptr_t)dst & (4 * sizeof(OT) - 1)) == 0) {
    store4<OT>(dst, v[0], v[1], v[2], v[3]);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) dst[r] = from_f32<OT>(v[r]);
  }
}

template <int WBITS, typename MT, typename OT, int BM, int BN, int WM, int WN, int PARTS, bool PARTIAL, int GK>
int launch_tile(KsArgs a, size_t table, hipStream_t st) {
  a.m_tiles = (int)cdiv(a.M, BM);
  a.n_tiles = (int)cdiv(a.N, BN);
  a.tile_gm = 4;
  auto kern = ksplit_kernel<WBITS, MT, OT, BM, BN, WM, WN, PARTS, PARTIAL, GK>;
  constexpr size_t kMostTable = (size_t)160 * 1024 - (size_t)2 * (BM + BN) * 128;
  if (table > kMostTable) return MLS_ERR_UNSUPPORTED;
  static const hipError_t attr =  // the largest table, once per instantiation
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMostTable);
  if (attr != hipSuccess) return fail(MLS_ERR_HIP, "K-split GEMM: cannot reserve %zu bytes of LDS", kMostTable);
  hipLaunchKernelGGL(kern, dim3((unsigned)((int64_t)a.m_tiles * a.n_tiles * a.splits)), dim3(64 * WM * WN), table, st,
                     a);
  return check_launch("K-split GEMM");
}

template <int WBITS, typename MT, typename OT, int PARTS, int GK>
int launch_shape_g(const KsArgs& a, int bm, int bn, size_t table, bool partial, hipStream_t st) {
#define MLS_KS(BM_, BN_, WM_, WN_)                                                                             \
  if (bm == BM_ && bn == BN_)                                                                                  \
    return partial ? launch_tile<WBITS, MT, float, BM_, BN_, WM_, WN_, PARTS, true, GK>(a, table, st)          \
                   : launch_tile<WBITS, MT, OT, BM_, BN_, WM_, WN_, PARTS, false, GK>(a, table, st)
  if constexpr (PARTS == 3) {
    MLS_KS(48, 128, 1, 8);
    MLS_KS(96, 128, 2, 4);
    MLS_KS(192, 128, 4, 2);
  } else {
    MLS_KS(64, 128, 2, 4);
    MLS_KS(128, 128, 4, 2);
    if constexpr (PARTS == 1) MLS_KS(192, 128, 4, 2);
    MLS_KS(256, 128, 4, 2);
    if constexpr (WBITS == 8) MLS_KS(256, 192, 2, 4);
    if constexpr (WBITS == 8) MLS_KS(256, 256, 2, 4);
  }
#undef MLS_KS
  return MLS_ERR_UNSUPPORTED;
}

template <int WBITS, typename MT, typename OT, int PARTS>
int launch_shape(const KsArgs& a, int bm, int bn, size_t table, bool partial, hipStream_t st) {
  if constexpr (WBITS == 4) {
    if constexpr (PARTS != 2)  // (two parts: groups are multiples of 64)
      if (a.group == 32) return launch_shape_g<WBITS, MT, OT, PARTS, 32>(a, bm, bn, table, partial, st);
    if (a.group == 64) return launch_shape_g<WBITS, MT, OT, PARTS, 64>(a, bm, bn, table, partial, st);
    if (a.group == 128) return launch_shape_g<WBITS, MT, OT, PARTS, 128>(a, bm, bn, table, partial, st);
    if (a.group % 64 != 0) return MLS_ERR_UNSUPPORTED;
  }
  return launch_shape_g<WBITS, MT, OT, PARTS, 0>(a, bm, bn, table, partial, st);
}

// Most bytes of partial products, and of x as three parts, that a launch works on (the Infinity
// Cache holds 256 MiB; the largest use at 2048 rows and 11008 columns is 258).
constexpr int64_t kMostBytes = (int64_t)384 << 20;

struct KsPlan {
  int bm = 0, bn = 0, splits = 0, parts = 1;  // bm 0: not taken
  int unit = 64, units = 0;
  int64_t rows = 0;  // rows of x a launch; more take several, one after another in one workspace
};

// k that a range is a multiple of: whole stages and whole groups (32 or multiples of 64)
int range_unit(int wbits, int group) { return wbits == 4 && group > 64 ? group : 64; }

KsPlan ks_plan(int wbits, int64_t M, int64_t N, int64_t K, int a_dt, int group);

int64_t rows_of(const KsPlan& p, int64_t M) { return p.parts == 1 ? M : cdiv(M, 16) * 16 * p.parts; }
int64_t up256(int64_t v) { return cdiv(v, 256) * 256; }
int64_t ld_part(int64_t N) { return cdiv(N, 4) * 4; }
int64_t ws_x(const KsPlan& p, int64_t M, int64_t K) { return p.parts == 1 ? 0 : up256(rows_of(p, M) * K * 2); }
int64_t ws_part(int splits, int64_t M, int64_t N) { return splits > 1 ? splits * M * ld_part(N) * 4 : 0; }
int64_t ws_need(const KsPlan& p, int64_t M, int64_t N, int64_t K) {
  const int64_t m = M < p.rows ? M : p.rows;
  return ws_x(p, m, K) + ws_part(p.splits, m, N);
}

int run_rows(int wbits, const KsPlan& pl, const WqArgs& w, uint8_t* ws) {
  KsArgs a{};
  a.a = w.a; a.lda = (int)w.lda;
  a.b = w.w; a.ldb = (int)w.ldw;
  a.s = w.s; a.s_dt = w.s_dt; a.ld_sn = w.ld_sn; a.ld_sg = w.ld_sg; a.group = wbits == 4 ? w.group : 64;
  a.M = (int)rows_of(pl, w.M); a.N = (int)w.N; a.K = (int)w.K; a.m_out = (int)w.M;
  a.splits = pl.splits; a.unit = pl.unit; a.units = pl.units;
  const bool partial = pl.splits > 1;
  float* part = reinterpret_cast<float*>(ws + ws_x(pl, w.M, w.K));
  a.c = partial ? (void*)part : w.c;
  a.ldc = partial ? ld_part(w.N) : w.ldc;
  a.c_sstride = w.M * ld_part(w.N);
  if (pl.parts > 1) {
    const int rc = launch_split_parts(static_cast<const float*>(w.a), w.lda, w.M, w.K, pl.parts, ws, w.stream);
    if (rc != MLS_OK) return rc;
    a.a = ws;
    a.lda = (int)w.K;
  }
  const size_t table = wbits == 4 ? (size_t)cdiv(pl.units, pl.splits) * (pl.unit / w.group) * pl.bn * 4 : 0;
  int rc;
  if (w.a_dt == MLS_F32) {
    if (pl.parts == 3)
      rc = wbits == 4 ? launch_shape<4, __bf16, float, 3>(a, pl.bm, pl.bn, table, partial, w.stream)
                      : launch_shape<8, __bf16, float, 3>(a, pl.bm, pl.bn, table, partial, w.stream);
    else
      rc = wbits == 4 ? launch_shape<4, __bf16, float, 2>(a, pl.bm, pl.bn, table, partial, w.stream)
                      : launch_shape<8, __bf16, float, 2>(a, pl.bm, pl.bn, table, partial, w.stream);
  } else if (w.a_dt == MLS_BF16) {
    rc = wbits == 4 ? launch_shape<4, __bf16, __bf16, 1>(a, pl.bm, pl.bn, table, partial, w.stream)
                    : launch_shape<8, __bf16, __bf16, 1>(a, pl.bm, pl.bn, table, partial, w.stream);
  } else {
    rc = wbits == 4 ? launch_shape<4, _Float16, _Float16, 1>(a, pl.bm, pl.bn, table, partial, w.stream)
                    : launch_shape<8, _Float16, _Float16, 1>(a, pl.bm, pl.bn, table, partial, w.stream);
  }
  if (rc != MLS_OK || !partial) return rc;
  const int ldp = (int)ld_part(w.N);
  const dim3 grid((unsigned)cdiv(w.M * (ldp / 4), 256));
#define MLS_KSUM(OT_, SC_)                                                                                     \
  hipLaunchKernelGGL((ksplit_sum_kernel<OT_, SC_>), grid, dim3(256), 0, w.stream, part, a.c_sstride, ldp, pl.splits, \
                     w.s, w.s_dt, (OT_*)w.c, w.ldc, (int)w.M, (int)w.N)
  if (wbits == 8) {
    if (w.a_dt == MLS_F32) MLS_KSUM(float, true);
    else if (w.a_dt == MLS_BF16) MLS_KSUM(__bf16, true);
    else MLS_KSUM(_Float16, true);
  } else {
    if (w.a_dt == MLS_F32) MLS_KSUM(float, false);
    else if (w.a_dt == MLS_BF16) MLS_KSUM(__bf16, false);
    else MLS_KSUM(_Float16, false);
  }
#undef MLS_KSUM
  return check_launch("K-split sum");
}

int run_plan(int wbits, const KsPlan& pl, const WqArgs& w, uint8_t* ws) {
  const int64_t sz = dt_size(w.a_dt);
  for (int64_t m = 0; m < w.M; m += pl.rows) {
    WqArgs c = w;
    c.a = static_cast<const uint8_t*>(w.a) + m * w.lda * sz;
    c.c = static_cast<uint8_t*>(w.c) + m * w.ldc * sz;
    c.M = std::min(pl.rows, w.M - m);
    const int rc = run_rows(wbits, pl, c, ws);
    if (rc != MLS_OK) return rc;  // (UNSUPPORTED comes from a tile's limits, so from the first rows)
  }
  return MLS_OK;
}

// What the kernels assume of pointers and strides (the sizes are the plan's).
bool layout_ok(int wbits, const WqArgs& w) {
  if (!w.a || !w.w || !w.s || !w.c) return false;  // (the general entry points say what is wrong)
  if (w.a_dt != MLS_F32 && (!aligned(w.a, 16) || w.lda % 8 != 0 || w.lda * 2 * 256 >= (1ll << 31))) return false;
  if (!aligned(w.w, 8) || w.ldw % 8 != 0 || w.ldw * 256 >= (1ll << 31)) return false;
  if (w.lda < w.K || w.ldw < (wbits == 4 ? w.K / 2 : w.K) || w.ldc < w.N || w.ld_sn < 0 || w.ld_sg < 0) return false;
  if (w.s_dt != MLS_F32 && w.s_dt != MLS_F16) return false;
  return aligned(w.c, 16);
}

// Time model of a tile shape, fitted to 7,600 timed launches (INT4 / INT8, M = 1 .. 2048,
// ten (N, K) from 512 x 512 to 4096 x 11008, every split; log error 3 to 10% rms, and the
// choice it makes is on average 2% off the fastest tile and split, 17% at worst). us:
//   base + rounds * (stages of a block * t1 + edge), a CU holding `share` blocks at t2 a stage,
//   + sum + per_mb * (MB of partial products) when K is split.
// INT4 stages take 1.12 times as long with groups of 64 and 1.42 times with groups of 32 (a
// group end is an FMA an accumulator).
struct TileCost {
  int bits, bm, bn, share;
  float t1, t2, edge, base, sum, per_mb;
};
constexpr TileCost kTiles[] = {
    {4, 48, 128, 2, 0.590f, 0.911f, 0.00f, 6.15f, 2.35f, 0.399f},
    {4, 64, 128, 2, 0.474f, 0.791f, 0.00f, 4.59f, 2.01f, 0.464f},
    {4, 96, 128, 2, 0.746f, 1.288f, 0.00f, 6.55f, 1.45f, 0.459f},
    {4, 128, 128, 1, 0.618f, 0.000f, 0.41f, 5.86f, 2.12f, 0.340f},
    {4, 192, 128, 1, 0.768f, 0.000f, 1.61f, 5.30f, 2.19f, 0.324f},
    {4, 256, 128, 1, 0.938f, 0.000f, 0.32f, 8.24f, 2.09f, 0.307f},
    {8, 48, 128, 1, 0.318f, 0.000f, 0.16f, 9.93f, 0.00f, 0.250f},
    {8, 64, 128, 2, 0.419f, 0.673f, 0.00f, 6.19f, 1.06f, 0.463f},
    {8, 96, 128, 2, 0.643f, 0.997f, 0.25f, 7.48f, 0.00f, 0.647f},
    {8, 128, 128, 1, 0.506f, 0.000f, 0.00f, 9.09f, 0.10f, 0.334f},
    {8, 192, 128, 1, 0.599f, 0.000f, 0.00f, 9.94f, 0.00f, 0.317f},
    {8, 256, 128, 1, 0.810f, 0.000f, 1.12f, 8.92f, 1.24f, 0.292f},
    {8, 256, 192, 1, 1.123f, 0.000f, 1.86f, 10.64f, 0.41f, 0.280f},
    {8, 256, 256, 1, 1.387f, 0.000f, 3.76f, 10.61f, 0.40f, 0.252f},
};

// The fastest tile and split by the model with at most `most` bytes of partial products, its time in
// us; bm = 0 when nothing fits.
KsPlan best_tile(int wbits, int64_t M, int64_t N, int64_t K, int group, int parts, int64_t most, float* us) {
  static constexpr int kSplits[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32};
  KsPlan best;
  best.parts = parts;
  best.unit = range_unit(wbits, group);
  best.units = (int)cdiv(K, best.unit);
  best.rows = M;
  *us = 1e30f;
  const int64_t rows = rows_of(best, M);
  const float slow = wbits == 8 || group >= 128 ? 1.0f : group == 64 ? 1.12f : 1.42f;
  for (const TileCost& t : kTiles) {
    const bool three = t.bm == 48 || t.bm == 96 || (t.bm == 192 && t.bn == 128);
    if (t.bits != wbits || (parts == 3 ? !three : t.bm % 64 != 0 || (parts == 2 && t.bm == 192))) continue;
    if (t.bm > 64 && t.bm != 96 && rows <= t.bm / 2) continue;  // mostly rows past M
    const int64_t tiles = cdiv(rows, t.bm) * cdiv(N, t.bn);
    if (tiles > 0xFFFFFF) continue;
    bool any = false;
    for (int s : kSplits) {
      if (s > best.units) break;
      if (wbits == 4 && cdiv(best.units, s) * (best.unit / group) * t.bn * 4 > 160 * 1024 - 256 * (t.bm + t.bn)) continue;
      if (s > 1 && ((any && tiles * s > 800) || ws_part(s, M, N) > most)) break;
      any = true;
      const float stages = (float)(cdiv(best.units, s) * (best.unit / 64)) * slow;
      const float r1 = stages * t.t1 + t.edge, r2 = stages * t.t2 + t.edge;
      const int64_t q = cdiv(tiles * s, 256);  // blocks of the fullest CU
      float c = t.base + (t.share == 1 ? (float)q * r1 : (float)(q / 2) * r2 + (q & 1 ? r1 : 0.0f));
      if (s > 1) c += t.sum + t.per_mb * (float)s * (float)M * (float)N * 4e-6f;
      if (c < *us) {
        *us = c;
        best.bm = t.bm;
        best.bn = t.bn;
        best.splits = s;
      }
    }
  }
  return best;
}

// What the general entry points would take for a shape, in us (0: always theirs; infinity: the kernel
// with one thread an output). *fitted: by the engine's model, which was fitted together with the
// K-split kernels' times (and with the pass that splits fp32 x); the others are off by a tenth or so.
float general_us(int wbits, int64_t M, int64_t N, int64_t K, int a_dt, int group, bool split, bool* fitted) {
  *fitted = true;
  const bool f32 = a_dt == MLS_F32;
  const int ks = wbits == 4 && group % 128 == 0 ? 128 : 64;  // k a step of the skinny and medium kernels
  const bool stepped = K % ks == 0 && (wbits == 8 || group % 64 == 0);
  if (M > 16 && (f32 ? split : stepped)) {
    const int64_t m = split ? split_rows(M) : M, bm = split && wbits == 8 && m >= 256 ? 256 : 128;
    if ((split ? m <= 512 : M <= 256) && cdiv(m, bm) * cdiv(N, 256) < 128)
      return *fitted = false, small_estimate_us(wbits, m, N, K, group, f32 ? 4 : 2, split);
    return engine_estimate_us(wbits, m, N, K, group, split);
  }
  if (M > 16 && !f32 && K % 64 == 0) return engine_estimate_us(wbits, M, N, K, group, false);
  *fitted = false;
  if (M > 1 && M <= 16 && stepped) return 0.0f;     // the skinny MFMA kernel
  // the register GEMVs: a pass over the weights for every `rows` rows of x (their registers
  // hold rows * K / 64 values a lane); measured 0.2 us a pass plus 0.15
  // (16-bit x) or 0.28 (fp32) a million weights
  const int kc = wbits == 4 ? 32 : 16;
  int64_t cpl = 1;
  while (cpl * 64 * kc < K) cpl *= 2;
  if (M == 1 && K * dt_size(a_dt) <= 32768 && (!f32 || wbits == 4)) return 0.0f;
  const int64_t rows = 128 / (cpl * (f32 ? kc : kc / 2));
  if (cpl > 16 || rows < 1) return 1e30f;
  return 3.0f + (float)cdiv(M, rows < 4 ? rows : 4) * (0.2f + (float)N * (float)K * 1e-6f * (f32 ? 0.28f : 0.15f));
}

// The plan for a shape, from its sizes and types alone (the workspace query and the call must
// agree); bm = 0 leaves it to the general entry points.
//
// fp32 activations: two bf16 parts where the general path takes two (K % 64 == 0, INT4 groups
// a multiple of 64, M >= 2), and three, which hold x exactly, where it multiplies in fp32
// (error against 64 bits at 200 x 4096 x 4096, groups of 32: 3.6e-7 in fp32, 1.5e-7 here).
KsPlan ks_plan(int wbits, int64_t M, int64_t N, int64_t K, int a_dt, int group) {
  if (K % 32 != 0 || K < 64 || M > (1 << 24) || N > (1 << 28) || K * 512 >= (1ll << 31)) return {};
  if (wbits == 4 && ((group != 32 && group % 64 != 0) || group < 32 || group > (1 << 20) || K % group != 0)) return {};
  const bool f32 = a_dt == MLS_F32;
  const bool split = f32 && M > 1 && K % 64 == 0 && (wbits == 8 || group % 64 == 0);
  bool fitted;
  const float general = general_us(wbits, M, N, K, a_dt, group, split, &fitted);
  if (general == 0.0f) return {};
  float us;
  const int parts = !f32 ? 1 : split ? 2 : 3;
  KsPlan p = best_tile(wbits, M, N, K, group, parts, INT64_MAX, &us);
  if (p.bm == 0) return {};
  auto over = [&](const KsPlan& q) {
    return ws_part(q.splits, q.rows, N) > kMostBytes || (parts == 3 && ws_x(q, q.rows, K) > kMostBytes);
  };
  if (over(p)) {
    // Past the workspace's bound (groups of 32 at K > 7424: a tile's scale table does not hold all of
    // K, so K is split however many tiles there are; fp32 x in three parts: 6 bytes a value): other
    // tiles, or the rows in several launches, whichever the model has faster.
    p = {};
    us = 1e30f;
    for (int64_t rows = M, next = 8192; rows >= 256; rows = next, next /= 2) {
      if (rows > M) continue;
      float t;
      const KsPlan q = best_tile(wbits, rows, N, K, group, parts, kMostBytes, &t);
      t *= (float)cdiv(M, rows);
      if (q.bm == 0 || over(q) || t >= us) continue;
      p = q;
      us = t;
    }
    if (p.bm == 0) return {};
  }
  if (fitted ? us + (f32 ? split_estimate_us(M, K) : 0.0f) >= general : us >= 0.92f * general) return {};
  // whole 192- or 256-column tiles without a split are the engine's own
  if (p.splits == 1 && p.bn > 128 && K % 64 == 0) return {};
  return p;
}

int run_ext(int wbits, const WqArgs& w, int c_dt, void* ws, int64_t ws_bytes, bool* taken) {
  *taken = false;
  if (c_dt != w.a_dt || !is_float_dt(w.a_dt) || w.M < 1 || w.N < 1 || w.K < 1 || !layout_ok(wbits, w)) return MLS_OK;
  const KsPlan pl = ks_plan(wbits, w.M, w.N, w.K, w.a_dt, w.group);
  if (pl.bm == 0) return MLS_OK;
  // two parts of fp32 x only where the general path takes two (split_ok); else it multiplies in fp32
  if (pl.parts == 2 && (!aligned(w.w, 16) || w.ldw % 16 != 0)) return MLS_OK;
  const int64_t need = ws_need(pl, w.M, w.N, w.K);
  if (need && (!ws || ws_bytes < need || !aligned(ws, 256))) return MLS_OK;
  *taken = true;
  return run_plan(wbits, pl, w, static_cast<uint8_t*>(ws));
}

}  // namespace

}  // namespace mls

using namespace mls;

extern "C" int64_t mlsx_wq_workspace(int wbits, int64_t M, int64_t N, int64_t K, int a_dt, int group) {
  if ((wbits != 4 && wbits != 8) || M <= 0 || N <= 0 || K <= 0 || !is_float_dt(a_dt)) return 0;
  const int64_t base = mls_wq_gemm_workspace(wbits, M, N, K, a_dt, group);
  const KsPlan pl = ks_plan(wbits, M, N, K, a_dt, group);
  const int64_t need = pl.bm ? ws_need(pl, M, N, K) : 0;
  return need > base ? need : base;
}

extern "C" int mlsx_wq_ksplit(int wbits, int64_t M, int64_t N, int64_t K, int a_dt, int group) {
  if ((wbits != 4 && wbits != 8) || M <= 0 || N <= 0 || K <= 0 || !is_float_dt(a_dt)) return 0;
  const KsPlan pl = ks_plan(wbits, M, N, K, a_dt, group);
  return pl.bm ? pl.splits : 0;
}

extern "C" int mlsx_int8_gemm(const void* a, int a_dt, int64_t lda, const int8_t* w, int64_t ldw, const void* s,
                              int s_dt, void* c, int c_dt, int64_t ldc, int64_t M, int64_t N, int64_t K,
                              void* workspace, int64_t ws_bytes, mls_stream_t stream) {
  const WqArgs p{a, a_dt, lda, reinterpret_cast<const uint8_t*>(w), ldw, s, s_dt, 1, 0, 0,
                 c, ldc, M, N, K, (hipStream_t)stream};
  bool taken;
  const int rc = run_ext(8, p, c_dt, workspace, ws_bytes, &taken);
  if (taken && rc != MLS_ERR_UNSUPPORTED) return rc;
  return mls_int8_gemm_ws(a, a_dt, lda, w, ldw, s, s_dt, c, c_dt, ldc, M, N, K, workspace, ws_bytes, stream);
}

extern "C" int mlsx_int4_gemm(const void* a, int a_dt, int64_t lda, const uint8_t* w, int64_t ldw, const void* s,
                              int s_dt, int64_t ld_sn, int64_t ld_sg, int group, void* c, int c_dt, int64_t ldc,
                              int64_t M, int64_t N, int64_t K, void* workspace, int64_t ws_bytes,
                              mls_stream_t stream) {
  const WqArgs p{a, a_dt, lda, w, ldw, s, s_dt, ld_sn, ld_sg, group, c, ldc, M, N, K, (hipStream_t)stream};
  bool taken;
  const int rc = run_ext(4, p, c_dt, workspace, ws_bytes, &taken);
  if (taken && rc != MLS_ERR_UNSUPPORTED) return rc;
  return mls_int4_gemm_ws(a, a_dt, lda, w, ldw, s, s_dt, ld_sn, ld_sg, group, c, c_dt, ldc, M, N, K, workspace,
                          ws_bytes, stream);
}

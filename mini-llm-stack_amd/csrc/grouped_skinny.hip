// INT4 grouped GEMMs of a routed MoE layer with few rows an expert (a decode batch): every
// expert's weights stream once, straight into MFMA operand layout.
//
// The chunk kernel (gemm_grouped.hip) widens each weight into LDS for a row chunk of at least
// 64 rows: two VALU instructions a weight, an LDS write and several LDS reads, whatever the
// segment holds. With 2 to 4 rows an expert it is bound by that work: 16 tokens, top-2 of 8
// experts (4096 -> 14336, g128), gate/up 201 us (2.4 TB/s of weights) and down 98; this kernel
// 120 us (4.0 TB/s) and 55 (4.4).
//
// Here a wavefront owns R tiles of 16 weight rows and MT tiles of 16 rows of x (segments longer
// than 16 MT rows take further passes over the block's weights, which are then in the Infinity
// Cache). A step is 128 k: a lane's 16 weight bytes and its x pieces come straight into
// registers, two steps in flight; nibbles are OR-ed into the mantissa of bf16 128 / fp16 1024
// (one v_and_or for two weights, x permuted alike) and the offset is removed with x's sums over
// the step, from one more MFMA against ones, as in the medium GEMM (gemm_small.hip); group
// scales apply to each step's fp32 sums from a table of the block's range in LDS (groups of 64:
// the two halves of a step are multiplied apart, with the other half of x zeroed; steps of 64 k
// with 8-byte loads ran at the chunk kernel's speed). The WK wavefronts of a block share its
// tiles and take the steps in turn, so that together they read whole cache lines of a weight
// row (each its own contiguous range: gate/up 150 us at 16 tokens); non-temporal loads measured
// slower (128 / 74 us). Their sums meet in LDS. Rows of x past the segment load from past the
// operand (zeros, no traffic).
//
// Gate/up: half of a wavefront's tiles are gate rows and half the same rows of up, so both
// products of one output sit in one lane and silu(g) * u needs no exchange.
#include <type_traits>

#include "mfma16.h"

namespace mls {

namespace {

template <typename AT> struct Nib4;
template <> struct Nib4<__bf16> {
  static constexpr uint32_t MAGIC = 0x43004300u, ONE2 = 0x3F803F80u;  // bf16 (128, 128), (1, 1)
  static constexpr float OFF = 136.0f;                                // 128 + 8
};
template <> struct Nib4<_Float16> {
  static constexpr uint32_t MAGIC = 0x64006400u, ONE2 = 0x3C003C00u;  // fp16 (1024, 1024), (1, 1)
  static constexpr float OFF = 1032.0f;
};

constexpr uint32_t kOutside = 0x80000000u;  // past every descriptor (they span < 2^31 bytes)

__device__ __forceinline__ uint4 perm_x4(const uint4& v) {  // k order 0..7 -> 0,4,1,5,2,6,3,7
  return make_uint4(__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
                    __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u));
}
__device__ __forceinline__ uint32_t and_or4(uint32_t a, uint32_t m, uint32_t c) { return (a & m) | c; }

// p.n_tiles: blocks a matrix; p.ksplit: K ranges whose products go to separate fp32 outputs
// (PARTIAL), else 1. NG: groups in a step of 128 k (2 for groups of 64, whose halves of a step
// are multiplied apart, x of the other half zeroed).
template <typename AT, int R, int MT, int WK, bool GU, bool PARTIAL, int NG>
__global__ __launch_bounds__(64 * WK) void grouped_skinny_kernel(const Mfma16Params p) {
  using MM = Mfma16<AT>;
  static_assert(R * 16 == 64, "scale table rows");
  constexpr int KS = 128, XP = 4;
  constexpr int RO = GU ? R / 2 : R;  // output tiles
  constexpr int TS = 68;              // floats a group of the scale table (64 rows, padded for the banks)
  extern __shared__ __align__(16) uint8_t smem[];  // [WK][R][MT][64] sums, then [groups of the range][TS] scales

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  int L = blockIdx.x;
  const int per = p.n_tiles * p.ksplit, e = L / per;
  L -= e * per;
  const int sp = L / p.n_tiles, n0 = (L - sp * p.n_tiles) * 16 * RO;
  int lo, hi;
  seg_rows(p, e, lo, hi);
  if (lo >= hi) return;
  const int N = p.N;
  // the range's steps go round the wavefronts, so that together they read whole cache lines
  const int steps = p.K / KS / p.ksplit, s_lo = steps * sp, s_hi = s_lo + steps;

  const uint8_t* wmat = p.b + (int64_t)e * p.b_estride;
  const __amdgpu_buffer_rsrc_t rsw =
      __builtin_amdgcn_make_buffer_rsrc((void*)wmat, (short)0, (int)((N - 1) * p.ldb + p.K / 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsu = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(GU ? p.b2 + (int64_t)e * p.b_estride : wmat), (short)0, (int)((N - 1) * p.ldb + p.K / 2), 0x00020000);
  const int x_rows = p.a_rows ? p.a_src_rows : p.M;
  const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.a, (short)0, (int)(((x_rows - 1) * p.lda + p.K) * 2), 0x00020000);

  // tile t < RO: weight rows n0 + 16 t ..; gate/up: tile RO + t the same rows of up
  int wo[R];
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int n = n0 + 16 * (t % RO) + r16;
    wo[t] = n < N ? n * (int)p.ldb + 16 * q : (int)kOutside;
  }

  struct Slot {
    uint4 w[R];
    uint4 x[MT][XP];
  };
  int xo[MT];
  auto rows_at = [&](int m0) __attribute__((always_inline)) {
#pragma unroll
    for (int tm = 0; tm < MT; ++tm) {
      const int m = m0 + 16 * tm + r16;
      int row = -1;
      if (m < hi) row = p.a_rows ? p.a_rows[m] : m;
      xo[tm] = row >= 0 && row < x_rows ? row * (int)p.lda * 2 + 64 * q : (int)kOutside;
    }
  };
  auto load = [&](Slot& sl, int st) __attribute__((always_inline)) {
    const int k = min(st, s_hi - 1);  // (a step past the range repeats the last one, unused)
#pragma unroll
    for (int t = 0; t < R; ++t)
      sl.w[t] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(t < RO ? rsw : rsu, wo[t], k * 64, 0));
#pragma unroll
    for (int tm = 0; tm < MT; ++tm)
#pragma unroll
      for (int h = 0; h < XP; ++h)
        sl.x[tm][h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsa, xo[tm] + 16 * h, k * KS * 2, 0));
  };
  Slot a, b;
  rows_at(lo);
  load(a, s_lo + wave);
  load(b, s_lo + wave + WK);

  // the block's scales as fp32 [group of the range][row of its 64]: 16 groups x 4 rows a
  // wavefront and instruction
  float* sc_lds = reinterpret_cast<float*>(smem + WK * R * MT * 1024);
  const int g_lo = s_lo * KS / p.group, groups = (s_hi * KS - 1) / p.group + 1 - g_lo;
  for (int r = wave * 4 + (lane >> 4); r < 64; r += 4 * WK) {
    const int t = r >> 4, n = min(n0 + 16 * (t % RO) + (r & 15), N - 1);
    const void* smat = GU && t >= RO ? p.s2 : p.s;
    const int64_t base = (int64_t)e * p.s_estride + (int64_t)n * p.ld_sn + (int64_t)g_lo * p.ld_sg;
    for (int g = lane & 15; g < groups; g += 16) sc_lds[g * TS + r] = scale_at(smat, p.s_dt, base + (int64_t)g * p.ld_sg);
  }
  __syncthreads();

  uint32_t nmask = 0x000F000Fu, magic = Nib4<AT>::MAGIC;
  asm volatile("" : "+v"(nmask), "+v"(magic));
  const uint4 ones = make_uint4(Nib4<AT>::ONE2, Nib4<AT>::ONE2, Nib4<AT>::ONE2, Nib4<AT>::ONE2);
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int m0 = lo; m0 < hi; m0 += 16 * MT) {
    if (m0 != lo) {
      rows_at(m0);
      load(a, s_lo + wave);
      load(b, s_lo + wave + WK);
    }
    f32x4 acc[R][MT];
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
      for (int tm = 0; tm < MT; ++tm) acc[t][tm] = zero;
    auto compute = [&](const Slot& sl, int st) __attribute__((always_inline)) {
      uint4 xpm[NG][MT][XP];
      f32x4 xs[NG][MT];
#pragma unroll
      for (int tm = 0; tm < MT; ++tm)
#pragma unroll
        for (int h = 0; h < NG; ++h) {
          xs[h][tm] = zero;
#pragma unroll
          for (int j = 0; j < XP; ++j) {
            uint4 v = perm_x4(sl.x[tm][j]);
            if constexpr (NG == 2) {
              const bool mine = (q >> 1) == h;  // lane groups 0, 1 hold the first 64 k, 2, 3 the others
              v = mine ? v : make_uint4(0u, 0u, 0u, 0u);
            }
            xpm[h][tm][j] = v;
            xs[h][tm] = MM::mma(ones, v, xs[h][tm]);
          }
        }
      const float* sg = sc_lds + (st * KS / p.group - g_lo) * TS + 4 * q;
#pragma unroll
      for (int t = 0; t < R; ++t) {
        const uint32_t d[4] = {sl.w[t].x, sl.w[t].y, sl.w[t].z, sl.w[t].w};
        f32x4 pp[NG][MT];
#pragma unroll
        for (int h = 0; h < NG; ++h)
#pragma unroll
          for (int tm = 0; tm < MT; ++tm) pp[h][tm] = zero;
#pragma unroll
        for (int j = 0; j < XP; ++j) {
          const uint4 wop = make_uint4(and_or4(d[j], nmask, magic), and_or4(d[j] >> 4, nmask, magic),
                                       and_or4(d[j] >> 8, nmask, magic), and_or4(d[j] >> 12, nmask, magic));
#pragma unroll
          for (int h = 0; h < NG; ++h)
#pragma unroll
            for (int tm = 0; tm < MT; ++tm) pp[h][tm] = MM::mma(wop, xpm[h][tm][j], pp[h][tm]);
        }
#pragma unroll
        for (int h = 0; h < NG; ++h) {
          const f32x4 sc = *reinterpret_cast<const f32x4*>(sg + h * TS + 16 * t);
#pragma unroll
          for (int tm = 0; tm < MT; ++tm)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              acc[t][tm][i] = fmaf(sc[i], fmaf(-Nib4<AT>::OFF, xs[h][tm][i], pp[h][tm][i]), acc[t][tm][i]);
        }
      }
    };
    for (int st = s_lo + wave; st < s_hi; st += 2 * WK) {
      compute(a, st);
      load(a, st + 2 * WK);
      if (st + WK < s_hi) {
        compute(b, st + WK);
        load(b, st + 3 * WK);
      }
    }

    // the WK partial sums meet in LDS
    f32x4* red = reinterpret_cast<f32x4*>(smem);
    if (m0 != lo) __syncthreads();  // (the last pass's sums have been read)
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
      for (int tm = 0; tm < MT; ++tm) red[((wave * R + t) * MT + tm) * 64 + lane] = acc[t][tm];
    __syncthreads();
    for (int slot = threadIdx.x; slot < RO * MT * 64; slot += 64 * WK) {
      const int l = slot & 63, tm = (slot >> 6) % MT, t = (slot >> 6) / MT;
      f32x4 v = red[(t * MT + tm) * 64 + l];
#pragma unroll
      for (int ww = 1; ww < WK; ++ww) v += red[((ww * R + t) * MT + tm) * 64 + l];
      if constexpr (GU) {
        f32x4 u = red[((RO + t) * MT + tm) * 64 + l];
#pragma unroll
        for (int ww = 1; ww < WK; ++ww) u += red[((ww * R + RO + t) * MT + tm) * 64 + l];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.0f + __expf(-v[i])) * u[i];
      }
      const int m = m0 + 16 * tm + (l & 15), nb = n0 + 16 * t + 4 * (l >> 4);
      if (m >= hi || nb >= N) continue;
      using OT = std::conditional_t<PARTIAL, float, AT>;
      OT* dst = static_cast<OT*>(p.c) + (PARTIAL ? (int64_t)sp * p.c_sstride : 0) + (int64_t)m * p.ldc + nb;
      if (nb + 3 < N && ((uintptr_t)dst & (4 * sizeof(OT) - 1)) == 0) {
        store4<OT>(dst, v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nb + i < N) dst[i] = from_f32<OT>(v[i]);
      }
    }
  }
}

template <typename AT, int MT, int WK, bool GU, bool PARTIAL, int NG>
int launch_skinny(Mfma16Params p, hipStream_t st) {
  constexpr int R = 4;
  p.n_tiles = (int)cdiv(p.N, 16 * (GU ? R / 2 : R));
  const int groups = (int)(p.K / p.ksplit / p.group) + 1;  // (a range may start and end inside a group)
  const size_t lds = (size_t)WK * R * MT * 1024 + (size_t)(groups + 1) * 68 * 4;
  const int64_t blocks = (int64_t)p.n_tiles * p.ksplit * p.E;
  if (lds > 64 * 1024 || blocks > 0x7FFFFFFF) return MLS_ERR_UNSUPPORTED;
  hipLaunchKernelGGL((grouped_skinny_kernel<AT, R, MT, WK, GU, PARTIAL, NG>), dim3((unsigned)blocks), dim3(64 * WK), lds,
                     st, p);
  return check_launch("grouped INT4 GEMM");
}

template <typename AT, bool GU, bool PARTIAL, int NG>
int launch_skinny_mt(const Mfma16Params& p, hipStream_t st) {
  // one tile of x rows where the average segment fills half of it or less (an uneven routing
  // then mostly fits), and 8 wavefronts a block where blocks are few and their ranges long
  const bool one = (int64_t)p.M * 2 <= (int64_t)p.E * 16;
  const bool wide = cdiv(p.N, GU ? 32 : 64) * p.ksplit * p.E < 1024 && p.K / 128 / p.ksplit >= 16;
  if (one) return wide ? launch_skinny<AT, 1, 8, GU, PARTIAL, NG>(p, st) : launch_skinny<AT, 1, 4, GU, PARTIAL, NG>(p, st);
  return wide ? launch_skinny<AT, 2, 8, GU, PARTIAL, NG>(p, st) : launch_skinny<AT, 2, 4, GU, PARTIAL, NG>(p, st);
}

}  // namespace

// Whether the skinny kernel takes a grouped GEMM (p.ksplit >= 1): ranges of whole steps, 32-bit
// offsets, and few rows an expert. The line lies where the two kernels meet (4096 -> 14336, 8
// experts, us): at 16 rows gate/up 205 -> 176, down 98 -> 84 (groups of 128) and 231 -> 211, 117
// -> 129 (groups of 64: two sets of products a step), at 24 gate/up 211 -> 227. Above, each
// further tile of rows streams the weights again.
bool grouped_skinny_fits(const Mfma16Params& p, bool gate_up) {
  const int rows = p.group == 64 && !gate_up ? 8 : 16;
  return (p.group == 64 || p.group % 128 == 0) && p.K % (128 * p.ksplit) == 0 && (int64_t)p.M <= (int64_t)p.E * rows &&
         p.N * p.ldb < (1ll << 31) && (int64_t)(p.a_rows ? p.a_src_rows : p.M) * p.lda * 2 < (1ll << 31);
}

int launch_grouped_skinny(const Mfma16Params& p, hipStream_t st, bool bf16, bool gate_up, bool partial) {
  const bool g64 = p.group == 64;
#define MLS_GS(AT_, S_)                                                                                   \
  return gate_up ? launch_skinny_mt<AT_, true, false, S_>(p, st)                                          \
                 : partial ? launch_skinny_mt<AT_, false, true, S_>(p, st) : launch_skinny_mt<AT_, false, false, S_>(p, st)
  if (bf16) {
    if (g64) MLS_GS(__bf16, 2);
    MLS_GS(__bf16, 1);
  }
  if (g64) MLS_GS(_Float16, 2);
  MLS_GS(_Float16, 1);
#undef MLS_GS
}

}  // namespace mls

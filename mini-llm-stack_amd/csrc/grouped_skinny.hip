// INT4 grouped GEMMs of a routed MoE layer with few rows an expert (a decode batch): every
// expert's weights stream once, straight into MFMA operand layout.
//
// The chunk kernel (gemm_grouped.hip) widens each weight into LDS for a row chunk of at least
// 64 rows: an LDS write and several LDS reads on top of the widening, whatever the segment
// holds, and it multiplies the rows that are not there. With 2 to 4 rows an expert it is bound by
// that work: 16 tokens, top-2 of 8 experts (4096 -> 14336, g128), gate/up 233 us and down in 4 K
// ranges 105; this kernel 126 (3.9 TB/s of weights) and 60.
//
// The result is the chunk kernel's, bit for bit, whichever of the two takes a call: the same
// exact weights 16 (v - 8), the same 32 k in each MFMA and in the same lanes, one chain of MFMAs
// over all k of an output, and the group scales applied at the same places in the same form. So a
// row does not depend on how many others share its call, non-finite ones included (as fp32
// arithmetic has them, but for the scale-table form, whose differences of scales may turn an
// infinity into a NaN). A wavefront therefore owns its outputs for the whole K range. (Taking the
// nibbles' offset off afterwards, (128 + v) x summed and 136 sum(x) subtracted, is half the
// widening, and with K shared by the wavefronts of a block it took 120 and 56 us; its sums were
// 10 (bf16) to 100 (fp16) times as far from the exact ones, and an infinite x became NaN.)
//
// Block: W wavefronts, a tile of 16 weight rows each, and MT tiles of 16 rows of x; segments longer
// than 16 MT rows take further passes over the block's weights, which are then in the Infinity
// Cache. Gate/up: the first half of the wavefronts holds gate rows, the second the same rows of up,
// which pass their products through LDS. A step is 128 k: a lane's 16 weight bytes come straight into
// registers, SPT steps in flight, and a 4 x 4 transpose over the wavefront's 16-lane rows
// (permlane swaps) gives each of the step's four MFMAs its own 32 k. The block's x goes through
// LDS, SPT steps a stage, double buffered: loaded into registers at the head of a stage, stored at
// its end, so there is one barrier a stage and no wait for the weights in flight. Rows of x past
// the segment load from past the operand (zeros, no traffic).
#include <type_traits>

#include "mfma16.h"

namespace mls {

namespace {

constexpr uint32_t kOutside = 0x80000000u;  // past every descriptor (they span < 2^31 bytes)

// v[i] of 16-lane row q becomes v[q] of row i.
__device__ __forceinline__ void transpose4(uint32_t (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(v[i], v[i + 2], false, false);
    v[i] = r[0];
    v[i + 2] = r[1];
  }
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const auto r = __builtin_amdgcn_permlane16_swap(v[i], v[i + 1], false, false);
    v[i] = r[0];
    v[i + 1] = r[1];
  }
}

// p.n_tiles: blocks a matrix; p.ksplit: K ranges whose products go to separate fp32 outputs
// (PARTIAL), else 1. G64: groups of 64, two in a step; else multiples of 128. TAB: the chunk
// kernel's scale-table form, sum_g (s_g - s_{g+1}) T_g over running sums T_g that are never
// cleared; else sum_g s_g P_g.
template <typename AT, int MT, int W, int SPT, bool GU, bool PARTIAL, bool G64, bool TAB>
__global__ __launch_bounds__(64 * W) void grouped_skinny_kernel(const Mfma16Params p) {
  using MM = Mfma16<AT>;
  constexpr int KS = 128, NT = 64 * W;
  constexpr int ROWS = 16 * W, TS = ROWS + 4;      // weight rows a block; floats a group of the scale table
  constexpr int CPR = SPT * KS / 8;              // 16-byte chunks a row of x and stage
  constexpr int XL = 16 * MT * CPR / NT;          // of them a thread loads
  constexpr int OUTN = GU ? ROWS / 2 : ROWS;    // output columns a block
  extern __shared__ __align__(16) uint8_t smem[]; // x: [2][16 MT][CPR] chunks; scales [groups of the range][TS]
  uint4* const xs = reinterpret_cast<uint4*>(smem);
  float* const sc_lds = reinterpret_cast<float*>(smem + 2 * 16 * MT * CPR * 16);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  int L = blockIdx.x;
  const int per = p.n_tiles * p.ksplit, e = L / per;
  L -= e * per;
  const int sp = L / p.n_tiles, n0 = (L - sp * p.n_tiles) * OUTN;
  int lo, hi;
  seg_rows(p, e, lo, hi);
  if (lo >= hi) return;
  const int N = p.N;
  const int steps = p.K / KS / p.ksplit, s_lo = steps * sp, s_hi = s_lo + steps;

  const int x_rows = p.a_rows ? p.a_src_rows : p.M;
  const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.a, (short)0, (int)(((x_rows - 1) * p.lda + p.K) * 2), 0x00020000);

  // this wavefront's tile: weight rows n_lo .. n_lo + 15 (gate/up: the second half of the wavefronts
  // the rows of up that the first half takes of the gate)
  const bool up = GU && wave >= W / 2;
  const int n_lo = n0 + 16 * (GU ? wave % (W / 2) : wave);
  const uint8_t* wmat = (up ? p.b2 : p.b) + (int64_t)e * p.b_estride;
  const __amdgpu_buffer_rsrc_t rsw = __builtin_amdgcn_make_buffer_rsrc(
      (void*)wmat, (short)0, (int)((N - 1) * p.ldb + p.K / 2), 0x00020000);
  const int wo = n_lo + r16 < N ? (n_lo + r16) * (int)p.ldb + 16 * q : (int)kOutside;
  uint4 w[SPT];
  auto load_w = [&](int i, int st) __attribute__((always_inline)) {
    const int k = min(st, s_hi - 1);  // (a step past the range repeats the last one, unused)
    w[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsw, wo, k * (KS / 2), 0));
  };
  // x: chunk c = tid + NT i of a stage is row c / CPR, 8 k at 8 (c % CPR)
  static_assert(NT % CPR == 0, "a thread's chunks share their column");
  const int x_col = tid % CPR, x_row0 = tid / CPR;
  int xo[XL];
  uint4 xr[XL];
  auto rows_at = [&](int m0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int m = m0 + x_row0 + i * (NT / CPR);
      int row = -1;
      if (m < hi) row = p.a_rows ? p.a_rows[m] : m;
      xo[i] = row >= 0 && row < x_rows ? row * (int)p.lda * 2 + 16 * x_col : (int)kOutside;
    }
  };
  auto load_x = [&](int st) __attribute__((always_inline)) {  // the stage that starts with step st
    const bool in = st * KS + 8 * x_col < s_hi * KS;
#pragma unroll
    for (int i = 0; i < XL; ++i)
      xr[i] = __builtin_bit_cast(
          uint4, __builtin_amdgcn_raw_buffer_load_b128(rsa, in ? xo[i] : (int)kOutside, st * KS * 2, 0));
  };
  auto store_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int row = x_row0 + i * (NT / CPR);
      xs[(buf * 16 * MT + row) * CPR + (x_col ^ swz(row))] = xr[i];
    }
  };
  // LDS only: the weight loads stay in flight
  auto barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  rows_at(lo);
  load_x(s_lo);
#pragma unroll
  for (int i = 0; i < SPT; ++i) load_w(i, s_lo + i);

  // the block's scales as fp32 [group of the range][weight row]: 16 groups x 4 rows a wavefront
  // and instruction
  const int g_lo = s_lo * KS / p.group, groups = steps * KS / p.group;  // (ranges are whole groups)
  for (int r = wave * 4 + q; r < ROWS; r += 4 * W) {
    const int n = min(n0 + (GU ? r % (ROWS / 2) : r), N - 1);
    const void* smat = GU && r >= ROWS / 2 ? p.s2 : p.s;
    const int64_t base = (int64_t)e * p.s_estride + (int64_t)n * p.ld_sn + (int64_t)g_lo * p.ld_sg;
    for (int g = r16; g < groups; g += 16) {
      float s = scale_at(smat, p.s_dt, base + (int64_t)g * p.ld_sg);
      if constexpr (TAB) {
        const int gn = min(g + 1, groups - 1);
        s = fmaf(g + 1 < groups ? -1.f : -0.f, scale_at(smat, p.s_dt, base + (int64_t)gn * p.ld_sg), s);
      }
      sc_lds[g * TS + r] = s;
    }
  }

  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  const int spg = G64 ? 1 : p.group / KS;  // steps a group
  for (int m0 = lo; m0 < hi; m0 += 16 * MT) {
    if (m0 != lo) {
      rows_at(m0);
      load_x(s_lo);
#pragma unroll
      for (int i = 0; i < SPT; ++i) load_w(i, s_lo + i);
    }
    store_x(0);
    barrier();
    f32x4 acc[MT], tot[MT];
#pragma unroll
    for (int tm = 0; tm < MT; ++tm) acc[tm] = tot[tm] = zero;
    const float* sg = sc_lds + 16 * wave + 4 * q;  // the running group's scales of this lane's outputs
    int left = spg;
    auto group_end = [&](const f32x4& sc) __attribute__((always_inline)) {
#pragma unroll
      for (int tm = 0; tm < MT; ++tm) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[tm][i] = fmaf(sc[i], tot[tm][i], acc[tm][i]);
        if constexpr (!TAB) tot[tm] = zero;
      }
      sg += TS;
    };
    auto compute = [&](int i, int buf) __attribute__((always_inline)) {  // step i of the stage in `buf`
      // every LDS read of the step first (the compiler would put each in front of its MFMA and wait)
      uint4 xop[4][MT];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int tm = 0; tm < MT; ++tm) {
          const int row = 16 * tm + r16;
          xop[j][tm] = xs[(buf * 16 * MT + row) * CPR + ((16 * i + 4 * j + q) ^ swz(row))];
        }
      f32x4 sc[G64 ? 2 : 1];
#pragma unroll
      for (int h = 0; h < (G64 ? 2 : 1); ++h) sc[h] = *reinterpret_cast<const f32x4*>(sg + h * TS);
      __builtin_amdgcn_sched_barrier(0);
      uint32_t d[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
      transpose4(d);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t o[4];
        widen_int4x16<AT>(d[j], o);
#pragma unroll
        for (int tm = 0; tm < MT; ++tm) tot[tm] = MM::mma(make_uint4(o[0], o[1], o[2], o[3]), xop[j][tm], tot[tm]);
        if constexpr (G64)
          if (j == 1 || j == 3) group_end(sc[j >> 1]);
      }
      if constexpr (!G64)
        if (--left == 0) {
          group_end(sc[0]);
          left = spg;
        }
    };
    int buf = 0;
    for (int st = s_lo; st < s_hi; st += SPT, buf ^= 1) {
      load_x(st + SPT);  // (past the range: zeros, unused)
      if (st + SPT <= s_hi) {
#pragma unroll
        for (int i = 0; i < SPT; ++i) {
          compute(i, buf);
          load_w(i, st + SPT + i);
        }
      } else {
#pragma unroll
        for (int i = 0; i < SPT; ++i)
          if (st + i < s_hi) compute(i, buf);
      }
      store_x(buf ^ 1);
      barrier();
    }

    if constexpr (GU) {  // the up products to the wavefronts of the same gate rows, through x's buffers
      f32x4* ex = reinterpret_cast<f32x4*>(smem) + (wave % (W / 2)) * MT * 64 + lane;
      if (up) {
#pragma unroll
        for (int tm = 0; tm < MT; ++tm) ex[tm * 64] = acc[tm];
      }
      barrier();
#pragma unroll
      for (int tm = 0; tm < MT; ++tm) tot[tm] = ex[tm * 64];
      barrier();  // (x's buffers are free for the next pass)
      if (up) continue;
    }
    // acc[tm][i] = C[m0 + 16 tm + r16][n_lo + 4 q + i] times 16
    using OT = std::conditional_t<PARTIAL, float, AT>;
    OT* c = static_cast<OT*>(p.c) + (PARTIAL ? (int64_t)sp * p.c_sstride : 0);
    const int nb = n_lo + 4 * q;
    if (nb >= N) continue;
#pragma unroll
    for (int tm = 0; tm < MT; ++tm) {
      const int m = m0 + 16 * tm + r16;
      if (m >= hi) continue;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = acc[tm][i] * 0.0625f;
        if constexpr (GU) {
          const float g = v[i];
          v[i] = g / (1.0f + __expf(-g)) * (tot[tm][i] * 0.0625f);
          asm("" : "+v"(v[i]));  // rounded to fp32 first, as in the chunk kernel (not fused with the fp16 convert)
        }
      }
      OT* dst = c + (int64_t)m * p.ldc + nb;
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

// One tile of x rows where the average segment fills half of it or less (an uneven routing then
// mostly fits), else two.
int skinny_mt(int64_t M, int E) { return M * 2 <= (int64_t)E * 16 ? 1 : 2; }

int64_t skinny_lds(int mt, int waves, int spt, int64_t K, int ksplit, int group) {
  return 2 * 16 * mt * spt * 128 * 2 + K / ksplit / group * (16 * waves + 4) * 4;
}

template <typename AT, int MT, int W, int SPT, bool GU, bool PARTIAL, bool G64, bool TAB>
int launch_skinny(Mfma16Params p, hipStream_t st) {
  p.n_tiles = (int)cdiv(p.N, 16 * W / (GU ? 2 : 1));
  const int64_t blocks = (int64_t)p.n_tiles * p.ksplit * p.E;
  const int64_t lds = skinny_lds(MT, W, SPT, p.K, p.ksplit, p.group);
  if (blocks > 0x7FFFFFFF) return MLS_ERR_UNSUPPORTED;
  auto kern = grouped_skinny_kernel<AT, MT, W, SPT, GU, PARTIAL, G64, TAB>;
  // (past the default limit a call a launch: the limit is the function's on the current device)
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return fail(MLS_ERR_HIP, "grouped INT4 GEMM: cannot reserve %lld bytes of LDS", (long long)lds);
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(64 * W), (unsigned)lds, st, p);
  return check_launch("grouped INT4 GEMM");
}

// The form for a shape, us measured with 4096 -> 14336, 8 experts, groups of 128, unless said:
// - 4 wavefronts a block: 16 tokens gate/up 124 and down in 4 ranges 57, 8 wavefronts 143 and 63; 24
//   tokens of 4 experts, 2048 -> 5632, 21.5 and 27.6 against 25.0 and 35.9. With two tiles of x and two
//   blocks or more a CU, 8 wavefronts share x's traffic better: 48 tokens 161 and 74 against 173 and 80.
// - stages of 2 steps, which leave registers and LDS for more blocks (gate/up at 16 tokens 124, 4
//   steps 138); of 4 where a wavefront walks far and the blocks of the experts that M rows can reach
//   come to less than four a CU (down unsplit at 16 tokens 80 and 72, at 1 token 60 and 52).
template <typename AT, bool GU, bool PARTIAL, bool G64, bool TAB>
int launch_skinny_tile(const Mfma16Params& p, hipStream_t st) {
  const int64_t rows = GU ? 2 * (int64_t)p.N : p.N;
  if (skinny_mt(p.M, p.E) == 2)
    return cdiv(rows, 128) * p.ksplit * p.E >= 512 ? launch_skinny<AT, 2, 8, 2, GU, PARTIAL, G64, TAB>(p, st)
                                                   : launch_skinny<AT, 2, 4, 2, GU, PARTIAL, G64, TAB>(p, st);
  const int64_t live = cdiv(rows, 64) * p.ksplit * (p.M < p.E ? p.M : p.E);
  return live < 1024 && p.K / p.ksplit >= 4096 ? launch_skinny<AT, 1, 4, 4, GU, PARTIAL, G64, TAB>(p, st)
                                               : launch_skinny<AT, 1, 4, 2, GU, PARTIAL, G64, TAB>(p, st);
}

template <typename AT, bool GU, bool PARTIAL>
int launch_skinny_form(const Mfma16Params& p, hipStream_t st, bool table) {
  if (p.group == 64)
    return table ? launch_skinny_tile<AT, GU, PARTIAL, true, true>(p, st)
                 : launch_skinny_tile<AT, GU, PARTIAL, true, false>(p, st);
  return table ? launch_skinny_tile<AT, GU, PARTIAL, false, true>(p, st)
               : launch_skinny_tile<AT, GU, PARTIAL, false, false>(p, st);
}

}  // namespace

// Whether the skinny kernel takes a grouped GEMM: ranges of whole steps and groups, scales and x
// stages within the LDS, and at most 16 rows an expert on average, to where it was measured ahead
// of the chunk kernel (us, chunk and this, 48 tokens, top-2 of 8, 4096 -> 14336: gate/up 208 and
// 164, down 142 and 95, in 4 ranges 101 and 77; 64 tokens with groups of 64 230 and 181, 187 and 115,
// 119 and 92).
// Above, each further pass of 32 rows streams the weights again.
bool grouped_skinny_takes(int64_t M, int E, int64_t K, int group, int ksplit) {
  return (group == 64 || group % 128 == 0) && K % (128 * (int64_t)ksplit) == 0 && K / ksplit % group == 0 &&
         M <= (int64_t)E * 16 &&
         (skinny_mt(M, E) == 1 ? skinny_lds(1, 4, 4, K, ksplit, group) : skinny_lds(2, 8, 2, K, ksplit, group)) <=
             160 * 1024;
}

bool grouped_skinny_fits(const Mfma16Params& p) {
  return grouped_skinny_takes(p.M, p.E, p.K, p.group, p.ksplit) && p.N * p.ldb < (1ll << 31) &&
         (int64_t)(p.a_rows ? p.a_src_rows : p.M) * p.lda * 2 < (1ll << 31);
}

int launch_grouped_skinny(const Mfma16Params& p, hipStream_t st, bool bf16, bool gate_up, bool partial, bool table) {
  if (bf16)
    return gate_up ? launch_skinny_form<__bf16, true, false>(p, st, table)
                   : partial ? launch_skinny_form<__bf16, false, true>(p, st, table)
                             : launch_skinny_form<__bf16, false, false>(p, st, table);
  return gate_up ? launch_skinny_form<_Float16, true, false>(p, st, table)
                 : partial ? launch_skinny_form<_Float16, false, true>(p, st, table)
                           : launch_skinny_form<_Float16, false, false>(p, st, table);
}

}  // namespace mls

extern "C" int mlsx_int4_grouped_few_rows(int64_t M_total, int E, int64_t K, int group, int splits) {
  return M_total > 0 && E > 0 && K > 0 && group > 0 && splits > 0 &&
         mls::grouped_skinny_takes(M_total, E, K, group, splits);
}

// dw[N][K] = dy[M][N]^T x[M][K], all fp32: the master weight's gradient of the INT8
// straight-through estimator (kernels/autograd_ops.py:132), on the bf16 matrix cores.
//
// gfx950 has no fp32 matrix rate near its 16-bit one (4096 x 4096 over 2048 tokens: 468 us in
// the fp32 library product, 147 TFLOP/s). Here every fp32 value becomes three bf16 parts that
// add up to it exactly (8 of its 24 significant bits each, by truncation, so all parts have
// its sign), and a product becomes the six part products above 2^-24 of it: hi hi, hi mid,
// mid hi, mid mid, hi lo, lo hi. bf16 keeps fp32's exponent range, so small values beside large
// ones keep their bits; and both operands are taken times 2^16, which lifts fp32's smallest value
// (2^-149) to bf16's (2^-133), so that no bit of any value is lost.
//
// Two launches on the caller's stream: dw_parts_kernel transposes both operands into parts with
// the reduction axis contiguous, [C][3][Mp] (row 3 c + part, Mp = M rounded up to 32, zeros past
// M), then dw_kernel multiplies. A part read from LDS once feeds two or three products, so the
// LDS traffic per MFMA is half that of a plain bf16 GEMM and the kernel is bound by the matrix
// cores: 320 us for both launches at that size, 1.29 PFLOP/s over the six products, the rate
// of a plain bf16 GEMM. Error against 64 bits there 2.8e-7 of the norm, the library product's 8.1e-7.
//
// dw_kernel: block tile BP (rows of dw) x BQ (columns) x 32 tokens, 8 wavefronts of 64 x WTQ
// outputs, two LDS buffers filled by LDS-direct loads one stage ahead, one barrier a stage.
// A stage reads its operands into registers before it issues the next stage's loads: the
// compiler would hold an LDS read behind every LDS-direct load in flight. hi hi has an
// accumulator of its own and the other five share one, so the large sum is rounded once per 32
// tokens, not six times.
//
// Infinities, NaN, values from 2^112 and sums from 2^96 leave a non-finite value in every tile that
// they touch: such a block computes its tile again from the operands themselves with fp32 FMAs
// (whole_tile), which gives what fp32 arithmetic gives, at a fraction of the speed.
#include <algorithm>

#include "mfma16.h"

namespace mls {

namespace {

constexpr int kStage = 32;  // tokens a stage: one MFMA step
constexpr float kLift = 65536.0f, kDrop = 1.0f / (65536.0f * 65536.0f);  // both operands' 2^16, off again

struct DwParams {
  const uint16_t* p;  // parts of dy [N][3][Mp]
  const uint16_t* q;  // parts of x [K][3][Mp]
  float* c;
  int64_t ldc;
  int P, Q, Mp;
  const float* dy;    // the operands themselves (whole_tile)
  const float* x;
  int64_t lddy, ldx;
  int M;
  int p_tiles, q_tiles;
};

// 64 tokens x 64 columns of fp32 through LDS. Loads: 16 consecutive lanes take 256 bytes of a
// row; stores: 8 lanes take 128 bytes of a part's row. blockIdx.z: 0 dy, 1 x.
__global__ __launch_bounds__(256) void dw_parts_kernel(const float* __restrict__ dy, int64_t lddy, int N,
                                                       const float* __restrict__ x, int64_t ldx, int K, int M, int Mp,
                                                       uint16_t* __restrict__ dyp, uint16_t* __restrict__ xp,
                                                       int vec) {
  __shared__ float tile[64][65];
  const bool second = blockIdx.z != 0;
  const float* src = second ? x : dy;
  const int64_t ld = second ? ldx : lddy;
  const int C = second ? K : N;
  uint16_t* dst = second ? xp : dyp;
  const int c0 = blockIdx.x * 64, m0 = blockIdx.y * 64, tid = threadIdx.x;
  if (c0 >= C) return;
  const bool v4 = (vec >> (second ? 1 : 0)) & 1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * 16 + tid / 16, c = (tid % 16) * 4, m = m0 + r;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (m < M) {
      const float* s = src + (int64_t)m * ld + c0 + c;
      if (v4 && c0 + c + 4 <= C) {
        const float4 f = *reinterpret_cast<const float4*>(s);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c0 + c + e < C) v[e] = s[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[r][c + e] = v[e];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = i * 32 + tid / 8, r0 = (tid % 8) * 8;
    if (c0 + c >= C || m0 + r0 >= Mp) continue;  // Mp is a multiple of 8
    uint32_t o[3][4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float part[3][2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float v = tile[r0 + 2 * h + e][c] * kLift;
        float rest, low;
        split_f32(v, part[0][e], rest);
        split_f32(rest, part[1][e], low);
        part[2][e] = low;
        if ((__float_as_uint(v) & 0x7F800000u) == 0x7F800000u) part[1][e] = part[2][e] = part[0][e];
      }
#pragma unroll
      for (int t = 0; t < 3; ++t) o[t][h] = pack2_bits((__bf16)part[t][0], (__bf16)part[t][1]);  // exact
    }
#pragma unroll
    for (int t = 0; t < 3; ++t)
      *reinterpret_cast<uint4*>(dst + ((int64_t)3 * (c0 + c) + t) * Mp + m0 + r0) =
          make_uint4(o[t][0], o[t][1], o[t][2], o[t][3]);
  }
}

// Where 16-byte chunk c of 64-byte row `row` sits: the 16 rows of an operand read cover all banks.
__device__ __forceinline__ int chunk_at(int row, int c) { return c ^ ((row >> 1) & 3); }

// One stage of ROWS values x 3 parts in LDS as [part][row][32 tokens]: an instruction of a
// wavefront fills 16 rows, the 8 wavefronts 128, so a lane's rows differ by constants and its
// chunk stays the same.
template <int ROWS>
struct Fill {
  static_assert(ROWS % 128 == 0, "whole instructions for 8 wavefronts");
  int off;
  __device__ __forceinline__ void init(int wave, int lane, int ld) {
    const int row = wave * 16 + lane / 4;
    off = 3 * row * ld + chunk_at(row, lane & 3) * 16;
  }
  __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rs, uint8_t* lds, int wave, int ld, int k_bytes) const {
    asm volatile("" : "+s"(ld));  // the offsets are made here, not kept in registers over the loop
#pragma unroll
    for (int i = 0; i < 3 * ROWS / 128; ++i)
      lds_load16(rs, lds + (i * 8 + wave) * 1024, off + (3 * (i * 128 % ROWS) + i * 128 / ROWS) * ld, k_bytes);
  }
};

// This wavefront's LDS-direct loads have landed, then everyone's. The empty asm statements keep
// LDS accesses on their side of the barrier.
__device__ __forceinline__ void stage_sync() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0 | 0x70 | 0xF00);  // vmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int BP, int BQ, int WP, int WQ>
struct DwTile {
  static constexpr int TP = BP / WP / 16, TQ = BQ / WQ / 16;
  static constexpr int P_STAGE = 3 * BP * 64, Q_STAGE = 3 * BQ * 64, STAGE = P_STAGE + Q_STAGE;
  static_assert(WP * WQ == 8, "8 wavefronts");

  // all stages of one tile
  __device__ static __forceinline__ void run(const DwParams& p, uint8_t* smem, int p0, int q0, int wave, int lane,
                                             f32x4 (&big)[TQ][TP], f32x4 (&rest)[TQ][TP]) {
    const int ld = p.Mp * 2;
    const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.p + (int64_t)3 * p0 * p.Mp), (short)0, 3 * min(BP, p.P - p0) * ld, 0x00020000);
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.q + (int64_t)3 * q0 * p.Mp), (short)0, 3 * min(BQ, p.Q - q0) * ld, 0x00020000);
    Fill<BP> fp;
    Fill<BQ> fq;
    fp.init(wave, lane, ld);
    fq.init(wave, lane, ld);
    const int lr = lane & 15, g = lane >> 4;
    const int wp0 = (wave / WQ) * (BP / WP), wq0 = (wave % WQ) * (BQ / WQ);
    // (rows wp0 + 16 j + lr share (row >> 1) & 3)
    const int pb = (wp0 + lr) * 64 + chunk_at(wp0 + lr, g) * 16;
    const int qb = P_STAGE + (wq0 + lr) * 64 + chunk_at(wq0 + lr, g) * 16;
#pragma unroll
    for (int i = 0; i < TQ; ++i)
#pragma unroll
      for (int j = 0; j < TP; ++j) big[i][j] = rest[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int nk = p.Mp / kStage;
    fp.issue(rp, smem, wave, ld, 0);
    fq.issue(rq, smem + P_STAGE, wave, ld, 0);
    stage_sync();
    for (int kt = 0; kt < nk; ++kt) {
      const int cur = (kt & 1) * STAGE;
      uint4 a[TQ][3], b[TP][3];
#pragma unroll
      for (int i = 0; i < TQ; ++i)
#pragma unroll
        for (int t = 0; t < 3; ++t)
          a[i][t] = *reinterpret_cast<const uint4*>(smem + cur + qb + t * BQ * 64 + i * 1024);
#pragma unroll
      for (int j = 0; j < TP; ++j)
#pragma unroll
        for (int t = 0; t < 3; ++t)
          b[j][t] = *reinterpret_cast<const uint4*>(smem + cur + pb + t * BP * 64 + j * 1024);
      __builtin_amdgcn_sched_barrier(0);
      if (kt + 1 < nk) {  // into the buffer that stage kt - 1 used
        uint8_t* nxt = smem + (STAGE - cur);
        fp.issue(rp, nxt, wave, ld, (kt + 1) * kStage * 2);
        fq.issue(rq, nxt + P_STAGE, wave, ld, (kt + 1) * kStage * 2);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < TP; ++j) {
        const uint4 bh = b[j][0], bm = b[j][1], bl = b[j][2];
        // a product at a time over the tiles: no MFMA waits for the one before it
        using X = Mfma16<__bf16>;
#pragma unroll
        for (int i = 0; i < TQ; ++i) rest[i][j] = X::mma(a[i][2], bh, rest[i][j]);
#pragma unroll
        for (int i = 0; i < TQ; ++i) rest[i][j] = X::mma(a[i][0], bl, rest[i][j]);
#pragma unroll
        for (int i = 0; i < TQ; ++i) rest[i][j] = X::mma(a[i][1], bm, rest[i][j]);
#pragma unroll
        for (int i = 0; i < TQ; ++i) rest[i][j] = X::mma(a[i][1], bh, rest[i][j]);
#pragma unroll
        for (int i = 0; i < TQ; ++i) rest[i][j] = X::mma(a[i][0], bm, rest[i][j]);
#pragma unroll
        for (int i = 0; i < TQ; ++i) big[i][j] = X::mma(a[i][0], bh, big[i][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
      stage_sync();
    }
  }
};

// dw[p0 .. p0 + BP)[q0 .. q0 + BQ) by fp32 FMAs, tokens in order: 16 tokens of both operands in LDS a
// step, BP / 32 x BQ / 16 outputs a thread.
template <int BP, int BQ>
__device__ __forceinline__ void whole_tile(const DwParams& p, float* smem, int p0, int q0) {
  constexpr int T = 16, RP = BP / 32, RQ = BQ / 16;
  float (*ds)[BP] = reinterpret_cast<float(*)[BP]>(smem);
  float (*xs)[BQ] = reinterpret_cast<float(*)[BQ]>(smem + T * BP);
  const int tid = threadIdx.x, tp = tid / 16, tq = tid % 16;
  float acc[RP][RQ];
#pragma unroll
  for (int i = 0; i < RP; ++i)
#pragma unroll
    for (int j = 0; j < RQ; ++j) acc[i][j] = 0.0f;
  for (int m0 = 0; m0 < p.M; m0 += T) {
    __syncthreads();
    const int n = min(T, p.M - m0);
    for (int t = tid; t < n * BP; t += 512) {
      const int m = t / BP, c = t % BP;
      ds[m][c] = p0 + c < p.P ? p.dy[(int64_t)(m0 + m) * p.lddy + p0 + c] : 0.0f;
    }
    for (int t = tid; t < n * BQ; t += 512) {
      const int m = t / BQ, c = t % BQ;
      xs[m][c] = q0 + c < p.Q ? p.x[(int64_t)(m0 + m) * p.ldx + q0 + c] : 0.0f;
    }
    __syncthreads();
    for (int m = 0; m < n; ++m) {
      float a[RP], b[RQ];
#pragma unroll
      for (int i = 0; i < RP; ++i) a[i] = ds[m][tp + 32 * i];
#pragma unroll
      for (int j = 0; j < RQ; ++j) b[j] = xs[m][tq + 16 * j];
#pragma unroll
      for (int i = 0; i < RP; ++i)
#pragma unroll
        for (int j = 0; j < RQ; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < RP; ++i)
#pragma unroll
    for (int j = 0; j < RQ; ++j) {
      const int r = p0 + tp + 32 * i, c = q0 + tq + 16 * j;
      if (r < p.P && c < p.Q) p.c[(int64_t)r * p.ldc + c] = acc[i][j];
    }
}

template <int BP, int BQ, int WP, int WQ>
__global__ __launch_bounds__(512) void dw_kernel(const DwParams p) {
  using T = DwTile<BP, BQ, WP, WQ>;
  extern __shared__ __align__(16) uint8_t smem[];
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  int pt, qt;
  tile_order(L, p.p_tiles, p.q_tiles, 4, pt, qt);
  const int p0 = pt * BP, q0 = qt * BQ;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  f32x4 big[T::TQ][T::TP], rest[T::TQ][T::TP];
  T::run(p, smem, p0, q0, wave, lane, big, rest);
  bool bad = false;
#pragma unroll
  for (int i = 0; i < T::TQ; ++i)
#pragma unroll
    for (int j = 0; j < T::TP; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = big[i][j][r] + rest[i][j][r];
        bad |= (__float_as_uint(v) & 0x7F800000u) == 0x7F800000u;
      }
  if (__syncthreads_or(bad)) {
    whole_tile<BP, BQ>(p, reinterpret_cast<float*>(smem), p0, q0);
    return;
  }

  // lane: dw[p = .. + lane % 16][q = .. + 4 (lane / 16) + r]
  const int lr = lane & 15, g = lane >> 4;
  const int wp0 = p0 + (wave / WQ) * (BP / WP), wq0 = q0 + (wave % WQ) * (BQ / WQ);
  const bool v4 = p.ldc % 4 == 0 && (uintptr_t)p.c % 16 == 0;
#pragma unroll
  for (int j = 0; j < T::TP; ++j) {
    const int row = wp0 + 16 * j + lr;
    if (row >= p.P) continue;
#pragma unroll
    for (int i = 0; i < T::TQ; ++i) {
      const int col = wq0 + 16 * i + 4 * g;
      const f32x4 v = (big[i][j] + rest[i][j]) * kDrop;
      float* dst = p.c + (int64_t)row * p.ldc + col;
      if (v4 && col + 3 < p.Q) {
        *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (col + r < p.Q) dst[r] = v[r];
      }
    }
  }
}

template <int BP, int BQ, int WP, int WQ>
int launch_dw(DwParams p, hipStream_t st) {
  p.p_tiles = (int)cdiv(p.P, BP);
  p.q_tiles = (int)cdiv(p.Q, BQ);
  constexpr int lds = 2 * DwTile<BP, BQ, WP, WQ>::STAGE;
  auto kern = dw_kernel<BP, BQ, WP, WQ>;
  // (a call a launch: the limit is the function's on the current device)
  if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return fail(MLS_ERR_HIP, "weight gradient: cannot reserve %d bytes of LDS", lds);
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.p_tiles * p.q_tiles)), dim3(512), lds, st, p);
  return check_launch("weight gradient");
}

// Outputs that the fullest CU computes (one block a CU at a time). The tile with fewer is taken,
// 256 x 128 where they tie: it reads a quarter less from L2 (4096 x 4096 over 2048 tokens 320 us,
// 128 x 128 355; 2048 x 2048, 256 tiles of 128 x 128, 138 and 99).
int64_t dw_cost(int64_t N, int64_t K, int64_t bp, int64_t bq) {
  return cdiv(cdiv(N, bp) * cdiv(K, bq), 256) * bp * bq;
}

int64_t padded(int64_t M) { return cdiv(M, kStage) * kStage; }

}  // namespace

}  // namespace mls

using namespace mls;

extern "C" int64_t mlsx_dw_fp32_workspace(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int64_t Mp = padded(M);
  // the row offsets of a block's buffers are 32-bit
  if (N > 0x3FFFFF || K > 0x3FFFFF || Mp > (0x7FFFFFFF / (3 * 256 * 2)) / kStage * kStage) return 0;
  return 6 * Mp * (N + K);
}

// Against the fp32 library product (us, this and that): 2048 x 4096 x 4096 320 and 468, 256 x 4096 x
// 4096 62 and 73, 1024 x 2048 x 2048 56 and 64, 1024 x 1024 x 4096 58 and 64, 2048 x 11008 x 4096 976
// and 1368. Below 2^32 products the launches and the parts weigh too much (256 x 4096 x 2048 37 and
// 36, 256 x 2048 x 2048 25 and 21), and where the last round of tiles leaves CUs idle the library's
// smaller tiles win (777 x 2048 x 1024, half of them, 47 and 30).
extern "C" int mlsx_dw_fp32_pays(int64_t M, int64_t N, int64_t K) {
  const int64_t need = mlsx_dw_fp32_workspace(M, N, K);
  if (need == 0 || need > ((int64_t)4 << 30)) return 0;
  const int64_t cost = std::min(dw_cost(N, K, 256, 128), dw_cost(N, K, 128, 128)) * 256;
  return M >= 256 && M * N >= ((int64_t)1 << 32) / K && cost * 85 <= N * K * 100;
}

extern "C" int mlsx_dw_fp32(const float* dy, int64_t lddy, const float* x, int64_t ldx, float* dw, int64_t lddw,
                            int64_t M, int64_t N, int64_t K, void* ws, int64_t ws_bytes, mls_stream_t stream) {
  const char* fn = "mlsx_dw_fp32";
  if (M < 0 || N < 0 || K < 0) return fail(MLS_ERR_ARG, "%s: negative size", fn);
  if (N == 0 || K == 0) return MLS_OK;
  const int64_t need = mlsx_dw_fp32_workspace(M, N, K);
  if (need == 0) return fail(MLS_ERR_UNSUPPORTED, "%s: M=%lld N=%lld K=%lld", fn, (long long)M, (long long)N, (long long)K);
  if (!dy || !x || !dw || !ws) return fail(MLS_ERR_ARG, "%s: null pointer", fn);
  if (lddy < N || ldx < K || lddw < K) return fail(MLS_ERR_ARG, "%s: bad leading dimension", fn);
  if (ws_bytes < need || !aligned(ws, 16)) return fail(MLS_ERR_ARG, "%s: workspace too small or misaligned", fn);
  const hipStream_t st = (hipStream_t)stream;
  const int Mp = (int)padded(M);
  uint16_t* dyp = (uint16_t*)ws;
  uint16_t* xp = dyp + 3 * N * Mp;
  const int vec = (aligned(dy, 16) && lddy % 4 == 0 ? 1 : 0) | (aligned(x, 16) && ldx % 4 == 0 ? 2 : 0);
  const int64_t rows = cdiv(Mp, 64);
  if (rows > 65535) return fail(MLS_ERR_UNSUPPORTED, "%s: M=%lld", fn, (long long)M);
  hipLaunchKernelGGL(dw_parts_kernel, dim3((unsigned)cdiv(std::max(N, K), 64), (unsigned)rows, 2), dim3(256), 0, st,
                     dy, lddy, (int)N, x, ldx, (int)K, (int)M, Mp, dyp, xp, vec);
  const int rc = check_launch(fn);
  if (rc != MLS_OK) return rc;
  const DwParams p{dyp, xp, dw, lddw, (int)N, (int)K, Mp, dy, x, lddy, ldx, (int)M, 0, 0};
  if (dw_cost(N, K, 256, 128) <= dw_cost(N, K, 128, 128)) return launch_dw<256, 128, 4, 2>(p, st);
  return launch_dw<128, 128, 2, 4>(p, st);
}

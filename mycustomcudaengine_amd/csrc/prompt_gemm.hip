// Prompt-sized GEMM for gfx950: out[M, N] (op)= x[M, K] . W[N, K]^T for the
// projections of a prefill of tens to hundreds of tokens (the reference runs
// them through torch.matmul, benchmarks/benchmark_engine.py:40-122), fp16 or
// bf16 in, fp32 accumulation; store, SwiGLU over [gate; up] rows, or add into
// the residual stream with the RMSNorm that follows it.
//
// Both operands are K-contiguous, so both are staged the same way: 64 k of a
// row are one 128-byte line, and a direct-to-LDS load instruction moves 8 rows
// (64 lanes x 16 bytes).  The 16-byte chunks of row r sit in its line permuted,
// chunk c at c ^ ((r >> 1) & 7), so that the fragment reads of
// v_mfma_f32_32x32x16 (32 rows x one chunk per half wave) spread over all banks;
// the permutation is applied by the lanes' global addresses.  A wave owns 32
// MF tokens x 32 NF columns (A = W, B = x: a lane ends with one token's 4
// consecutive columns); a workgroup is MW x NG waves.
//
// STAGES buffers of 64 k, one barrier per 64 k: the wait before it leaves the
// loads of the STAGES - 2 younger stages in flight; behind it the oldest
// buffer is free for the stage STAGES - 1 ahead.
//
// What bounds it: in-flight bytes over latency.  With 96 KB staged ahead per CU
// a CU takes in ~54 GB/s (~1.8 us of loaded latency; L2 hits alone would allow
// 128), so the tile grows with M -- fewer staged bytes per multiplication --
// and at M <= 128, where the weights' HBM stream is the floor, two workgroups
// per CU share the latency.  Small grids cut K into slices over workgroups
// (fp32 partial sums, added up by a second launch that also does the residual
// and the norm).  K slices and tiles that touch the same W rows are numbered
// next to each other on one XCD, so that W comes from HBM once.
//
// us per call, 3B shapes, weights from HBM, hipBLASLt (with the separate
// SwiGLU kernel) -> this, K slices summed: M = 64 q/k/v 17.3 -> 13.1, o 16.0 ->
// 11.2, gate/up 28.7 -> 23.7, down 23.8 -> 17.0; M = 100 18.6 -> 15.1, 16.5 ->
// 12.9, 36.5 -> 26.1, 27.5 -> 20.4; M = 300 gate/up 53.7 -> 47.6, down 40.4 ->
// 33.4; M = 512 69.4 -> 53.8, 49.2 -> 42.5.
#include "mce_common.h"
#include "mce_internal.h"
#include "mce_lds_dma.h"

#include <algorithm>

namespace mce {

struct PromptGemmArgs {
  const uint16_t *x, *w;
  uint16_t *out;
  float *part;  // [split, M, N] (split > 1)
  int M, N, K, x_stride, out_stride;
  int x_bytes, w_bytes;
  int mt, nt, split;  // token tiles, column tiles, K slices
  const uint16_t *norm_w;
  uint16_t *normed;  // [M, N]
  float eps;
};

constexpr int PG_BK = 64;  // k per stage
enum { PG_STORE, PG_ADD, PG_SWIGLU, PG_PART };

__device__ inline float pg_silu_mul(float g, float u) { return g / (1.0f + __expf(-g)) * u; }

// NT: W with the non-temporal policy (one token tile: every line is used once)
template <class T, int MW, int MF, int NG, int NF, int STAGES, int EPI, bool NT, int WPE>
__global__ __launch_bounds__(MW * NG * 64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void prompt_gemm_kernel(PromptGemmArgs a) {
  constexpr int BM = 32 * MW * MF, BN = 32 * NG * NF, NW = MW * NG;
  constexpr int STAGE = (BM + BN) * PG_BK * 2;
  constexpr int NIX = BM / 8 / NW, NIW = BN / 8 / NW;  // loads per wave and stage
  static_assert(NIX * 8 * NW == BM && NIW * 8 * NW == BN, "whole loads per wave");
  static_assert(EPI != PG_SWIGLU || NF % 2 == 0, "gate / up pairs of 32-column blocks");
  __shared__ __attribute__((aligned(1024))) char lds[STAGES * STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mw = wave % MW, ng = wave / MW;
  const int l32 = lane & 31, hf = lane >> 5;

  // workgroup -> (column tile, K slice, token tile): column tiles round-robin
  // over the XCDs, everything of one column tile on one XCD
  const int id = blockIdx.x, per = a.mt * a.split;
  const int ntile = (id >> 3) / per * 8 + (id & 7), rest = (id >> 3) % per;
  if (ntile >= a.nt) return;
  const int mtile = rest % a.mt, sl = rest / a.mt;
  const int steps = a.K / PG_BK;
  const int s0 = sl * steps / a.split;
  const int n_st = (sl + 1) * steps / a.split - s0;  // >= 1 (split <= steps)
  const int m0 = mtile * BM;
  const int n0 = ntile * (EPI == PG_SWIGLU ? BN / 2 : BN);

  // staging: load j of this wave fills rows 8 (wave NI + j) .. + 7 of the x /
  // W part of a stage (token rows past M re-read the last one; never stored)
  const i32x4 xr = buffer_rsrc(a.x, a.x_bytes), wr = buffer_rsrc(a.w, a.w_bytes);
  int vx[NIX], vw[NIW];
  const int p8 = lane & 7, r8 = lane >> 3;
#pragma unroll
  for (int j = 0; j < NIX; ++j) {
    const int row = 8 * (wave * NIX + j) + r8;
    vx[j] = min(m0 + row, a.M - 1) * a.x_stride * 2 + 16 * (p8 ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int j = 0; j < NIW; ++j) {
    const int row = 8 * (wave * NIW + j) + r8;
    // SwiGLU: 32-row blocks alternate between gate and up rows
    const int wrow = EPI == PG_SWIGLU ? n0 + 32 * (row >> 6) + (row & 31) + ((row >> 5) & 1) * a.N
                                      : n0 + row;
    vw[j] = wrow * a.K * 2 + 16 * (p8 ^ ((row >> 1) & 7));
  }
  const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)lds);
  const unsigned x_m0 = __builtin_amdgcn_readfirstlane(lds0 + wave * NIX * 1024);
  const unsigned w_m0 = __builtin_amdgcn_readfirstlane(lds0 + BM * 128 + wave * NIW * 1024);
  auto stage = [&](int s, int buf) {
    const int soff = (s0 + s) * (PG_BK * 2);
#pragma unroll
    for (int j = 0; j < NIW; ++j)
      buffer_load_lds16<NT>(wr, vw[j], soff, w_m0 + buf * STAGE + j * 1024);
#pragma unroll
    for (int j = 0; j < NIX; ++j) buffer_load_lds16(xr, vx[j], soff, x_m0 + buf * STAGE + j * 1024);
  };
  // fragment of 16 k, quarter j of the stage: chunk 2 j + hf of row l32 of a block
  int fo[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) fo[j] = l32 * 128 + 16 * ((2 * j + hf) ^ ((l32 >> 1) & 7));
  const int xb = mw * MF * 4096, wb = BM * 128 + ng * NF * 4096;

  floatx16 acc[NF][MF];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[f][m][e] = 0.f;
  auto compute = [&](int buf) {
    const char *b = lds + buf * STAGE;
    __builtin_amdgcn_iglp_opt(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u32x4 wf[NF], xf[MF];
#pragma unroll
      for (int f = 0; f < NF; ++f) wf[f] = *reinterpret_cast<const u32x4 *>(b + wb + f * 4096 + fo[j]);
#pragma unroll
      for (int m = 0; m < MF; ++m) xf[m] = *reinterpret_cast<const u32x4 *>(b + xb + m * 4096 + fo[j]);
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int m = 0; m < MF; ++m) acc[f][m] = mfma32<T>(wf[f], xf[m], acc[f][m]);
    }
  };
  int cur = 0, nxt = STAGES - 1, s = 0;
  // (slices of fewer than STAGES - 1 steps stage their last one again, into
  // buffers nobody reads: the waits count on STAGES - 1 stages)
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) stage(min(t, n_st - 1), t);
  for (; s + STAGES - 1 < n_st; ++s) {
    wait_loads<(NIX + NIW) * (STAGES - 2)>();  // this wave's part of stage s has landed
    lds_barrier();                             // everybody's; buffer nxt is read out
    stage(s + STAGES - 1, nxt);
    compute(cur);
    cur = cur + 1 == STAGES ? 0 : cur + 1;
    nxt = nxt + 1 == STAGES ? 0 : nxt + 1;
  }
  wait_loads<0>();
  lds_barrier();
  for (; s < n_st; ++s) {
    compute(cur);
    cur = cur + 1 == STAGES ? 0 : cur + 1;
  }

  // lane: token l32 of each token block, columns 8 q4 + 4 hf .. + 3 of each
  // column block
#pragma unroll
  for (int m = 0; m < MF; ++m) {
    const int tok = m0 + 32 * (mw * MF + m) + l32;
    if (tok >= a.M) continue;
#pragma unroll
    for (int f = 0; f < NF; f += EPI == PG_SWIGLU ? 2 : 1)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        floatx4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = EPI == PG_SWIGLU ? pg_silu_mul(acc[f][m][4 * q4 + e], acc[f + (NF > 1)][m][4 * q4 + e])
                                  : acc[f][m][4 * q4 + e];
        const int col = 32 * (EPI == PG_SWIGLU ? (ng * NF + f) / 2 : ng * NF + f) + 8 * q4 + 4 * hf;
        if constexpr (EPI == PG_PART) {
          *reinterpret_cast<floatx4 *>(a.part + ((int64_t)sl * a.M + tok) * a.N + n0 + col) = o;
        } else {
          u32x2 *op = reinterpret_cast<u32x2 *>(a.out + (int64_t)tok * a.out_stride + n0 + col);
          if constexpr (EPI == PG_ADD) {
            const u32x2 old = *op;
            o += floatx4{T::lo(old[0]), T::hi(old[0]), T::lo(old[1]), T::hi(old[1])};
          }
          u32x2 v;
          v[0] = pack2<T>(o[0], o[1]);
          v[1] = pack2<T>(o[2], o[3]);
          *op = v;
        }
      }
  }
}

// Sums the K slices' partials into out (ADD: onto its old value), one rounding.
// Bounds: launch latency and one round trip of split + 1 loads.
template <class T, bool ADD>
__global__ __launch_bounds__(256) void prompt_sum_kernel(PromptGemmArgs a) {
  const int64_t i4 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t total = (int64_t)a.M * a.N;
  if (i4 >= total) return;
  floatx4 s = *reinterpret_cast<const floatx4 *>(a.part + i4);
  for (int p = 1; p < a.split; ++p) s += *reinterpret_cast<const floatx4 *>(a.part + p * total + i4);
  const int64_t m = i4 / a.N, n = i4 - m * a.N;
  u32x2 *op = reinterpret_cast<u32x2 *>(a.out + m * a.out_stride + n);
  if (ADD) {
    const u32x2 old = *op;
    s += floatx4{T::lo(old[0]), T::hi(old[0]), T::lo(old[1]), T::hi(old[1])};
  }
  u32x2 v;
  v[0] = pack2<T>(s[0], s[1]);
  v[1] = pack2<T>(s[2], s[3]);
  *op = v;
}

// out += sum of the K slices' partials, normed = RMSNorm(out): a workgroup per
// row, a thread per 16-byte chunk of it, so that every load of a row is in
// flight at once (one wave per row with the row in its registers took 12.4 us
// at 512 x 3072, 5 slices).  The rounded row goes through LDS, from which every
// wave takes the sum of squares in mce_rmsnorm's chunk order (its bits).  Takes
// the place of the sum and of the norm's own launch and read.
constexpr int PG_NORM_MAX = 4096;
template <class T>
__global__ __launch_bounds__(PG_NORM_MAX / 8) void prompt_sum_norm_kernel(PromptGemmArgs a) {
  __shared__ u32x4 row_lds[PG_NORM_MAX / 8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t row = blockIdx.x;
  const int nvec = a.N >> 3, idx = min(tid, nvec - 1);
  const int64_t slice = (int64_t)a.M * a.N / 4;
  u32x4 *const xr = reinterpret_cast<u32x4 *>(a.out + row * a.out_stride);
  const floatx4 *const pr = reinterpret_cast<const floatx4 *>(a.part + row * a.N) + 2 * idx;
  u32x4 v = xr[idx];
  const u32x4 wv = reinterpret_cast<const u32x4 *>(a.norm_w)[idx];
  floatx4 s0 = pr[0], s1 = pr[1];
  for (int p = 1; p < a.split; p += 4) {
    floatx4 t[4][2];
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // slices past the last re-read it
      const floatx4 *const pp = pr + min(p + u, a.split - 1) * slice;
      t[u][0] = pp[0];
      t[u][1] = pp[1];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (p + u < a.split) {
        s0 += t[u][0];
        s1 += t[u][1];
      }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const floatx4 &t = k < 2 ? s0 : s1;
    v[k] = pack2<T>(T::lo(v[k]) + t[2 * (k & 1)], T::hi(v[k]) + t[2 * (k & 1) + 1]);
  }
  if (tid < nvec) {
    xr[tid] = v;
    row_lds[tid] = v;
  }
  lds_barrier();
  float ss = 0.f;
  for (int i = lane; i < nvec; i += 64) ss = sumsq8<T>(row_lds[i], ss);
  const float inv = rms_inv(wave_sum(ss), a.N, a.eps);
  if (tid < nvec) reinterpret_cast<u32x4 *>(a.normed + row * a.N)[tid] = rms_scale8<T>(v, wv, inv);
}

}  // namespace mce

using namespace mce;

namespace {

// Tile of a call.  64 x 64 (two 2-wave workgroups per CU), 128 x 64 (two of 4
// waves), 128 x 128 and 256 x 128 (one of 8): the smallest that covers the
// tokens, up to 256 (in-flight bytes per multiplication, above).  A 256-token
// tile stays ahead of two of 128 for the unsplit gate/up from M = 257 (M = 300:
// 47.6 against 59.6 us, 256 against 384 workgroups), for the split projections
// of long K from M = 385 (M = 300: 37.0 against 33.4; M = 400: 41.3 against
// 41.8); with short K the partials of its five slices cost more than the tile
// saves (o_proj with the norm, M = 385: 28.0 against 22.8, 512 32.2 against 26.1).
struct PromptPlan {
  int bm = 0, bn = 0, mt = 0, nt = 0, split = 1;
};

// The calls this kernel takes; the library GEMM is the better one elsewhere
// (3B shapes, library against this kernel): SwiGLU up to 512 tokens (M = 700: 91
// against 93 us).  The residual add, with the norm behind it on both sides: long
// K up to 768 (down, M = 512 50.4 against 44.4, 520 52.8 against 51.5, 768 66
// against 55; 800 64.2 against 64.2, 896 66.8 against 70.2), short K up to 448
// (o_proj, M = 300 23.5 against 20.5, 384 23.5 against 22.5, 448 24.1 against
// 23.8; 512 24.7 against 26.1).  The plain store up to 128 (M = 176 19.9 against
// 21.5, 280 21.3 against 24), and up to 256 the multiples of 32, where the
// library's time jumps (160 / 192 / 224 / 256: 23.9 / 27.2 / 29.7 / 32.0 against
// 20.5 / 21.9 / 22.7 / 22.6).  None of 16 tokens and fewer (down 15.5 against
// 15.9).  Narrower projections were not measured and stay with the library.
bool prompt_takes(int m, int n, int k, int epilogue) {
  if (m < 17 || n < 1024 || k < 2048 || k % PG_BK != 0 || n % 128 != 0) return false;
  if (epilogue == MCE_EPI_STORE) return m <= 128 || (m <= 256 && m % 32 == 0);
  if (epilogue == MCE_EPI_ADD) return m <= (k >= 6144 ? 768 : 448);
  return m <= 512;
}

PromptPlan prompt_plan(int m, int n, int epilogue, int k) {
  PromptPlan p;
  const bool glu = epilogue == MCE_EPI_SWIGLU;
  if (m <= 64)
    p.bm = p.bn = 64;
  else if (m <= 128)
    p.bm = 128, p.bn = 64;
  else if (m <= (glu ? 256 : k < 6144 ? 448 : 384))
    p.bm = p.bn = 128;
  else
    p.bm = 256, p.bn = 128;
  p.mt = (m + p.bm - 1) / p.bm;
  p.nt = n / (glu ? p.bn / 2 : p.bn);
  // K slices: as many as one workgroup per CU leaves room for (3B shapes, M =
  // 100: down 48 tiles x 5 slices 20.4 us, x 4 20.9; q/k/v 80 x 3 15.1, x 2
  // 16.2), each of at least 6 stages
  if (!glu) p.split = std::max(1, std::min({cu_count() / (p.mt * p.nt), k / PG_BK / 6, 16}));
  return p;
}

template <class T, int EPI>
void launch_tile(const PromptGemmArgs &a, const PromptPlan &p, hipStream_t st) {
  const int grid = (a.nt + 7) / 8 * 8 * a.mt * a.split;
  if (p.bm == 64)
    prompt_gemm_kernel<T, 2, 1, 1, 2, 4, EPI, true, 1><<<grid, 128, 0, st>>>(a);
  else if (p.bm == 128 && p.bn == 64)
    prompt_gemm_kernel<T, 4, 1, 1, 2, 3, EPI, true, 2><<<grid, 256, 0, st>>>(a);
  else if (p.bm == 128)
    prompt_gemm_kernel<T, 4, 1, 2, 2, 4, EPI, false, 2><<<grid, 512, 0, st>>>(a);
  else
    prompt_gemm_kernel<T, 4, 2, 2, 2, 3, EPI, false, 2><<<grid, 512, 0, st>>>(a);
}

template <class T>
int prompt_gemm_launch(int dtype, PromptGemmArgs &a, const PromptPlan &p, int epilogue,
                       hipStream_t st) {
  if (epilogue == MCE_EPI_SWIGLU)
    launch_tile<T, PG_SWIGLU>(a, p, st);
  else if (a.split > 1)
    launch_tile<T, PG_PART>(a, p, st);
  else if (epilogue == MCE_EPI_ADD)
    launch_tile<T, PG_ADD>(a, p, st);
  else
    launch_tile<T, PG_STORE>(a, p, st);
  const bool norm = a.norm_w != nullptr;
  if (norm && a.split > 1 && a.N <= PG_NORM_MAX) {
    prompt_sum_norm_kernel<T><<<a.M, (a.N / 8 + 63) / 64 * 64, 0, st>>>(a);
    return check_launch("mce_prompt_gemm");
  }
  if (a.split > 1) {
    const unsigned grid = (unsigned)(((int64_t)a.M * a.N / 4 + 255) / 256);
    if (epilogue == MCE_EPI_ADD)
      prompt_sum_kernel<T, true><<<grid, 256, 0, st>>>(a);
    else
      prompt_sum_kernel<T, false><<<grid, 256, 0, st>>>(a);
  }
  const int rc = check_launch("mce_prompt_gemm");
  if (rc != MCE_OK || !norm) return rc;
  return mce_rmsnorm(dtype, a.out, a.norm_w, a.normed, a.M, a.N, a.out_stride, a.N, a.eps, st);
}

}  // namespace

extern "C" int mce_prompt_gemm_takes(int m, int n, int k, int epilogue) {
  return prompt_takes(m, n, k, epilogue) ? 1 : 0;
}

extern "C" size_t mce_prompt_gemm_workspace_size(int m, int n, int k, int epilogue) {
  if (!prompt_takes(m, n, k, epilogue)) return 0;
  const PromptPlan p = prompt_plan(m, n, epilogue, k);
  return p.split > 1 ? (size_t)p.split * m * n * sizeof(float) : 0;
}

extern "C" int mce_prompt_gemm(int dtype, const void *x, const void *w, void *out, int m, int n,
                               int k, int64_t x_stride, int64_t out_stride, int epilogue,
                               const void *norm_weight, float eps, void *normed, void *workspace,
                               size_t workspace_bytes, void *stream) {
  clear_error();
  const char *name = "mce_prompt_gemm";
  MCE_REQUIRE(dtype == MCE_F16 || dtype == MCE_BF16, "%s: unknown dtype %d", name, dtype);
  MCE_REQUIRE(epilogue >= MCE_EPI_STORE && epilogue <= MCE_EPI_SWIGLU, "%s: unknown epilogue %d", name,
              epilogue);
  MCE_REQUIRE((norm_weight != nullptr) == (normed != nullptr) &&
                  (!norm_weight || epilogue == MCE_EPI_ADD),
              "%s: the norm goes with the residual add", name);
  constexpr int64_t LIM = (int64_t)1 << 31;  // bytes behind a 32-bit offset
  if (!prompt_takes(m, n, k, epilogue) || x_stride < k || x_stride % 8 != 0 || out_stride < n ||
      out_stride % 8 != 0 || x_stride >= LIM || out_stride >= LIM || x_stride * m * 2 >= LIM ||
      (int64_t)n * k * 2 * (epilogue == MCE_EPI_SWIGLU ? 2 : 1) >= LIM)
    return set_error(MCE_ERR_UNSUPPORTED, "%s: m=%d n=%d k=%d is left to the library GEMM", name, m, n, k);
  MCE_REQUIRE(x && w && out, "%s: null pointer", name);
  if (!aligned16(x) || !aligned16(w) || !aligned16(out) || !aligned16(norm_weight) || !aligned16(normed))
    return set_error(MCE_ERR_UNSUPPORTED, "%s: operands must be 16-byte aligned", name);
  const PromptPlan p = prompt_plan(m, n, epilogue, k);
  const size_t need = mce_prompt_gemm_workspace_size(m, n, k, epilogue);
  if (need > 0 && (workspace == nullptr || workspace_bytes < need ||
                   (reinterpret_cast<uintptr_t>(workspace) & 255) != 0))
    return set_error(MCE_ERR_WORKSPACE, "%s: a 256-byte aligned workspace of %zu bytes is required",
                     name, need);
  PromptGemmArgs a{};
  a.x = (const uint16_t *)x;
  a.w = (const uint16_t *)w;
  a.out = (uint16_t *)out;
  a.part = (float *)workspace;
  a.M = m;
  a.N = n;
  a.K = k;
  a.x_stride = (int)x_stride;
  a.out_stride = (int)out_stride;
  a.x_bytes = (int)(((int64_t)(m - 1) * x_stride + k) * 2);
  a.w_bytes = (int)((int64_t)n * k * 2 * (epilogue == MCE_EPI_SWIGLU ? 2 : 1));
  a.mt = p.mt;
  a.nt = p.nt;
  a.split = p.split;
  a.norm_w = (const uint16_t *)norm_weight;
  a.normed = (uint16_t *)normed;
  a.eps = eps;
  hipStream_t st = (hipStream_t)stream;
  return dtype == MCE_F16 ? prompt_gemm_launch<F16T>(dtype, a, p, epilogue, st)
                          : prompt_gemm_launch<BF16T>(dtype, a, p, epilogue, st);
}

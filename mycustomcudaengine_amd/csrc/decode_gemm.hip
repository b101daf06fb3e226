// Decode-sized GEMM for gfx950: out[M, N] (op)= xn[M, K] . W[N, K]^T with
// M <= 16 (one token per sequence), fp16 in, fp32 accumulation; xn is x or
// RMSNorm(x) (fused in front), and the epilogue stores, adds into the
// residual stream or applies SwiGLU.  This is the projection work of the
// engine's decode step (engine/models/llama.py:94-174 runs it through
// torch.matmul with separate RMSNorm and SwiGLU kernels); at these shapes it
// is a weight-streaming problem: every W byte is read once and the MFMA work
// is negligible.
//
// Layout of one launch (grid = N / columns per workgroup, 8 waves each):
//   * a workgroup owns TT tiles of R <= 16 output columns (R rows of W each;
//     SwiGLU: gate rows j and up rows n + j); wave w takes the K slice
//     [w K / 8, (w + 1) K / 8) as C = K / 256 chunks of 32;
//   * x is staged in LDS as the MFMA B operand: 16-byte groups of 8
//     consecutive k, [k / 8][token slot], swizzled (xs_group) so that the
//     staging writes and the fragment reads spread over the banks.  Without
//     the norm each wave stages its own K slice of every token (whole 128-byte
//     lines, no workgroup barrier: nobody else reads it); with the norm each
//     wave stages whole token rows, whose scale needs the full row;
//   * every load instruction of W reads 8 rows x 128 contiguous bytes, 8
//     consecutive lanes per row.  In the MFMA operand pattern (lane l: row
//     l % 16, 16 rows x 64 bytes) each group of four lanes touches four cache
//     lines, and the address path, not HBM, sets the rate.  A chunk pair (64
//     k) then goes through a 2 KB wave-private LDS buffer (XOR-swizzled:
//     conflict-free writes of 8 rows and reads of 16) to become two A
//     fragments;
//   * the loads are non-temporal: no weight byte is used twice in a step, and
//     whole lines stream 5-10% faster that way (in the 64-byte pattern they
//     were 10% slower: the second half of a line came from HBM again);
//   * the x loads go out first (loads return in order, so staging x waits for
//     x only), then the W loads -- all of them, or as many as the registers
//     hold beside x, the rest once x is staged -- so that with every workgroup
//     of a launch resident the whole weight is in flight at once;
//   * one v_mfma_f32_16x16x32_f16 per chunk and tile.  Up to 8 tokens fill
//     half of the 16 operand columns, so one x fragment carries chunk c in
//     columns 0-7 and chunk c + 1 in columns 8-15, and the two chunks
//     accumulate apart, each using its own half (the other half's sums, and
//     those of slots past M, are never read);
//   * the 8 K-slice partials are summed through LDS by one thread per output,
//     consecutive threads on consecutive columns, which apply the epilogue:
//       STORE  out[m, n] = acc
//       ADD    out[m, n] = out[m, n] + acc          (residual stream, in place;
//              the old value is loaded with x, off the kernel's tail)
//       SWIGLU out[m, j] = silu(acc_gate) * acc_up  (W = [2 n, K], gate rows first)
// The fused RMSNorm computes each token's scale exactly as mce_rmsnorm does
// (same per-lane chunk order, reduction and rounding), so xn is bit-identical
// to that op's output.
//
// What bounds it (MI355X, 8 tokens, weights from HBM, us per call in graphs of
// back-to-back calls, previous kernel -> this one): about 2 us of launch, 1 us
// to the first bytes, the stream at 6.2-7 TB/s and 1 us of tail.  q/k/v (31 MB)
// 8.7 -> 8.5, o_proj (19 MB) 6.9 -> 5.8, gate/up (101 MB) 20.7 -> 18.9, down
// (50 MB) 13.9 -> 11.9, lm_head (788 MB) 134.6 -> 121.4; one token: 8.1 ->
// 7.6, 5.9 -> 5.5, 19.3 -> 17.7, 12.4 -> 11.6, 125.4 -> 113.8.
#include "mce_common.h"

namespace mce {

constexpr int DG_WAVES = 8;

struct DecodeGemmArgs {
  const uint16_t *x, *w, *norm_w;
  uint16_t *out;
  int M, N;
  int64_t x_stride, out_stride;
  float eps;
};

// 16-byte group index of k group kg, token slot t in the staged x.  8 slots:
// the k groups of a fragment read's two column halves (4 apart) land in
// different halves of the banks.
template <int MP>
__device__ __forceinline__ int xs_group(int kg, int t) {
  if constexpr (MP == 16)
    return kg * 16 + (t ^ (kg & 15));
  else
    return (kg ^ ((kg >> 2) & 1)) * 8 + (t ^ ((kg >> 1) & 7));
}

__device__ __forceinline__ float silu_mul(float g, float u) {
  return g / (1.0f + __expf(-g)) * u;
}
__device__ __forceinline__ u32x4 ld_w(const uint16_t *p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
}

// A wave's own LDS operations complete in order: only the compiler has to keep
// the order of its writes and reads.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// EPI: 0 store, 1 add, 2 SwiGLU; TT tiles per workgroup (SwiGLU: half of them
// gate, half up tiles); MP token slots (8 or 16); NORM: fuse RMSNorm; C chunks
// of 32 k per wave; R output columns per tile (16, 12, 10 or 8: rows past R
// re-read row R - 1 and their results are dropped), so that the grid can be
// sized to a whole number of workgroups per CU.
// LOOP: the workgroup keeps its staged x and walks a contiguous range of
// tiles, each chunk pair's registers refilled for the next tile as soon as
// they are consumed.
template <int EPI, int TT, int MP, bool NORM, int C, int WPE, int R, bool LOOP>
__global__ __launch_bounds__(DG_WAVES * 64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void decode_gemm_kernel(DecodeGemmArgs a) {
  static_assert(R % 2 == 0 && R >= 8 && R <= 16, "tile rows");
  constexpr int K = C * 256;
  constexpr int XP = MP == 8 ? 2 : 1;  // chunks per x fragment
  constexpr int VPT = K / 512;         // 16-byte groups of a token slot's x per lane
  constexpr int NTOK = MP / 8;         // token slots staged per wave
  // W chunks fetched before x is staged: all that fit beside x (and the norm
  // weights) at the occupancy target
  constexpr int NXR = NTOK * VPT + (NORM ? VPT : 0);
  constexpr int BUDGET = (512 / WPE - 28) / 4 - NXR;
  constexpr int C1 = BUDGET >= TT * C ? C : (BUDGET / TT) / 2 * 2;
  constexpr int WXW = TT > 2 ? TT * 256 : 512;  // words per wave: a chunk pair of W, then the partial sums
  __shared__ __attribute__((aligned(16))) uint16_t xs[K / 8 * MP * 8];
  __shared__ __attribute__((aligned(16))) uint32_t wx[DG_WAVES * WXW];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int NT = EPI == 2 ? TT / 2 : TT;  // output tiles
  const int r = lane & 15, q = lane >> 4;
  const int l8 = lane >> 3, k8 = lane & 7;  // row and k group of a 128-byte-row load

  // 1. x (and the norm weights)
  u32x4 xv[NTOK][VPT], nw[NORM ? VPT : 1];
#pragma unroll
  for (int j = 0; j < NTOK; ++j)
    if constexpr (NORM) {
      const int m = wave + 8 * j;
      if (m < a.M) {
        const uint16_t *xr = a.x + (int64_t)m * a.x_stride;
#pragma unroll
        for (int i = 0; i < VPT; ++i) xv[j][i] = *reinterpret_cast<const u32x4 *>(xr + (lane + 64 * i) * 8);
      }
    } else {
      const uint16_t *xr = a.x + (int64_t)min(l8 + 8 * j, a.M - 1) * a.x_stride + wave * (K / 8) + 8 * k8;
#pragma unroll
      for (int i = 0; i < VPT; ++i) xv[j][i] = *reinterpret_cast<const u32x4 *>(xr + 64 * i);
    }
  if constexpr (NORM) {
    if (wave < a.M) {
#pragma unroll
      for (int i = 0; i < VPT; ++i) nw[i] = *reinterpret_cast<const u32x4 *>(a.norm_w + (lane + 64 * i) * 8);
    }
  }
  // 2. W: load c of a tile reads rows 8 (c & 1) .. +7 of its 16 at chunk pair
  // c / 2
  u32x4 wf[TT][C];
  const uint16_t *wp[TT][2];
  auto set_tile = [&](int col0) {
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int trow = EPI == 2 ? (t % NT) * R + (t / NT) * a.N : t * R;
        wp[t][h] = a.w + (int64_t)(col0 + trow + min(l8 + 8 * h, R - 1)) * K + wave * (K / 8) + 8 * k8;
      }
  };
  auto load_w = [&](int lo, int hi) {
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (c >= lo && c < hi) {
#pragma unroll
        for (int t = 0; t < TT; ++t) wf[t][c] = ld_w(wp[t][c & 1] + 64 * (c >> 1));
      }
  };
  const int n_tiles = a.N / (R * NT);
  int tile = LOOP ? (int)((int64_t)blockIdx.x * n_tiles / gridDim.x) : (int)blockIdx.x;
  const int tile_end = LOOP ? (int)((int64_t)(blockIdx.x + 1) * n_tiles / gridDim.x) : tile + 1;
  set_tile(tile * (R * NT));
  // the output a thread finishes: column oc, token om, tiles ot + OTS p
  const int oc = tid & 15, om = (tid >> 4) & (MP - 1), ot = tid / (16 * MP);
  constexpr int OTS = DG_WAVES * 64 / (16 * MP);
  constexpr int OPT = (NT + OTS - 1) / OTS;
  uint16_t old[OPT];
  if constexpr (EPI == 1) {
#pragma unroll
    for (int p = 0; p < OPT; ++p) {
      const int t = min(ot + p * OTS, NT - 1);
      old[p] = a.out[(int64_t)min(om, a.M - 1) * a.out_stride + tile * (R * NT) + t * R +
                     min(oc, R - 1)];
    }
  }
  load_w(0, C1);
  // keep these loads ahead of the staging below (the scheduler would
  // otherwise sink most of them past it to save registers)
  __builtin_amdgcn_sched_barrier(0);

  // 3. stage x (normalised) into LDS; slots past M stay as they are
#pragma unroll
  for (int j = 0; j < NTOK; ++j) {
    if constexpr (NORM) {
      const int m = wave + 8 * j;
      if (m < a.M) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < VPT; ++i) ss = sumsq8<F16T>(xv[j][i], ss);
        const float inv = rms_inv(wave_sum(ss), K, a.eps);
#pragma unroll
        for (int i = 0; i < VPT; ++i)
          *reinterpret_cast<u32x4 *>(&xs[xs_group<MP>(lane + 64 * i, m) * 8]) = rms_scale8<F16T>(xv[j][i], nw[i], inv);
      }
    } else {
#pragma unroll
      for (int i = 0; i < VPT; ++i)
        *reinterpret_cast<u32x4 *>(&xs[xs_group<MP>(wave * (C * 4) + 8 * i + k8, l8 + 8 * j) * 8]) = xv[j][i];
    }
  }
  load_w(C1, C);
  if constexpr (NORM) lds_barrier();
  else wave_lds_fence();

  // 4. the MFMAs.  This lane's write slot (row l / 8 + 8 h, k group l % 8) and
  // read slot (row l % 16, k group 4 hh + l / 16) in the swizzled pair buffer:
  // row pitch 128 bytes, k group g of row p at group g ^ ((p >> 1) & 7)
  uint32_t *const wxw = wx + wave * WXW;
  auto wslot = [&](int h) {
    const int p = l8 + 8 * h;
    return p * 32 + 4 * (k8 ^ ((p >> 1) & 7));
  };
  auto rslot = [&](int hh) { return r * 32 + 4 * ((4 * hh + q) ^ ((r >> 1) & 7)); };
  for (;;) {
    floatx4 acc[TT][XP];
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int p = 0; p < XP; ++p) acc[t][p] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (LOOP) set_tile(min(tile + 1, tile_end - 1) * (R * NT));
#pragma unroll
    for (int c = 0; c < C; c += 2) {
      u32x4 xg[2];
#pragma unroll
      for (int hh = 0; hh < 2 / XP; ++hh) {
        const int kg = (wave * C + c + hh + (MP == 8 ? r >> 3 : 0)) * 4 + q;
        xg[hh] = *reinterpret_cast<const u32x4 *>(&xs[xs_group<MP>(kg, r & (MP - 1)) * 8]);
      }
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        u32x4 f[2];
        *reinterpret_cast<u32x4 *>(wxw + wslot(0)) = wf[t][c];
        *reinterpret_cast<u32x4 *>(wxw + wslot(1)) = wf[t][c + 1];
        wave_lds_fence();
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) f[hh] = *reinterpret_cast<const u32x4 *>(wxw + rslot(hh));
        wave_lds_fence();
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
          acc[t][XP == 2 ? hh : 0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(half8, f[hh]), __builtin_bit_cast(half8, xg[XP == 2 ? 0 : hh]),
              acc[t][XP == 2 ? hh : 0], 0, 0, 0);
      }
      if constexpr (LOOP) load_w(c, c + 2);
    }
    // 5. partial sums of this wave's K slice, in its own part of wx: component i
    // of lane l at 64 i + (l ^ 4 i)
    float *const red = reinterpret_cast<float *>(wxw);
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        red[(t * 4 + i) * 64 + (lane ^ (4 * i))] = XP == 2 ? (r < 8 ? acc[t][0][i] : acc[t][XP - 1][i]) : acc[t][0][i];
    lds_barrier();
    const int ri = oc & 3, rl = (16 * (oc >> 2) + om) ^ (4 * ri);
    auto total = [&](int t) {
      float s = 0.f;
#pragma unroll
      for (int sl = 0; sl < DG_WAVES; ++sl) {
        const float *p = reinterpret_cast<const float *>(wx + sl * WXW) + (t * 4 + ri) * 64;
        s += p[rl];
        if constexpr (XP == 2) s += p[rl ^ 8];
      }
      return s;
    };
#pragma unroll
    for (int p = 0; p < OPT; ++p) {
      const int t = ot + p * OTS;
      if (t < NT && oc < R && om < a.M) {
        float o;
        if constexpr (EPI == 2) o = silu_mul(total(t), total(t + NT));
        else o = total(t);
        if constexpr (EPI == 1) o += F16T::lo(old[p]);
        a.out[(int64_t)om * a.out_stride + tile * (R * NT) + t * R + oc] = F16T::from_float(o);
      }
    }
    if (!LOOP || ++tile >= tile_end) return;
    lds_barrier();  // the sums are read before the next tile's W goes through wx
  }
}

template <int EPI, int TT, int MP, bool NORM, int C, int R>
void launch_dg(const DecodeGemmArgs &a, hipStream_t st) {
  // registers of the W fragments decide how many waves fit per SIMD; every
  // workgroup of a launch should be resident at once
  constexpr int WPE = TT * C <= 24 && MP == 8 ? 4 : 2;
  const int grid = a.N / (EPI == 2 ? R * TT / 2 : R * TT);
  // Many rounds of workgroups (lm_head: 8016 over 256 CUs).  With 16 token
  // slots staging x (and its norm) costs a workgroup as much as streaming its
  // tile: one workgroup per CU keeps x and walks its tiles, 199 -> 129 us at 16
  // tokens.  With 8 slots the dispatcher's turnover of two workgroups per CU
  // overlaps the staging and is the faster form (121 against 124-128 us).
  if constexpr (EPI == 0 && TT == 1 && R == 16 && MP == 16) {
    if (grid >= 8 * cu_count()) {
      decode_gemm_kernel<EPI, TT, MP, NORM, C, WPE, R, true><<<cu_count(), DG_WAVES * 64, 0, st>>>(a);
      return;
    }
  }
  decode_gemm_kernel<EPI, TT, MP, NORM, C, WPE, R, false><<<grid, DG_WAVES * 64, 0, st>>>(a);
}

template <int EPI, int TT, int MP, bool NORM, int R>
int dispatch_k(const DecodeGemmArgs &a, int k, hipStream_t st) {
  switch (k) {
    case 2048: launch_dg<EPI, TT, MP, NORM, 8, R>(a, st); return MCE_OK;
    case 3072: launch_dg<EPI, TT, MP, NORM, 12, R>(a, st); return MCE_OK;
    case 4096: launch_dg<EPI, TT, MP, NORM, 16, R>(a, st); return MCE_OK;
    case 8192:
      if constexpr (TT == 1 && !NORM && MP == 8) {  // 128 KB of staged x
        launch_dg<EPI, TT, MP, NORM, 32, R>(a, st);
        return MCE_OK;
      }
      break;
  }
  return MCE_ERR_UNSUPPORTED;
}

// Output columns per workgroup: R columns per tile times TT tiles (SwiGLU: R
// gate / up column pairs).  The widest tile is kept unless a narrower one
// cuts the columns of the busiest CU (whole rounds of workgroups over the
// CUs times the columns per workgroup) by more than 10%: 3072 columns run as
// 256 workgroups of 12, 5120 as 256 of 2 x 10, instead of 192 / 320 of 16.
struct DgTile {
  int r, tt;
};

DgTile pick_tile(int n, bool swiglu, int k) {
  static const DgTile plain[] = {{16, 1}, {12, 1}, {10, 2}, {8, 1}};
  static const DgTile glu[] = {{16, 2}, {8, 2}};
  const int64_t cus = cu_count();
  DgTile best = swiglu ? glu[0] : plain[0];
  int64_t best_cost = -1;
  const DgTile *cand = swiglu ? glu : plain;
  const int n_cand = swiglu ? 2 : 4;
  for (int i = 0; i < n_cand; ++i) {
    const DgTile &t = cand[i];
    if (t.tt == 2 && !swiglu && k == 8192) continue;  // one tile only at k = 8192
    const int cols = swiglu ? t.r : t.r * t.tt;
    if (n % cols != 0) continue;
    const int64_t cost = ((n / cols) + cus - 1) / cus * cols;
    if (best_cost < 0 || 10 * cost < 9 * best_cost) {
      best = t;
      best_cost = cost;
    }
  }
  return best;
}

template <int EPI, int MP, bool NORM>
int dispatch_tile(const DecodeGemmArgs &a, int k, const DgTile &t, hipStream_t st) {
  if constexpr (EPI == 2) {
    return t.r == 8 ? dispatch_k<EPI, 2, MP, NORM, 8>(a, k, st) : dispatch_k<EPI, 2, MP, NORM, 16>(a, k, st);
  } else {
    switch (t.r) {
      case 12: return dispatch_k<EPI, 1, MP, NORM, 12>(a, k, st);
      case 10: return dispatch_k<EPI, 2, MP, NORM, 10>(a, k, st);
      case 8: return dispatch_k<EPI, 1, MP, NORM, 8>(a, k, st);
      default: return dispatch_k<EPI, 1, MP, NORM, 16>(a, k, st);
    }
  }
}

template <bool NORM>
int dispatch(const DecodeGemmArgs &a, int k, int epilogue, hipStream_t st) {
  const bool small = a.M <= 8;
  const DgTile t = pick_tile(a.N, epilogue == MCE_EPI_SWIGLU, k);
  if (epilogue == MCE_EPI_STORE)
    return small ? dispatch_tile<0, 8, NORM>(a, k, t, st) : dispatch_tile<0, 16, NORM>(a, k, t, st);
  if (epilogue == MCE_EPI_ADD)
    return small ? dispatch_tile<1, 8, NORM>(a, k, t, st) : dispatch_tile<1, 16, NORM>(a, k, t, st);
  return small ? dispatch_tile<2, 8, NORM>(a, k, t, st) : dispatch_tile<2, 16, NORM>(a, k, t, st);
}

int decode_gemm_impl(const char *name, int dtype, const void *x, const void *norm_w, float eps,
                     const void *w, void *out, int m, int n, int k, int64_t x_stride,
                     int64_t out_stride, int epilogue, void *stream) {
  clear_error();
  MCE_REQUIRE(dtype == MCE_F16 || dtype == MCE_BF16, "%s: unknown dtype %d", name, dtype);
  if (dtype != MCE_F16) return set_error(MCE_ERR_UNSUPPORTED, "%s: only fp16 is implemented", name);
  MCE_REQUIRE(epilogue >= MCE_EPI_STORE && epilogue <= MCE_EPI_SWIGLU, "%s: unknown epilogue %d",
              name, epilogue);
  MCE_REQUIRE(m >= 0 && n >= 0 && k >= 0, "%s: bad shape", name);
  if (m == 0 || n == 0) return MCE_OK;
  const bool norm = norm_w != nullptr;
  const bool k_ok = k == 2048 || k == 3072 || k == 4096 ||
                    (k == 8192 && !norm && epilogue != MCE_EPI_SWIGLU && m <= 8);
  if (m > 16 || n % 16 != 0 || !k_ok)
    return set_error(MCE_ERR_UNSUPPORTED,
                     "%s: needs m <= 16, n %% 16 == 0 and k in {2048, 3072, 4096} (8192 for m <= 8 "
                     "without the fused RMSNorm or SwiGLU) (got m=%d n=%d k=%d)",
                     name, m, n, k);
  MCE_REQUIRE(x && w && out, "%s: null pointer", name);
  MCE_REQUIRE(x_stride >= k && x_stride % 8 == 0 && out_stride >= n && out_stride % 4 == 0,
              "%s: bad row strides", name);
  MCE_REQUIRE(aligned16(x) && aligned16(w) && (!norm || aligned16(norm_w)) &&
                  (reinterpret_cast<uintptr_t>(out) & 7) == 0,
              "%s: x, w and the norm weight must be 16-byte aligned, out 8-byte aligned", name);
  {
    // every workgroup reads all of x while others already write their
    // columns of out: the two must not overlap
    const uintptr_t x0 = reinterpret_cast<uintptr_t>(x), o0 = reinterpret_cast<uintptr_t>(out);
    const uintptr_t x1 = x0 + (uintptr_t)(((int64_t)(m - 1) * x_stride + k) * 2);
    const uintptr_t o1 = o0 + (uintptr_t)(((int64_t)(m - 1) * out_stride + n) * 2);
    MCE_REQUIRE(x1 <= o0 || o1 <= x0, "%s: out must not overlap x", name);
  }
  MCE_REQUIRE((int64_t)n * k * (epilogue == MCE_EPI_SWIGLU ? 2 : 1) < ((int64_t)1 << 31),
              "%s: weight too large", name);
  DecodeGemmArgs a{};
  a.x = (const uint16_t *)x;
  a.w = (const uint16_t *)w;
  a.norm_w = (const uint16_t *)norm_w;
  a.out = (uint16_t *)out;
  a.M = m;
  a.N = n;
  a.x_stride = x_stride;
  a.out_stride = out_stride;
  a.eps = eps;
  hipStream_t st = (hipStream_t)stream;
  const int rc = norm ? dispatch<true>(a, k, epilogue, st) : dispatch<false>(a, k, epilogue, st);
  if (rc != MCE_OK) return set_error(rc, "%s: no kernel for k=%d", name, k);
  return check_launch(name);
}

}  // namespace mce

using namespace mce;

extern "C" int mce_decode_gemm(int dtype, const void *x, const void *w, void *out, int m, int n,
                               int k, int64_t x_stride, int64_t out_stride, int epilogue,
                               void *stream) {
  return decode_gemm_impl("mce_decode_gemm", dtype, x, nullptr, 0.f, w, out, m, n, k, x_stride,
                          out_stride, epilogue, stream);
}

extern "C" int mce_rmsnorm_decode_gemm(int dtype, const void *x, const void *norm_weight,
                                       float eps, const void *w, void *out, int m, int n, int k,
                                       int64_t x_stride, int64_t out_stride, int epilogue,
                                       void *stream) {
  clear_error();
  MCE_REQUIRE(norm_weight != nullptr, "mce_rmsnorm_decode_gemm: null norm weight");
  MCE_REQUIRE(eps >= 0.f, "mce_rmsnorm_decode_gemm: eps must be >= 0");
  return decode_gemm_impl("mce_rmsnorm_decode_gemm", dtype, x, norm_weight, eps, w, out, m, n, k,
                          x_stride, out_stride, epilogue, stream);
}

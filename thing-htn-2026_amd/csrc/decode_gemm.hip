// Decode projections at M <= 32 rows as weight streams through a ring of LDS stages.
//
// Operator, epilogues and rounding points as gemm.hip (engine/kernels/gemm.py:12-15, gemm_fused.py:5-19,
// :179-193): out = x @ W^T with optional RMSNorm of x, and a plain, residual (with the next norm's partial sums
// of squares) or SwiGLU epilogue, over the MFMA-B tiles of weights.hip.
//
// A step reads each weight once, so a launch is bound by HBM: a plain stream of these direct global -> LDS loads
// takes 2.4 us plus the bytes at 7.5 TB/s. 160 to 200 CUs reach that rate, so a workgroup takes NT whole n-tiles over
// all of k (at most one workgroup per CU: 160 for O, 192 for QKV, 203 for gate/up) and no partial sum leaves its
// workgroup. Its 8 wavefronts split a stage's 32-k steps KW ways and its n-tiles CW ways; weights and activations
// both come through the ring, with at least 256 bytes of an activation row per load (the 64-byte row pieces that
// gemm.hip's fragment loads ask for run at half the L1's rate), and the RMSNorm of an activation fragment is
// formed once per workgroup (CW times). Wavefront partials are summed through LDS in k order.
//
// us per launch, graph-replayed over 8 - 16 weight copies, before (gemm.hip's best shape) -> here:
//             M = 3            M = 8            M = 16           M = 20           M = 32
//   QKV       8.4 -> 8.3       8.8 -> 8.5       9.8 -> 9.0       11.8 -> 10.1     13.5 -> 10.7
//   O         7.3 -> 6.4       7.4 -> 7.1       8.7 -> 7.8       10.2 -> 8.7      11.2 -> 9.5
//   gate/up   20.6 -> 20.0     20.5 -> 19.4     23.5 -> 19.7     25.0 -> 20.9     25.1 -> 21.1
// The down projection (k = 9728) stays with gemm.hip's split of k in three, 240 workgroups: here 160 would each move
// its 311 KB of weights and M / 16 times that of activations, while 96 CUs idle. 12.1 -> 12.5 us at M = 8, 12.4 -> 14.7
// at 16, 16.5 -> 18.6 at 32 (and 12.0 -> 11.3 at 3).
#include "common.h"
#include "lds_ring.h"

namespace {

enum { EPI_STORE = 0, EPI_RES = 1, EPI_SWIGLU = 2 };

typedef unsigned du4 __attribute__((ext_vector_type(4)));

struct DecodeGemmParams {
  const bf16_t* x;      // [M, K] row-major
  const bf16_t* w;      // MFMA-B tiled weight, N x K
  const bf16_t* nw;     // [K] RMSNorm gain (NORM)
  const bf16_t* res;    // [M, ld_out] residual (EPI_RES; may alias out)
  bf16_t* out;          // [M, ld_out]
  const float* psq_in;  // [M, K/16] partial sums of squares of x per 16 columns (NORM)
  float* psq_out;       // [M, N/16] same for the output rows (EPI_RES, may be null)
  int M, N, K, ld_out;
  float eps;
};

constexpr int DG_WAVES = 8;

// LDS: S stages [A: 16 MT rows x KW x 64 bytes | W: NT x KW tiles of 1 KB], the residual tile, the RMSNorm
// factors, and (NORM) the gain. Every wavefront loads a share of both (measured: four wavefronts for W and four
// for A, with stage counts of their own: up to 27 % slower).
constexpr int dg_stage(int MT, int NT, int KW) { return (MT + NT) * KW * 1024; }
constexpr int dg_res(int MT, int NT) { return MT * NT * 512; }
constexpr long long dg_lds(int MT, int NT, int KW, int S, int K, bool norm) {
  return (long long)S * dg_stage(MT, NT, KW) + dg_res(MT, NT) + 128 + (norm ? 2ll * K : 0);
}

template <int MT, int NT, int KW, int CW, int S, bool NORM, int EPI>
__global__ void __launch_bounds__(64 * DG_WAVES, 1) decode_gemm_kernel(DecodeGemmParams p) {
  static_assert(KW * CW == DG_WAVES && NT % CW == 0 && (EPI != EPI_SWIGLU || NT % 2 == 0), "wavefront split");
  constexpr int NTW = NT / CW;             // n-tiles of a wavefront
  constexpr int C = 4 * KW;                // 16-byte chunks of a staged A row; chunk c of row r at c ^ (r % 16)
  constexpr int ABYTES = MT * KW * 1024, STAGE = dg_stage(MT, NT, KW);
  constexpr int PA = (MT * KW + DG_WAVES - 1) / DG_WAVES, PW = NT * KW / DG_WAVES, PER = PA + PW;
  static_assert(NT * KW % DG_WAVES == 0 && KW * MT * NT * 1024 <= S * STAGE, "stage split");
  extern __shared__ __align__(16) unsigned char dg_smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wave % KW, cw = wave / KW;
  const int qq = lane >> 4, rr = lane & 15;
  const int KT = p.K / 32, G = KT / KW;    // G stages
  const int nt0 = (int)blockIdx.x * NT;    // the workgroup's first n-tile
  bf16_t* res_s = reinterpret_cast<bf16_t*>(dg_smem + S * STAGE);                       // [16 MT][16 NT]
  float* rinv_s = reinterpret_cast<float*>(dg_smem + S * STAGE + dg_res(MT, NT));       // [32]
  uint4* gain_s = reinterpret_cast<uint4*>(dg_smem + S * STAGE + dg_res(MT, NT) + 128);  // [K / 8]
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)dg_smem;

  // ---- RMSNorm inputs, requested before the ring's loads (loads return in issue order): this
  // wavefront's rows' partial sums and a piece of the gain
  constexpr int RPW = MT * 16 / DG_WAVES;  // rows whose factor a wavefront derives
  constexpr int GV = 2;                    // gain pieces per thread kept in registers (K <= 8192)
  float ss[NORM ? RPW : 1];
  du4 gv[NORM ? GV : 1];
  if constexpr (NORM) {
    const int n4 = p.K >> 6;               // float4 pieces of a row's partial sums
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int m = min(wave + i * DG_WAVES, p.M - 1);
      const f32x4_t* ps = reinterpret_cast<const f32x4_t*>(p.psq_in + (size_t)m * (p.K >> 4));
      float s = 0.f;
      for (int c = lane; c < n4; c += 64) {
        const f32x4_t v = ps[c];
        s += (v.x + v.y) + (v.z + v.w);
      }
      ss[i] = s;
    }
#pragma unroll
    for (int i = 0; i < GV; ++i) gv[i] = reinterpret_cast<const du4*>(p.nw)[min(tid + i * 64 * DG_WAVES, p.K / 8 - 1)];
  }

  // ---- the ring. W tile t (n-tile t / KW, k-step t % KW) = PW wave + i; A block b (1 KB of the stage's rows) =
  // PA wave + i, past the last block the last one again (the same bytes to the same place). Rows past M re-read
  // row M - 1 and are never stored. 32-bit offsets: checked by the host.
  const char* abase = reinterpret_cast<const char*>(p.x);
  const char* wbase = reinterpret_cast<const char*>(p.w) + (long long)nt0 * KT * 1024;
  unsigned avoff[PA], wvoff[PW];
  int ablk[PA];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    ablk[i] = min(wave * PA + i, MT * KW - 1);
    const int s = ablk[i] * 64 + lane, row = s / C, pc = s % C;
    avoff[i] = (unsigned)min(row, p.M - 1) * (unsigned)(p.K * 2) + (unsigned)((pc ^ (row & 15)) * 16);
  }
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int t = wave * PW + i, n = min(t / KW, p.N / 16 - 1 - nt0);   // (tiles past N: the last one again)
    wvoff[i] = (unsigned)(n * KT + t % KW) * 1024u + lane * 16u;
  }
  auto issue = [&](int g) __attribute__((always_inline)) {   // the next stage, g, into slot g % S
    const unsigned sb = lds0 + (g % S) * STAGE;
#pragma unroll
    for (int i = 0; i < PW; ++i) ring_load16_nt(wbase, wvoff[i], sb + ABYTES + (wave * PW + i) * 1024);
#pragma unroll
    for (int i = 0; i < PA; ++i) ring_load16(abase, avoff[i], sb + ablk[i] * 1024);
    abase += KW * 64;
    wbase += KW * 1024;
  };

  // residual tile -> LDS (two columns per lane; read straight from memory at the end if it is not 4-byte aligned)
  const bool res_lds = EPI == EPI_RES && (((uintptr_t)p.res | (uintptr_t)(p.ld_out * 2)) & 3) == 0;
  if (res_lds) {
    constexpr int PAIRS = NT * 8;          // 4-byte pieces per row
    for (int i = wave; i < MT * NT * 2; i += DG_WAVES) {
      const int d = i * 64 + lane, row = min(d / PAIRS, p.M - 1);
      ring_load4(p.res + nt0 * 16, (unsigned)row * (unsigned)(p.ld_out * 2) + (unsigned)(d % PAIRS) * 4u,
                 lds0 + S * STAGE + i * 256);
    }
  }
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < G) issue(s);

  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const float t = wave_sum_dpp(ss[i]);
      if (lane == 0) rinv_s[wave + i * DG_WAVES] = rms_rinv(t, p.K, p.eps);
    }
#pragma unroll
    for (int i = 0; i < GV; ++i)
      if (tid + i * 64 * DG_WAVES < p.K / 8) reinterpret_cast<du4*>(gain_s)[tid + i * 64 * DG_WAVES] = gv[i];
  }

  f32x4_t acc[MT][NTW];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[mt][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float rinv[MT];
  for (int g = 0; g < G; ++g) {
    ring_wait_stages<PER, S - 2>(G - 1 - g);   // stage g has landed, later ones may be in flight
    __syncthreads();                           // for every wavefront; and stage g - 1's slot is free
    if (g + S - 1 < G) issue(g + S - 1);
    if constexpr (NORM) {
      if (g == 0) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) rinv[mt] = rinv_s[mt * 16 + rr];
      }
    }
    const uint4* st = reinterpret_cast<const uint4*>(dg_smem + (g % S) * STAGE);
    uint4 a[MT], b[NTW], gn;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) a[mt] = st[(mt * 16 + rr) * C + ((4 * kw + qq) ^ rr)];
    if constexpr (NORM) gn = gain_s[(g * KW + kw) * 4 + qq];
#pragma unroll
    for (int j = 0; j < NTW; ++j) b[j] = st[ABYTES / 16 + ((cw * NTW + j) * KW + kw) * 64 + lane];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if constexpr (NORM) {   // bf16(bf16(x * rinv) * gain)
        float f[8], gf[8];
        unpack8(a[mt], f);
        unpack8(gn, gf);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = mul_rn(gf[e], rbf(mul_rn(f[e], rinv[mt])));
        a[mt] = pack8(f);
      }
#pragma unroll
      for (int j = 0; j < NTW; ++j)
        acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[mt]), as_bf16x8(b[j]), acc[mt][j], 0, 0, 0);
    }
  }

  // ---- sum the k parts (in order) through LDS and store. Fragment (mt, n) of the k part kw at
  // ((kw MT + mt) NT + n) KB; wavefront w finishes fragments (SwiGLU: gate / up pairs) w, w + 8, ..
  __syncthreads();
  f32x4_t* red = reinterpret_cast<f32x4_t*>(dg_smem);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NTW; ++j) red[((kw * MT + mt) * NT + cw * NTW + j) * 64 + lane] = acc[mt][j];
  __syncthreads();
  auto total = [&](int mt, int n) __attribute__((always_inline)) {
    f32x4_t v[KW];
#pragma unroll
    for (int k = 0; k < KW; ++k) v[k] = red[((k * MT + mt) * NT + n) * 64 + lane];
    f32x4_t t = v[0];
#pragma unroll
    for (int k = 1; k < KW; ++k) t += v[k];
    return t;   // lane (q, r): D[16 mt + 4 q + i][16 (nt0 + n) + r]
  };
  constexpr int UN = EPI == EPI_SWIGLU ? NT / 2 : NT;   // output tiles
  for (int f = wave; f < MT * UN; f += DG_WAVES) {
    const int mt = f / UN, n = f % UN;
    if (nt0 + n * (NT / UN) >= p.N / 16) continue;   // past N
    if constexpr (EPI == EPI_SWIGLU) {
      const f32x4_t tg = total(mt, 2 * n), tu = total(mt, 2 * n + 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = mt * 16 + 4 * qq + i;
        const float gt = rbf(tg[i]), u = rbf(tu[i]);
        const float s = rbf(gt / (1.0f + expf(-gt)));
        if (m < p.M) p.out[(size_t)m * p.ld_out + (nt0 / 2 + n) * 16 + rr] = f2bf(mul_rn(s, u));
      }
    } else {
      const f32x4_t t = total(mt, n);
      const int col = (nt0 + n) * 16 + rr;
      bf16_t rv[4];
      if constexpr (EPI == EPI_RES) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = mt * 16 + 4 * qq + i;
          rv[i] = res_lds ? res_s[m * (16 * NT) + n * 16 + rr] : p.res[(size_t)min(m, p.M - 1) * p.ld_out + col];
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = mt * 16 + 4 * qq + i;
        const bool live = m < p.M;
        if constexpr (EPI == EPI_RES) {
          const bf16_t o = f2bf(add_rn(bf2f(rv[i]), rbf(t[i])));
          if (live) p.out[(size_t)m * p.ld_out + col] = o;
          if (p.psq_out) {   // partial sum of squares of the new row over these 16 columns
            const float v = bf2f(o);
            const float sq = row16_sum(mul_rn(v, v));
            if (live && rr == 0) p.psq_out[(size_t)m * (p.N >> 4) + nt0 + n] = sq;
          }
        } else if (live) {
          p.out[(size_t)m * p.ld_out + col] = f2bf(t[i]);
        }
      }
    }
  }
}

// Wavefront split, and stages at one and two row tiles. Three to five are best: with the LDS filled (9 / 6 stages of
// NT = 1, 6 / 4 of NT = 2) the first stage comes back later and the launches take 0.1 - 0.8 us longer.
template <int NT>
struct DgShape;
template <> struct DgShape<1> { static constexpr int KW = 8, CW = 1, S1 = 5, S2 = 5; };
template <> struct DgShape<2> { static constexpr int KW = 8, CW = 1, S1 = 4, S2 = 3; };
template <> struct DgShape<6> { static constexpr int KW = 4, CW = 2, S1 = 4, S2 = 3; };

template <int MT, int NT, bool NORM, int EPI>
int dg_launch(const DecodeGemmParams& p, hipStream_t stream) {
  using H = DgShape<NT>;
  constexpr int S = MT == 1 ? H::S1 : H::S2;
  const long long lds = dg_lds(MT, NT, H::KW, S, p.K, NORM);
  if (lds > 160 * 1024) return QWEN_EARG;
  auto kern = decode_gemm_kernel<MT, NT, H::KW, H::CW, S, NORM, EPI>;
  static bool attr = false;  // one-time opt-in to more than 64 KB of dynamic LDS
  if (!attr) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
      return QWEN_EARG;
    attr = true;
  }
  kern<<<(p.N / 16 + NT - 1) / NT, 64 * DG_WAVES, lds, stream>>>(p);
  QWEN_RETURN_LAUNCH();
}

template <int NT>
int dg_dispatch(const DecodeGemmParams& p, bool norm, int epi, hipStream_t stream) {
  const bool two = p.M > 16;
  if (epi == EPI_STORE && norm) return two ? dg_launch<2, NT, true, EPI_STORE>(p, stream) : dg_launch<1, NT, true, EPI_STORE>(p, stream);
  if (epi == EPI_STORE) return two ? dg_launch<2, NT, false, EPI_STORE>(p, stream) : dg_launch<1, NT, false, EPI_STORE>(p, stream);
  if (epi == EPI_RES) return two ? dg_launch<2, NT, false, EPI_RES>(p, stream) : dg_launch<1, NT, false, EPI_RES>(p, stream);
  if constexpr (NT >= 2) {
    if (epi == EPI_SWIGLU)
      return two ? dg_launch<2, NT, true, EPI_SWIGLU>(p, stream) : dg_launch<1, NT, true, EPI_SWIGLU>(p, stream);
  }
  return QWEN_EARG;
}

}  // namespace

extern "C" int qwen_linear(const void* x, const void* w_tiled, void* out, int M, int N, int K, int ld_out,
                           const void* norm_w, const float* psq_in, float eps, const void* residual, float* psq_out,
                           int epi, int ntw, int wpg, int ks, void* workspace, long long workspace_bytes,
                           hipStream_t stream);   // gemm.hip

extern "C" int qwen_linear_stream(const void* x, const void* w_tiled, void* out, int M, int N, int K, int ld_out,
                                  const void* norm_w, const float* psq_in, float eps, const void* residual,
                                  float* psq_out, int epi, int nt, hipStream_t stream) {
  if (!x || !w_tiled || !out) return QWEN_ENULL;
  if (M < 1 || M > 32 || N <= 0 || K <= 0 || K % 256 || (nt != 1 && nt != 2 && nt != 6)) return QWEN_EARG;
  if (N % 16 || (epi == EPI_SWIGLU && N % 32) || (epi == EPI_RES && N % (16 * nt)) || (norm_w && K > 8192) || K > 1 << 22 ||
      ld_out > 1 << 26)
    return QWEN_EARG;
  if (epi < EPI_STORE || epi > EPI_SWIGLU) return QWEN_EARG;
  if (epi == EPI_RES && !residual) return QWEN_ENULL;
  if (norm_w && !psq_in) return QWEN_ENULL;
  if (epi == EPI_RES ? norm_w != nullptr : psq_out != nullptr) return QWEN_EARG;
  if (epi == EPI_SWIGLU && (!norm_w || nt < 2)) return QWEN_EARG;
  if (ld_out < (epi == EPI_SWIGLU ? N / 2 : N)) return QWEN_EARG;
  // (direct global -> LDS loads want 16-byte aligned rows; others take gemm.hip's launch of the same operator)
  if (((uintptr_t)x | (uintptr_t)w_tiled) & 15)
    return qwen_linear(x, w_tiled, out, M, N, K, ld_out, norm_w, psq_in, eps, residual, psq_out, epi,
                       epi == EPI_SWIGLU ? 2 : 1, 8, 1, nullptr, 0, stream);
  DecodeGemmParams p{(const bf16_t*)x, (const bf16_t*)w_tiled, (const bf16_t*)norm_w, (const bf16_t*)residual,
                     (bf16_t*)out, psq_in, psq_out, M, N, K, ld_out, eps};
  const bool norm = norm_w != nullptr;
  switch (nt) {
    case 1: return dg_dispatch<1>(p, norm, epi, stream);
    case 2: return dg_dispatch<2>(p, norm, epi, stream);
    default: return dg_dispatch<6>(p, norm, epi, stream);
  }
}

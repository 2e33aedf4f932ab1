// Prompt-forward attention: causal flash attention of a chunk of the prompt.
//
// The reference's prompt forward (engine/engine.py:1181-1221) runs cuBLAS GEMMs and SDPA
// over B x S rows. Here the prompt goes through in position chunks of all sequences; the
// projections are in prompt_gemm.hip, the norms, RoPE + cache write and the first-token LM
// head are the decode path's kernels.
//
// pf_attn_kernel: causal GQA attention of the T queries of a chunk (positions p0 + t) over
//   the cache slots [0, p0 + t] (engine/engine.py:1123-1179's SDPA, with the decode
//   attention's rounding points, engine/kernels/torch_ref.py:168-227: fp32 scores times
//   scale, probabilities rounded to bf16 for the value product, fp32 row sums, one final
//   rounding). One workgroup per (sequence, KV head, 16 query tokens) holds the 64 query
//   rows (16 tokens x the 4 heads of the group); wavefront w owns tokens 4w .. 4w + 3. K and
//   V blocks of 64 keys are staged in LDS once per workgroup (double buffered, padded rows)
//   and shared by the 4 wavefronts: S = Q K^T and O += P V on the matrix cores, online
//   softmax in the accumulator layout, V^T fragments by ds_read_b64_tr_b16 (as in
//   attention_mfma.hip). Workgroups with the most keys are launched first.
//
// Chunks of more than 16 tokens take pf_attn_wide_kernel (16 or 32 query tokens per 4-wavefront workgroup, two
// workgroups per CU), described at its definition below.
#include "common.h"
#include "lds_ring.h"

namespace {

// 16 bytes held as a native vector: arrays of these stay in VGPRs (an array of the HIP uint4
// struct is placed in scratch memory, and every load into it then waits at its store).
typedef unsigned pv4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ causal flash attention
constexpr int AD = 128;      // head dim
constexpr int AG = 4;        // query heads per KV head
constexpr int AQ = 16;       // query tokens per workgroup
constexpr int AKB = 64;      // keys per block
constexpr int AKROW = 136;   // bf16 per LDS row of K (272 B)
constexpr int AVROW = 144;   // bf16 per LDS row of V (288 B: banked transpose reads)
constexpr float ANEG = -1e30f;

typedef short av4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) av4i16 lds_av4i16;

struct PfAttnParams {
  const bf16_t* q;   // [B, T, Nq, D] (normed + rotated)
  const bf16_t* kc;  // [B, Nkv, CAP, D]
  const bf16_t* vc;
  bf16_t* out;       // [B, T, Nq * D]
  int T, Nkv, CAP, p0, qblocks;
  long long bh_count;
  float scale;
};

struct PfAttnSmem {
  bf16_t k[2][AKB][AKROW];
  bf16_t v[2][AKB][AVROW];
  bf16_t pm[4][16][AKB];
};

__global__ void __launch_bounds__(256, 2) pf_attn_kernel(PfAttnParams p) {
  __shared__ PfAttnSmem sm;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qq = lane >> 4, rr = lane & 15;
  // heaviest query blocks first
  const long long id = blockIdx.x;
  const int qb = p.qblocks - 1 - (int)(id / p.bh_count);
  const long long bh = id % p.bh_count;
  const long long b = bh / p.Nkv;
  const int kvh = (int)(bh - b * p.Nkv);
  const int T = p.T, Nq = p.Nkv * AG;
  const int t_lo = qb * AQ;
  const int kmax = p.p0 + min(T, t_lo + AQ);  // keys [0, kmax) are visible to some query here
  const int nblk = (kmax + AKB - 1) / AKB;
  const bf16_t* kbase = p.kc + bh * (long long)p.CAP * AD;
  const bf16_t* vbase = p.vc + bh * (long long)p.CAP * AD;

  // Q A-operand fragments: lane (q, r) holds row r of this wavefront's tile (token
  // 4 wave + r / 4, head r % 4), dims 32 kt + 8 q .. +8. Tokens past T re-read token T - 1.
  bf16x8_t qa[4];
  {
    const int t = min(t_lo + 4 * wave + (rr >> 2), T - 1);
    const bf16_t* qr = p.q + (((b * T + t) * Nq) + kvh * AG + (rr & 3)) * (long long)AD + 8 * qq;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) qa[kt] = as_bf16x8(*reinterpret_cast<const uint4*>(qr + 32 * kt));
  }
  // accumulator rows 4 qq + i: token t_lo + 4 wave + qq, head i; its last visible key
  const int my_tok = t_lo + 4 * wave + qq;
  const int my_last = p.p0 + my_tok;

  // K / V staging: thread -> 16-byte chunk c of keys (tid >> 4) + 16 i (keys past kmax are
  // read from slot 0 and their V rows zeroed, so a stale or non-finite slot never enters)
  const int sc = tid & 15;
  pv4 kst[4], vst[4];
  auto load_kv = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = blk * AKB + (tid >> 4) + 16 * i;
      const long long off = (long long)(key < kmax ? key : 0) * AD + sc * 8;
      kst[i] = *reinterpret_cast<const pv4*>(kbase + off);
      vst[i] = *reinterpret_cast<const pv4*>(vbase + off);
    }
  };
  auto store_kv = [&](int buf, int blk) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kr = (tid >> 4) + 16 * i;
      const bool live = blk * AKB + kr < kmax;
      *reinterpret_cast<pv4*>(&sm.k[buf][kr][sc * 8]) = kst[i];
      *reinterpret_cast<pv4*>(&sm.v[buf][kr][sc * 8]) = live ? vst[i] : pv4{0u, 0u, 0u, 0u};
    }
  };

  float m[4], l[4];
  f32x4_t o[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) { m[i] = ANEG; l[i] = 0.f; }
#pragma unroll
  for (int nd = 0; nd < 8; ++nd) o[nd] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  bf16_t* pl = &sm.pm[wave][0][0];

  load_kv(0);
  store_kv(0, 0);
  __syncthreads();
  for (int blk = 0; blk < nblk; ++blk) {
    const int nb = blk + 1 < nblk ? blk + 1 : blk;
    load_kv(nb);
    const int buf = blk & 1;
    const int kb0 = blk * AKB;
    // S = Q K^T for 4 tiles of 16 keys: lane (q, r) takes key 16 nt + r, dims 32 kt + 8 q ..
    f32x4_t s[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      s[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
        const uint4 kf = *reinterpret_cast<const uint4*>(&sm.k[buf][16 * nt + rr][32 * kt + 8 * qq]);
        s[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[kt], as_bf16x8(kf), s[nt], 0, 0, 0);
      }
    }
    // online softmax (rows 4 qq + i share the token, so one causal limit per lane)
    float alpha[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float sv[4];
      float mx = ANEG;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const bool vis = kb0 + 16 * nt + rr <= my_last;
        sv[nt] = vis ? s[nt][i] * p.scale : ANEG;
        mx = fmaxf(mx, sv[nt]);
      }
      mx = row16_max(mx);
      const float mn = fmaxf(m[i], mx);
      alpha[i] = __expf(m[i] - mn);
      float psum = 0.f;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const float pr = sv[nt] > ANEG ? __expf(sv[nt] - mn) : 0.f;
        psum += pr;
        pl[(4 * qq + i) * AKB + 16 * nt + rr] = f2bf(pr);  // P rounded to bf16 for PV
      }
      l[i] = l[i] * alpha[i] + psum;
      m[i] = mn;
    }
#pragma unroll
    for (int nd = 0; nd < 8; ++nd)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[nd][i] *= alpha[i];
    // P in the A layout (lane (q, r): row r, keys 32 kk + 8 q ..); the round trip stays inside
    // the wavefront (LDS instructions complete in order)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    bf16x8_t pa[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) pa[kk] = as_bf16x8(*reinterpret_cast<const uint4*>(pl + rr * AKB + 32 * kk + 8 * qq));
    // O += P V: V^T fragments by transpose reads, source lane s -> V[8 q + s / 4 (+4)][16 nd + 4 (s % 4)]
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const bf16_t* vs = &sm.v[buf][32 * kk + 8 * qq + (rr >> 2)][4 * (rr & 3)];
#pragma unroll
      for (int nd = 0; nd < 8; ++nd) {
        const av4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_av4i16*)(vs + 16 * nd));
        const av4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_av4i16*)(vs + 4 * AVROW + 16 * nd));
        const uint4 vv = make_uint4(__builtin_bit_cast(uint2, lo).x, __builtin_bit_cast(uint2, lo).y,
                                    __builtin_bit_cast(uint2, hi).x, __builtin_bit_cast(uint2, hi).y);
        o[nd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[kk], as_bf16x8(vv), o[nd], 0, 0, 0);
      }
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    store_kv(buf ^ 1, nb);  // buffer last read one iteration ago (behind the barrier below)
    __syncthreads();
  }

  // ---- normalise and write: the wavefront's 16 rows x 128 dims through LDS (bf16), 16-byte stores
#pragma unroll
  for (int i = 0; i < 4; ++i) l[i] = row16_sum(l[i]);
  bf16_t* ot = &sm.k[0][0][0] + wave * 16 * AKROW;  // 16 rows of 272 B per wavefront
#pragma unroll
  for (int nd = 0; nd < 8; ++nd)
#pragma unroll
    for (int i = 0; i < 4; ++i) ot[(4 * qq + i) * AKROW + 16 * nd + rr] = f2bf(o[nd][i] / l[i]);
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int c = lane + 64 * it;        // 16 rows x 16 chunks
    const int row = c >> 4, ch = c & 15;
    const int t = t_lo + 4 * wave + (row >> 2);
    if (t < T) {
      const uint4 v = *reinterpret_cast<const uint4*>(ot + row * AKROW + ch * 8);
      bf16_t* dst = p.out + ((b * T + t) * Nq + kvh * AG + (row & 3)) * (long long)AD + ch * 8;
      *reinterpret_cast<uint4*>(dst) = v;
    }
  }
}


// Wide form of the prompt attention (qwen_attn_prefill for chunks of more than 16 tokens):
// 4 wavefronts x QT query tiles per workgroup, i.e. 16 QT query tokens x the 4 heads of the GQA group
// over the same 64-key K / V block in LDS. Wavefront w owns tokens 4 QT w .. 4 QT w + 4 QT - 1
// (tile mt: tokens 4 QT w + 4 mt .. + 3), so every K fragment read from LDS feeds all tiles' MFMAs. A block
// takes a workgroup 0.95 us with one tile, 1.36 with two, 2.1 with three (alone on its CU): two carry the most when
// the chip is full, one ends first while it is not (three, at 250 VGPRs: -4 to +3 % on full chips, up to 50 % slower
// elsewhere). A query's result is the same bit for bit with any QT. Two
// workgroups share a CU (64 KB of LDS each), so the two wavefronts on a SIMD belong to different
// workgroups with their own barriers and drift apart: one's softmax runs under the other's MFMAs
// (measured on MI355X at the 32 x 512-token chunks: 2-3 % faster than one 8-wavefront
// workgroup of 64 tokens per CU, 20 % on the first chunk).
constexpr int AW2 = 4;               // wavefronts per workgroup
constexpr int AGPW = AKB / 4 / AW2;  // 4-row groups of a K / V block staged by each wavefront

// The score tiles are computed transposed, S^T = K Q^T (K as the MFMA's A operand, Q^T as B).
// Lane (q, r) then holds query r's scores for keys 16 nt + 4 q + i, which is already the
// B-operand layout of O^T += V^T P^T once the k-slots of the PV product are ordered
// (32 kk + 4 q + j, 32 kk + 16 + 4 q + j): P goes from the score accumulators into the PV MFMA
// through packed bf16 conversions, with no LDS round trip, and the V^T fragments are transposed
// LDS reads in that same key order. Softmax state is one (m, l) per lane and tile; a query's 64
// scores sit on 4 lanes (r, r + 16, r + 32, r + 48), so a block maximum is 15 in-lane maxima and
// 2 cross-lane steps. The causal mask is applied only to blocks that reach past the wavefront's
// first token. exp(x - m) is evaluated as exp2((x - m) log2 e) with scale folded in, and the
// rescale factor as exp2((m_old - m_new) scale log2 e), exactly 1 when the maximum is unchanged:
// a block that is fully masked for a query leaves that query's state bit for bit as it was, so
// the result does not depend on how many such blocks a workgroup walks. Rounding points as
// pf_attn_kernel (P rounded to bf16 for PV, l from the unrounded P, O normalised in fp32, then
// rounded). exp2 is the hardware v_exp_f32: a P below 2^-126 of the block maximum flushes to 0,
// far under bf16's resolution of the row sum.
__device__ __forceinline__ float xlane_max4(float v) { return xor32_max(xor16_max(v)); }
__device__ __forceinline__ float xlane_sum4(float v) { return xor32_sum(xor16_sum(v)); }

template <int QT>
__global__ void __launch_bounds__(AW2 * 64, 2) pf_attn_wide_kernel(PfAttnParams p) {
  constexpr int AQW = AW2 * 4 * QT;  // query tokens per workgroup
  // K / V blocks in 256-byte rows with no padding (direct-to-LDS loads fill 1 KB runs), swizzled
  // so that the fragment reads stay conflict-free: K's 16-byte chunk c of key row r at c ^ (r % 16)
  // (the S^T operand reads 16 rows of one chunk), V's 32-byte block j of row r at j ^ (r % 8) (a
  // transposed read takes 8 bytes from 4 consecutive rows of one block, two groups of lanes at
  // once take rows 4 apart).
  __shared__ union {
    struct {
      pv4 k[2][AKB][16];
      pv4 v[2][AKB][16];
    } kv;
    bf16_t ot[AW2][16 * QT][AKROW];  // output staging: 16 QT rows per wavefront
  } sm;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qq = lane >> 4, rr = lane & 15;
  // Launch order: workgroup g runs on XCD g % 8 and takes logical item (g % 8) * ceil(G / 8) +
  // g / 8, so each XCD walks a contiguous run of items; an item is (head group bh, query block),
  // all query blocks of a head group consecutive, heaviest first. The workgroups that read the
  // same K / V (every query block of one head group) then run at the same time on one XCD and
  // stream its blocks in step, through that XCD's L2, instead of each reading them from HBM in
  // a different round.
  const long long G = p.bh_count * p.qblocks;
  const long long per_xcd = (G + 7) / 8;
  const long long item = (long long)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (item >= G) return;
  const long long bh = item / p.qblocks;
  const int qb = p.qblocks - 1 - (int)(item - bh * p.qblocks);
  const long long b = bh / p.Nkv;
  const int kvh = (int)(bh - b * p.Nkv);
  const int T = p.T, Nq = p.Nkv * AG;
  const int t_lo = qb * AQW;
  const int kmax = p.p0 + min(T, t_lo + AQW);  // keys [0, kmax) are visible to some query here
  const int nblk = (kmax + AKB - 1) / AKB;
  const bf16_t* kbase = p.kc + bh * (long long)p.CAP * AD;
  const bf16_t* vbase = p.vc + bh * (long long)p.CAP * AD;

  // Q^T B-operand fragments: lane (q, r) of tile mt holds query r (token 8 wave + 4 mt + r / 4,
  // head r % 4), dims 32 kt + 8 q .. +8. Tokens past T re-read token T - 1.
  bf16x8_t qb8[QT][4];
  int my_last[QT];                   // last key visible to this lane's query, per tile
#pragma unroll
  for (int mt = 0; mt < QT; ++mt) {
    const int tq = t_lo + 4 * QT * wave + 4 * mt + (rr >> 2);
    const bf16_t* qr = p.q + (((b * T + min(tq, T - 1)) * Nq) + kvh * AG + (rr & 3)) * (long long)AD + 8 * qq;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) qb8[mt][kt] = as_bf16x8(*reinterpret_cast<const uint4*>(qr + 32 * kt));
    my_last[mt] = p.p0 + tq;
  }
  const int wave_first = p.p0 + t_lo + 4 * QT * wave;  // every query of the wavefront sees keys <= this
  const float c = p.scale * 1.4426950408889634f;  // scale * log2(e)

  // K / V staging by direct global -> LDS loads: wavefront w fills key rows 16 w .. 16 w + 15
  // of a block (four 1 KB runs of 4 rows each for K and for V). Lane l lands at row
  // 4 (AGPW w + i) + l / 16, physical chunk l % 16, so it loads the logical chunk the swizzle
  // puts there. Keys past kmax read slot kmax - 1, one of this chunk's keys (written before the
  // attention runs, so finite), and every query weighs them with P = 0 exactly: a stale or
  // non-finite slot never enters.
  const int srow = lane >> 4, spc = lane & 15;
  const unsigned lds_k = (unsigned)(uintptr_t)(__attribute__((address_space(3))) pv4*)&sm.kv.k[0][0][0];
  const unsigned lds_v = (unsigned)(uintptr_t)(__attribute__((address_space(3))) pv4*)&sm.kv.v[0][0][0];
  // (K and V are issued separately, so a block's eight loads per wavefront do not go out in one
  // burst)
  // A lane's byte offset within a block is the same for every block: row r's logical chunk,
  // r * 256 + chunk * 16, added to the block's address in the scalar base. In the
  // workgroup's last block, if it reaches past kmax, rows at or past kmax read row kmax - 1
  // instead (still within the block, so every offset stays below 16 KB whatever the cache
  // capacity).
  unsigned koff[AGPW], voff[AGPW];
#pragma unroll
  for (int i = 0; i < AGPW; ++i) {
    const int r = 4 * (AGPW * wave + i) + srow;
    koff[i] = (unsigned)(r * 256 + (spc ^ (r & 15)) * 16);                          // logical K chunk
    voff[i] = (unsigned)(r * 256 + (2 * ((spc >> 1) ^ (r & 7)) + (spc & 1)) * 16);  // V chunk
  }
  auto issue_kv = [&](int blk, int buf, bool k) __attribute__((always_inline)) {
    const bf16_t* sb = (k ? kbase : vbase) + (long long)blk * AKB * AD;
    const unsigned lds0 = (k ? lds_k : lds_v) + (unsigned)((buf * AKB + 4 * AGPW * wave) * 256);
    if ((blk + 1) * AKB <= kmax) {
#pragma unroll
      for (int i = 0; i < AGPW; ++i) ring_load16(sb, k ? koff[i] : voff[i], lds0 + i * 1024);
    } else {
      const int last = kmax - 1 - blk * AKB;   // last row of the block below kmax (>= 0)
#pragma unroll
      for (int i = 0; i < AGPW; ++i) {
        const int r = 4 * (AGPW * wave + i) + srow;   // row of the block
        const unsigned off = k ? koff[i] : voff[i];
        ring_load16(sb, r <= last ? off : off - (unsigned)((r - last) * 256), lds0 + i * 1024);
      }
    }
  };

  float m[QT], l[QT];
  f32x4_t o[QT][8];                  // O^T: lane (q, r) holds dims 16 nd + 4 q + i of query r
#pragma unroll
  for (int mt = 0; mt < QT; ++mt) {
    m[mt] = ANEG;
    l[mt] = 0.f;
#pragma unroll
    for (int nd = 0; nd < 8; ++nd) o[mt][nd] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  issue_kv(0, 0, true);
  issue_kv(0, 0, false);
  ring_wait<0>();
  __syncthreads();
  for (int blk = 0; blk < nblk; ++blk) {
    const int buf = blk & 1;
    const bool more = blk + 1 < nblk;
    if (more) issue_kv(blk + 1, buf ^ 1, true);  // that buffer was last read one block ago
    const int kb0 = blk * AKB;
    // S^T for 4 tiles of 16 keys: A = K rows 16 nt + r, dims 32 kt + 8 q (one LDS read per
    // (nt, kt), all query tiles)
    f32x4_t st[QT][4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
#pragma unroll
      for (int mt = 0; mt < QT; ++mt) st[mt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
        const uint4 kf = __builtin_bit_cast(uint4, sm.kv.k[buf][16 * nt + rr][(4 * kt + qq) ^ rr]);
#pragma unroll
        for (int mt = 0; mt < QT; ++mt)
          st[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf), qb8[mt][kt], st[mt][nt], 0, 0, 0);
      }
    }
    if (more) issue_kv(blk + 1, buf ^ 1, false);
    if (kb0 + AKB - 1 > wave_first) {  // block reaches past some query's last key: mask
#pragma unroll
      for (int mt = 0; mt < QT; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kb0 + 16 * nt + 4 * qq + i > my_last[mt]) st[mt][nt][i] = ANEG;
    }
    // online softmax per tile (one query per lane); P^T as packed bf16 B fragments
    uint4 pb[QT][2];
    float alpha[QT];
    bool moved = false;
#pragma unroll
    for (int mt = 0; mt < QT; ++mt) {
      float mx = st[mt][0][0];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, st[mt][nt][i]);
      mx = xlane_max4(mx);
      const float mn = fmaxf(m[mt], mx);
      const float mc = mn * c;
      alpha[mt] = __builtin_amdgcn_exp2f((m[mt] - mn) * c);  // 1 exactly if mn == m
      moved |= alpha[mt] != 1.f;
      float pr[4][4];
      float psum = 0.f;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          pr[nt][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[mt][nt][i], c, -mc));  // masked: 0
          psum += pr[nt][i];
        }
      l[mt] = l[mt] * alpha[mt] + psum;
      m[mt] = mn;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        pb[mt][kk] = make_uint4(f2bf2(pr[2 * kk][0], pr[2 * kk][1]), f2bf2(pr[2 * kk][2], pr[2 * kk][3]),
                                f2bf2(pr[2 * kk + 1][0], pr[2 * kk + 1][1]), f2bf2(pr[2 * kk + 1][2], pr[2 * kk + 1][3]));
    }
    // rescale O only when some query's maximum moved (alpha is exactly 1 otherwise)
    if (__builtin_amdgcn_ballot_w64(moved) != 0) {
#pragma unroll
      for (int mt = 0; mt < QT; ++mt)
#pragma unroll
        for (int nd = 0; nd < 8; ++nd)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[mt][nd][i] *= alpha[mt];
    }
    // O^T += V^T P^T: A = V^T rows (dims) 16 nd + r, k-slots j -> key 32 kk + 4 q + j (lo) and
    // 32 kk + 16 + 4 q + j (hi), by transpose reads of 4 keys x 16 dims (source lane s ->
    // V[32 kk + 4 q + s / 4 (+16)][16 nd + 4 (s % 4)]), one read pair per (kk, nd) for all tiles
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      // row 32 kk + 4 q + r / 4 (+ 16), 8 bytes at column 16 nd + 4 (r % 4) of its swizzled block
      const int vr = 32 * kk + 4 * qq + (rr >> 2);
      const bf16_t* vlo = reinterpret_cast<const bf16_t*>(&sm.kv.v[buf][vr][0]) + 4 * (rr & 3);
      const bf16_t* vhi = reinterpret_cast<const bf16_t*>(&sm.kv.v[buf][vr + 16][0]) + 4 * (rr & 3);
#pragma unroll
      for (int nd = 0; nd < 8; ++nd) {
        const av4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_av4i16*)(vlo + 16 * (nd ^ (vr & 7))));
        const av4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_av4i16*)(vhi + 16 * (nd ^ ((vr + 16) & 7))));
        const uint4 vv = make_uint4(__builtin_bit_cast(uint2, lo).x, __builtin_bit_cast(uint2, lo).y,
                                    __builtin_bit_cast(uint2, hi).x, __builtin_bit_cast(uint2, hi).y);
#pragma unroll
        for (int mt = 0; mt < QT; ++mt)
          o[mt][nd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(vv), as_bf16x8(pb[mt][kk]), o[mt][nd], 0, 0, 0);
      }
    }
    ring_wait<0>();  // this wavefront's next-block loads have landed ...
    __syncthreads();  // ... and, past the barrier, every wavefront's
  }

  // ---- normalise and write: rows 16 mt + r (query r of tile mt) x 128 dims through LDS (bf16,
  // 4 dims per 8-byte store), then 16-byte global stores (the K / V buffers are free: every
  // wavefront passed the loop's last barrier)
  bf16_t* ot = &sm.ot[wave][0][0];
#pragma unroll
  for (int mt = 0; mt < QT; ++mt) {
    const float inv = 1.f / xlane_sum4(l[mt]);
#pragma unroll
    for (int nd = 0; nd < 8; ++nd)
      *reinterpret_cast<uint2*>(ot + (16 * mt + rr) * AKROW + 16 * nd + 4 * qq) =
          make_uint2(f2bf2(o[mt][nd][0] * inv, o[mt][nd][1] * inv), f2bf2(o[mt][nd][2] * inv, o[mt][nd][3] * inv));
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int it = 0; it < 4 * QT; ++it) {
    const int cidx = lane + 64 * it;     // 16 QT rows x 16 chunks
    const int row = cidx >> 4, ch = cidx & 15;
    const int t = t_lo + 4 * QT * wave + (row >> 2);
    if (t < T) {
      const uint4 v = *reinterpret_cast<const uint4*>(ot + row * AKROW + ch * 8);
      bf16_t* dst = p.out + ((b * T + t) * Nq + kvh * AG + (row & 3)) * (long long)AD + ch * 8;
      *reinterpret_cast<uint4*>(dst) = v;
    }
  }
}
}  // namespace

extern "C" {

int qwen_attn_prefill(const void* q, const void* k_cache, const void* v_cache, void* out, int B, int T, int Nq,
                      int Nkv, int D, int CAP, int p0, float scale, hipStream_t stream) {
  if (!q || !k_cache || !v_cache || !out) return QWEN_ENULL;
  if (D != AD || Nkv <= 0 || Nq != AG * Nkv || B < 0 || T < 0 || p0 < 0 || CAP <= 0) return QWEN_EARG;
  if ((long long)p0 + T > CAP) return QWEN_EARG;
  if (B == 0 || T == 0) return QWEN_OK;
  PfAttnParams p{};
  p.q = (const bf16_t*)q;
  p.kc = (const bf16_t*)k_cache;
  p.vc = (const bf16_t*)v_cache;
  p.out = (bf16_t*)out;
  p.T = T; p.Nkv = Nkv; p.CAP = CAP; p.p0 = p0;
  const bool wide = T > AQ;   // one 16-token workgroup per head group suffices for short chunks
  p.bh_count = (long long)B * Nkv;
  // One query tile per wavefront where that lets a launch end sooner, else two. Two workgroups per CU run at a time, the
  // heaviest query blocks first. While all of the one-tile form's run at once, the longest decides, and its blocks are
  // shorter; with more of them the first to end (at p0 + T (1 - slots / n)) takes another of that length, which
  // has to end with the longest: 2 (p0 + T (1 - slots / n)) <= p0 + T. us, two tiles -> one, where this takes one: 128
  // tokens 7.7 -> 7.1, 300 after 2,000 keys 52 -> 40, 1,024 after 4,096 110 -> 101, 3 x 517 24.5 -> 20.7, 1,536 38 -> 30,
  // 2,048 52 -> 50; and where it takes two: 2 x 700 after 1,000 51 -> 51, 1,900 after 3,000 138 -> 158,
  // 2 x 2,048 83 -> 95, 4 x 1,024 after 7,168 503 -> 613 (but 8 x 300 21.1 -> 19.6).
  const long long n = p.bh_count * ((T + 15LL) / 16), slots = 2LL * device_cu_count();
  const bool two = n > slots && (n > 2 * slots || (long long)p0 * n > (long long)T * (2 * slots - n));
  const int tokens = wide && two ? 32 : 16;   // of a workgroup
  p.qblocks = (T + tokens - 1) / tokens;
  p.scale = scale;
  const long long blocks = p.bh_count * p.qblocks;
  if (blocks > 0x7fffffffLL) return QWEN_EARG;
  const dim3 runs((unsigned)((blocks + 7) / 8 * 8));   // 8 equal runs of the wide kernel
  if (wide && two) pf_attn_wide_kernel<2><<<runs, AW2 * 64, 0, stream>>>(p);
  else if (wide) pf_attn_wide_kernel<1><<<runs, AW2 * 64, 0, stream>>>(p);
  else pf_attn_kernel<<<dim3((unsigned)blocks), 256, 0, stream>>>(p);
  QWEN_RETURN_LAUNCH();
}

}  // extern "C"

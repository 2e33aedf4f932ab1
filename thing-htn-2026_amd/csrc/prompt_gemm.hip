// The prompt forward's projections: out[M, N] = A[M, K] @ W[N, K]^T for any number of rows M, bf16
// operands, fp32 accumulation and one bf16 rounding (engine/kernels/gemm.py:12-15), with the fused
// epilogues of the decode projections (engine/kernels/gemm_fused.py:5-19):
//   STORE : out = bf16(acc)
//   RES   : out = bf16(res + bf16(acc))              (residual may alias out)
//   SWIGLU: out = bf16(bf16(silu(bf16(g))) * bf16(u)) for a pair-interleaved gate|up weight
//
// W is in the MFMA-B tile layout (weights.hip): tile (nt, kt) = 16 rows x 32 k, 1 KB, lane l = 16 q + r
// holding W[16 nt + r][32 kt + 8 q .. +8]. The product is computed transposed, D^T = W X^T: a weight tile is
// the A operand of v_mfma_f32_16x16x32_bf16 as it stands and 16 rows of A its B operand.
//
// Both operands go through LDS, filled by direct global -> LDS loads (1 KB per instruction) into a ring of
// stages; a stage is read into registers while the one before it is multiplied, so that a slot is free
// for the next load one stage early and no multiplication waits for its own LDS reads. Loads are
// waited for by count, never all at once. (Measured on MI355X: such loads reach 64 bytes per clock
// and CU, 150 GB/s, when each row's segment is at least 128 bytes, and 62 GB/s with 64-byte segments, so A
// rows are staged 64 or 128 k at a time.)
//
// Every element accumulates its k range in steps of 32 from 0 up in one accumulator, whatever the tile: the
// bits of a row do not depend on how many rows the launch has (no split of k, which the prompt forward's
// independence of its chunking rules out). The tile is therefore the only freedom: small tiles put
// every CU to work when there are few rows, large ones move fewer bytes per flop when there are many.
// prompt_gemm_kernel covers 32 x 32 to 256 x 128; prompt_gemm_big_kernel is the 256 x 256 one. The
// choice is made in qwen_gemm at the end of this file.
#include "common.h"
#include "lds_ring.h"

#include <algorithm>

namespace {

enum { PEPI_STORE = 0, PEPI_RES = 1, PEPI_SWIGLU = 2 };

typedef unsigned pv4 __attribute__((ext_vector_type(4)));  // (an array of the uint4 struct would be placed in scratch)
typedef pv4 pv4_any __attribute__((aligned(2)));           // the same at any bf16 element

struct PfGemmParams {
  const bf16_t* a;    // [M, K] row-major
  const bf16_t* w;    // tiled [N, K]
  const bf16_t* res;  // [M, ldo] (RES; may alias out)
  bf16_t* out;        // [M, ldo]
  int M, N, K, ldo;
  int mtiles, ntiles;
  int pull;           // workgroups without a tile pull weights
};

// Output tile walk of a persistent workgroup. gridDim.x = 8 s workgroups; workgroup g runs on XCD g % 8
// and takes run positions g / 8, g / 8 + s, .. of that XCD's contiguous run of logical tiles, which go in
// groups of PGROUP row tiles, the row tile fastest: the tiles an XCD works on at one time then share
// their A and W k-slabs in its L2.
constexpr int PGROUP = 4;
struct TileWalk {
  int first, stride, mine;   // this workgroup's first logical tile, the step to its next, how many
  int slot, run;             // its place among its XCD's workgroups, the XCD's tiles
  int mtiles, ntiles;
  __device__ __forceinline__ TileWalk(const PfGemmParams& p) : mtiles(p.mtiles), ntiles(p.ntiles) {
    const int tiles = p.mtiles * p.ntiles, per_xcd = (tiles + 7) / 8;
    const int xcd = (int)(blockIdx.x & 7);
    slot = (int)(blockIdx.x >> 3);
    stride = (int)(gridDim.x >> 3);
    run = min(per_xcd, tiles - xcd * per_xcd);   // may be <= 0
    first = xcd * per_xcd + slot;
    mine = run > slot ? (run - slot + stride - 1) / stride : 0;
  }
  __device__ __forceinline__ void at(int step, int& mt, int& nt) const {   // row tile, column tile
    const int lt = first + step * stride, gsize = PGROUP * ntiles;
    const int grp = lt / gsize, rem = lt - grp * gsize;
    const int gsz = min(PGROUP, mtiles - grp * PGROUP);
    nt = rem / gsz;
    mt = grp * PGROUP + rem - nt * gsz;
  }
};

// A workgroup without a tile: reads the weights of its XCD's tiles ahead of the ones that have tiles, so that they come
// from the XCD's L2. A CU that multiplies a few rows has its loads in flight limited by its L1: with the weights in HBM it
// moves about 60 GB/s of both operands however deep its ring, with them in the caches 90 and more. Pieces of
// 4 KB (a 64-byte line per lane) of one n-tile after the other, k ascending, as the tiles use them: 64-byte steps
// beat 128 by 0 - 5 %, four loads in flight eight by 0 - 7 %. us per launch with cold weights, without -> with:
// O 128 rows 16.7 -> 12.5, 256 rows 20.8 -> 16.1; down 34.2 -> 25.2, 44.8 -> 33.5; gate/up 128 rows 32.2 -> 27.2.
template <int BN, int NW>
__device__ __forceinline__ void pull_weights(const PfGemmParams& p, const TileWalk& walk, int wave, int lane) {
  constexpr int PIECE = 4096, DEPTH = 4;
  const int run = walk.run;
  if (run <= 0) return;
  const int gsize = PGROUP * p.ntiles, lt0 = walk.first - walk.slot, lt1 = lt0 + run - 1, grp = lt0 / gsize;
  const int gsz = min(PGROUP, p.mtiles - grp * PGROUP);
  const int b0 = (lt0 - grp * gsize) / gsz;   // column tiles b0 .. b1 (of a run over two row groups: the first group's)
  const int b1 = lt1 / gsize == grp ? (lt1 - grp * gsize) / gsz : p.ntiles - 1;
  const int n = (b1 - b0 + 1) * (BN / 16), bytes = p.K * 32;   // n-tiles, bytes of one
  const int items = n * ((bytes + PIECE - 1) / PIECE), workers = (walk.stride - run) * NW;
  const char* base = reinterpret_cast<const char*>(p.w) + (long long)b0 * (BN / 16) * bytes;
  for (int at = (walk.slot - run) * NW + wave; at < items; at += DEPTH * workers) {
    unsigned v[DEPTH];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      const int it = min(at + i * workers, items - 1), piece = it / n;
      v[i] = *reinterpret_cast<const unsigned*>(base + (long long)(it - piece * n) * bytes +
                                                min(piece * PIECE + lane * 64, bytes - 4));
    }
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) asm volatile("" ::"v"(v[i]));
  }
}

// Epilogue of a wavefront's MB x NB accumulator tiles (rows row0 .., weight n-tiles nt0 ..): lane (q, r) of
// tile (mb, nb) holds D[16 mb + r][16 nb + 4 q + i]. Two neighbouring output tiles exchange their odd and
// even 16-lane rows (permlane16_swap), after which a lane holds 8 adjacent columns: lane (q, r) those
// of tile 2 j + (q & 1) from 8 (q >> 1), one 16-byte store (and residual load) instead of two of 8.
// get(mb, nb, i) reads an accumulator element.
template <int MB, int NB, int EPI, typename Get>
__device__ __forceinline__ void store_tiles(const PfGemmParams& p, int row0, int nt0, int lane, Get&& get) {
  constexpr int OT = EPI == PEPI_SWIGLU ? NB / 2 : NB;   // output tiles of 16 columns
  const int qq = lane >> 4, rr = lane & 15;
  const int ot0 = EPI == PEPI_SWIGLU ? nt0 / 2 : nt0;
  auto value = [&](int mb, int t, int i) __attribute__((always_inline)) -> float {
    if constexpr (EPI == PEPI_SWIGLU) {
      const float g = rbf(get(mb, 2 * t, i));
      const float u = rbf(get(mb, 2 * t + 1, i));
      return mul_rn(rbf(g / (1.0f + expf(-g))), u);
    } else {
      return get(mb, t, i);
    }
  };
  static_assert(OT == 1 || OT % 2 == 0, "output tiles go in pairs, or there is one");
  const long long coff = OT == 1 ? (long long)ot0 * 16 + 4 * qq : (long long)(ot0 + (qq & 1)) * 16 + 8 * (qq >> 1);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const long long row = row0 + mb * 16 + rr;
    const bool live = row < p.M;
    const long long at = (live ? row : 0) * p.ldo + coff;
    if constexpr (OT == 1) {
      static_assert(OT > 1 || EPI == PEPI_SWIGLU, "a single output tile comes from a gate / up pair");
      const uint2 v = make_uint2(f2bf2(value(mb, 0, 0), value(mb, 0, 1)), f2bf2(value(mb, 0, 2), value(mb, 0, 3)));
      if (live) *reinterpret_cast<uint2*>(p.out + at) = v;
    } else {
      uint4 rv[EPI == PEPI_RES ? OT / 2 : 1];
      if constexpr (EPI == PEPI_RES) {
#pragma unroll
        for (int j = 0; j < OT / 2; ++j) rv[j] = *reinterpret_cast<const uint4*>(p.res + at + 32 * j);
      }
#pragma unroll
      for (int j = 0; j < OT / 2; ++j) {
        uint32_t d[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          d[h][0] = f2bf2(value(mb, 2 * j + h, 0), value(mb, 2 * j + h, 1));
          d[h][1] = f2bf2(value(mb, 2 * j + h, 2), value(mb, 2 * j + h, 3));
        }
        const auto s0 = __builtin_amdgcn_permlane16_swap(d[0][0], d[1][0], false, false);
        const auto s1 = __builtin_amdgcn_permlane16_swap(d[0][1], d[1][1], false, false);
        uint4 v = make_uint4(s0[0], s1[0], s0[1], s1[1]);
        if constexpr (EPI == PEPI_RES) {
          // Used by every lane: a residual load that only live lanes use counts as pending when the next
          // tile's loop begins, and the compiler then waits there for every outstanding load on each
          // pass (measured: O and down 25 % slower).
          asm volatile("" : "+v"(rv[j].x), "+v"(rv[j].y), "+v"(rv[j].z), "+v"(rv[j].w));
          float a[8], r[8];
          unpack8(v, a);
          unpack8(rv[j], r);
#pragma unroll
          for (int e = 0; e < 8; ++e) a[e] = add_rn(r[e], a[e]);
          v = pack8(a);
        }
        if (live) *reinterpret_cast<uint4*>(p.out + at + 32 * j) = v;
      }
    }
    __builtin_amdgcn_sched_barrier(0);   // one row block's accumulators in flight at a time
  }
}

// ---------------------------------------------------------------- tiles of 32 x 32 to 256 x 128
// BM x BN output tiles, WM x WN wavefronts, stages of 32 SUB k, a ring of S stages, persistent workgroups
// (one per CU: the ring fills most of its LDS). Per stage: wait for the next stage's loads, one barrier, then
// the multiplications of this stage between the next one's LDS reads and the loads of the stage S on,
// into the slot just left. What bounds it at few rows is the loads, see pull_weights (a wavefront that runs ahead in
// the same CU made every shape 5 - 40 % slower, non-temporal W loads 10 - 50 %). Against the one 256 x 256
// tile that all shapes ran before (Qwen3-4B, us per launch, graph replays over 1.2 GB of weights):
//                QKV            O              gate/up        down
//   23 rows      57 -> 10.7     89 -> 11.0     62 -> 23.0     206 -> 20.6
//   128 rows     63 -> 13.6     97 -> 12.7     70 -> 29.4     220 -> 25.3
//   512 rows     72 -> 24.4     105 -> 23.2    75 -> 63       237 -> 48
//   2048 rows    69 -> 58       103 -> 51      207 -> 187     223 -> 109
// LDS: A rows of 4 SUB 16-byte chunks, chunk c of row r at c ^ f(r), so that the 16 rows of a fragment
// read hit different banks; W as its 1 KB tiles, those of one n-tile side by side.
// DIRECT false (operands that are not 16-byte aligned, which the direct loads need): a stage is loaded into registers
// by ordinary loads and stored to its LDS slot one step later, behind that step's barrier.
template <int BM, int BN, int WM, int WN, int SUB, int S, int EPI, bool DIRECT>
__global__ void __launch_bounds__(64 * WM * WN, 1) prompt_gemm_kernel(PfGemmParams p) {
  constexpr int NW = WM * WN;
  constexpr int MB = BM / WM / 16, NB = BN / WN / 16;
  constexpr int C = 4 * SUB;   // 16-byte chunks per staged A row (SUB >= 2: at least 128 bytes)
  constexpr int AI = BM * SUB / 16, WI = BN * SUB / 16;   // 1 KB loads per stage
  constexpr int PA = AI / NW, PW = WI / NW, PER = PA + PW;
  constexpr int STAGE = (AI + WI) * 1024;
  static_assert(AI % NW == 0 && WI % NW == 0 && MB * WM * 16 == BM && NB * WN * 16 == BN, "tile split");
  static_assert(SUB == 2 || SUB == 4, "stages of 64 or 128 k");
  static_assert(DIRECT || S >= 3, "a slot that is stored one step late is neither being read nor read next");
  static_assert(EPI != PEPI_SWIGLU || NB % 2 == 0, "gate / up pairs stay in one wavefront");
  __shared__ pv4 lds[S * STAGE / 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int qq = lane >> 4, rr = lane & 15;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) pv4*)lds;

  const int KT = p.K / 32, KB = KT / SUB;
  const TileWalk walk(p);
  const int mine = walk.mine;
  if (mine <= 0) {
    if (p.pull) pull_weights<BN, NW>(p, walk, wave, lane);
    return;
  }
  const int G = mine * KB;   // stages of all this workgroup's tiles, run through without a break between tiles
  auto tile_at = [&](int step, int& m0, int& nt0) __attribute__((always_inline)) {
    walk.at(step, m0, nt0);
    m0 *= BM;
    nt0 *= BN / 16;
  };

  // ---- load cursor: the next stage to request. Wavefront w loads A blocks and W tiles PA w .., PW w ..;
  // rows past M re-read row M - 1 and are never stored. The lane offsets fit 32 bits: (M - 1) K < 2^31 elements
  // for A (checked by the host), and for W the tiles after a wavefront's first n-tile (host, too).
  int istep = 0, ikb = 0, islot = 0;
  const char* abase = nullptr;
  const char* wbase = nullptr;
  unsigned avoff[PA], wvoff[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int t = wave * PW + i;
    wvoff[i] = (unsigned)((t / SUB - wave * PW / SUB) * KT + t % SUB) * 1024u + lane * 16u;
  }
  auto open_tile = [&]() __attribute__((always_inline)) {
    int m0, nt0;
    tile_at(istep, m0, nt0);
    abase = reinterpret_cast<const char*>(p.a) + (long long)m0 * p.K * 2;
    wbase = reinterpret_cast<const char*>(p.w) + (long long)(nt0 + wave * PW / SUB) * KT * 1024;
    const int last = p.M - 1 - m0;
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int s = (wave * PA + i) * 64 + lane;
      const int row = s / C, pc = s % C;
      avoff[i] = (unsigned)min(row, last) * (unsigned)(p.K * 2) + (unsigned)((pc ^ (row & (C - 1))) * 16);
    }
  };
  pv4 hold[DIRECT ? 1 : PER];   // the last requested stage (not DIRECT)
  bool held = false;            // .. is still to be stored
  auto issue_one = [&](int i) __attribute__((always_inline)) {
    if constexpr (DIRECT) {
      const unsigned sb = lds0 + islot * STAGE;
      if (i < PA) ring_load16(abase, avoff[i < PA ? i : 0], sb + (wave * PA + i) * 1024);
      else ring_load16(wbase, wvoff[i < PA ? 0 : i - PA], sb + (AI + wave * PW + i - PA) * 1024);
    } else {
      hold[i] = *reinterpret_cast<const pv4_any*>(i < PA ? abase + avoff[i < PA ? i : 0] : wbase + wvoff[i < PA ? 0 : i - PA]);
      held = true;
    }
  };
  auto store_held = [&]() __attribute__((always_inline)) {   // into the slot before the cursor's
    if constexpr (!DIRECT) {
      if (held) {
        pv4* st = lds + (islot == 0 ? S - 1 : islot - 1) * (STAGE / 16) + lane;
#pragma unroll
        for (int i = 0; i < PER; ++i) st[(i < PA ? wave * PA + i : AI + wave * PW + i - PA) * 64] = hold[i];
        held = false;
      }
    }
  };
  auto issue_next = [&]() __attribute__((always_inline)) {  // advance the issue cursor by one stage
    islot = islot + 1 == S ? 0 : islot + 1;
    abase += SUB * 64;
    wbase += SUB * 1024;
    if (++ikb == KB) {
      ikb = 0;
      if (++istep < mine) open_tile();
    }
  };

  f32x4_t acc[MB][NB];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  struct Frags {
    bf16x8_t w[SUB][NB], x[SUB][MB];
  };
  // fragment r of a stage's SUB * (NB + MB), in the order they are used
  auto read_one = [&](Frags& f, int slot, int r) __attribute__((always_inline)) {
    const pv4* st = lds + slot * (STAGE / 16);
    const int sub = r / (NB + MB), j = r % (NB + MB);
    if (j < NB) {
      f.w[sub][j] = __builtin_bit_cast(bf16x8_t, st[AI * 64 + ((wn * NB + j) * SUB + sub) * 64 + lane]);
    } else {
      const int row = (wm * MB + j - NB) * 16 + rr;
      f.x[sub][j - NB] = __builtin_bit_cast(bf16x8_t, st[row * C + ((sub * 4 + qq) ^ (row & (C - 1)))]);
    }
  };

  constexpr int R = SUB * (NB + MB);
  constexpr int GP = SUB * MB;              // groups of NB MFMAs
  constexpr int RG = GP >= 2 ? GP / 2 : 1;  // groups over which the reads are spread
  int g = 0, cslot = 0;
  auto step = [&](auto steady, const Frags& cur, Frags& nxt) __attribute__((always_inline)) {
    constexpr bool ST = decltype(steady)::value;
    const bool load = ST || g + S < G;
    if constexpr (DIRECT) {
      if constexpr (ST) ring_wait<PER * (S - 2)>();
      else if (g + 1 < G) ring_wait_stages<PER, S - 2>(G - g - 2);
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    store_held();
    cslot = cslot + 1 == S ? 0 : cslot + 1;   // stage g + 1's slot
#pragma unroll
    for (int gp = 0; gp < GP; ++gp) {
      const int sub = gp / MB, mb = gp % MB;
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (gp < RG && r >= R * gp / RG && r < R * (gp + 1) / RG) read_one(nxt, cslot, r);
      if (load) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
          if (i >= PER * gp / GP && i < PER * (gp + 1) / GP) issue_one(i);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur.w[sub][nb], cur.x[sub][mb], acc[mb][nb], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (load) issue_next();
    ++g;
  };

  open_tile();
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (s < G) {
#pragma unroll
      for (int i = 0; i < PER; ++i) issue_one(i);
      issue_next();
      store_held();
    }
  }
  Frags f0, f1;
  if constexpr (DIRECT) ring_wait_stages<PER, S - 1>(G - 1);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) read_one(f0, 0, r);
  for (int t = 0; t < mine; ++t) {
    clear();
    int kb = 0;
    const int steady = min(KB, G - S - g);  // k-steps of this tile after which a stage is left to issue
    for (; kb + 2 <= steady; kb += 2) {
      step(std::true_type{}, f0, f1);
      step(std::true_type{}, f1, f0);
    }
    for (; kb < KB; ++kb) {
      step(std::false_type{}, f0, f1);
      f0 = f1;
    }
    int m0, nt0;
    tile_at(t, m0, nt0);
    store_tiles<MB, NB, EPI>(p, m0 + wm * MB * 16, nt0 + wn * NB, lane, [&](int mb, int nb, int i) { return acc[mb][nb][i]; });
  }
}

// ---------------------------------------------------------------- 256 x 256 tiles
// Many rows: four wavefronts, one per SIMD, each with a 128 x 128 quadrant (8 x 8 accumulator tiles: all 256
// AGPRs). A stages of 64 k (3 slots of 32 KB), W half-stages of 32 k (4 slots of 16 KB): all 160 KB. A phase is 32 k:
// one barrier, 64 MFMAs, and between them, one at a time, the next phase's 16 LDS reads (first half), 8 direct
// loads and the cursor arithmetic. One wavefront per SIMD issues everything in order, so whatever stands
// between two groups of MFMAs instead of inside one leaves the matrix cores idle: each of these was measured
// (16,384 rows): reads and loads in one group before 8 MFMAs and the cursors after the phase 1,280 TFLOP/s,
// interleaved 1,315, cursors in between as well 1,390 (gate/up). A load is requested two phases before
// the barrier that waits for it (vmcnt(16): the last two phases' loads stay in flight).
// Against the 8-wavefront kernel with two full stages that it replaces, us per launch at 16,384 rows, the same launch
// back to back: QKV 425 -> 370, O 322 -> 283, gate/up + SwiGLU 1,363 -> 1,221, down 750 -> 633; between the other kernels
// of a prompt forward 352 / 284 / 1,179 / 604 (1,464 / 1,210 / 1,385 / 1,352 TFLOP/s; O and down are 2.5 rounds
// of tiles that cost three). 64 MFMAs alone on every SIMD, random operands in registers, run at 1,766 TFLOP/s (the chip
// lowers its clock), with this phase's LDS reads, barrier and L2-resident loads at 1,531.
constexpr int GM = 256, GN = 256;
constexpr int G_ASLOTS = 3, G_WSLOTS = 4;
constexpr int G_ABYTES = 32 * 1024;   // 256 A rows x 64 k; 16-byte chunk c of row r at c ^ (r % 8)
constexpr int G_WBYTES = 16 * 1024;   // 16 W tiles: 256 weight rows x 32 k

// The accumulators must stay in AGPRs: with the builtin the compiler moves some of them to VGPRs and back on
// every pass (1,260 -> 780 TFLOP/s). The assembly form gives up the compiler's hazard handling, so: an
// accumulator is reused only after 63 other MFMAs; operands come from LDS reads (waited for by the
// compiler), never from a VALU instruction right before; and s_nops stand between the last MFMA and the reads.
__device__ __forceinline__ void mfma_acc(f32x4_t& c, const bf16x8_t& a, const bf16x8_t& b) {
  asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_new(f32x4_t& c, const bf16x8_t& a, const bf16x8_t& b) {
  asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ float acc_read(float c) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(c));
  return v;
}

template <int EPI>
__global__ void __launch_bounds__(256, 1) prompt_gemm_big_kernel(PfGemmParams p) {
  __shared__ pv4 lds[(G_ASLOTS * G_ABYTES + G_WSLOTS * G_WBYTES) / 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int qq = lane >> 4, rr = lane & 15;
  const unsigned lds_a = (unsigned)(uintptr_t)(__attribute__((address_space(3))) pv4*)lds;
  const unsigned lds_w = lds_a + G_ASLOTS * G_ABYTES;

  const int KT = p.K / 32, KB = p.K / 64;
  const TileWalk walk(p);
  const int mine = walk.mine;
  if (mine <= 0) return;
  const int G = mine * KB;   // stages of all this workgroup's tiles
  auto tile_at = [&](int step, int& m0, int& nt0) __attribute__((always_inline)) {
    walk.at(step, m0, nt0);
    m0 *= GM;
    nt0 *= GN / 16;
  };

  // A cursor: the stage to request next. Block b (8 rows) = 8 wave + i; rows past M re-read row M - 1.
  int astep = 0, akb = 0;
  unsigned aslot = 0, aat = lds_a + wave * 8192;   // slot to fill next, this wavefront's part of it
  const char* abase = nullptr;
  unsigned avoff[8];
  auto open_a = [&]() __attribute__((always_inline)) {
    int m0, nt0;
    tile_at(astep, m0, nt0);
    abase = reinterpret_cast<const char*>(p.a) + (long long)m0 * p.K * 2;
    const int last = p.M - 1 - m0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = (wave * 8 + i) * 8 + (lane >> 3);
      avoff[i] = (unsigned)min(row, last) * (unsigned)(p.K * 2) + (unsigned)(((lane & 7) ^ (row & 7)) * 16);
    }
  };
  auto issue_a = [&](auto i) __attribute__((always_inline)) {
    ring_load16_at<decltype(i)::value * 1024>(abase, avoff[decltype(i)::value], aat);
  };
  auto bump_a = [&]() __attribute__((always_inline)) {
    aslot = aslot + 1 == G_ASLOTS ? 0 : aslot + 1;
    aat = lds_a + wave * 8192 + aslot * G_ABYTES;
    abase += 128;
  };
  auto next_a = [&]() __attribute__((always_inline)) {
    if (__builtin_expect(++akb == KB, 0)) {
      akb = 0;
      if (++astep < mine) open_a();
    }
  };
  // W cursor: half-stages. W tile t = 4 wave + i.
  int wstep = 0, wkt = 0;
  unsigned wslot = 0, wat = lds_w + wave * 4096;
  const char* wbase = nullptr;
  unsigned wvoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) wvoff[i] = (unsigned)((wave * 4 + i) * KT) * 1024u + lane * 16u;
  auto open_w = [&]() __attribute__((always_inline)) {
    int m0, nt0;
    tile_at(wstep, m0, nt0);
    wbase = reinterpret_cast<const char*>(p.w) + (long long)nt0 * KT * 1024;
  };
  auto issue_w = [&](auto i) __attribute__((always_inline)) {
    ring_load16_at<decltype(i)::value * 1024>(wbase, wvoff[decltype(i)::value], wat);
  };
  auto bump_w = [&]() __attribute__((always_inline)) {
    wslot = (wslot + 1) & 3;
    wat = lds_w + wave * 4096 + wslot * G_WBYTES;
    wbase += 1024;
  };
  auto next_w = [&]() __attribute__((always_inline)) {
    if (__builtin_expect(++wkt == KT, 0)) {
      wkt = 0;
      if (++wstep < mine) open_w();
    }
  };

  f32x4_t acc[8][8];
  struct Frags {
    bf16x8_t w[8], x[8];
  };
  Frags f0, f1;
  // This lane's LDS byte addresses in slot 0: its 16 bytes of the wavefront's W tiles (1 KB apart) and
  // chunk (4 sub + q) of its A row (rows of the next 16-row block 2 KB on; the swizzle repeats every 8 rows).
  const unsigned wread = lds_w + wn * 8192 + lane * 16;
  const unsigned aread0 = lds_a + (wm * 128 + rr) * 128 + ((qq ^ (rr & 7)) * 16);
  const unsigned aread1 = lds_a + (wm * 128 + rr) * 128 + (((4 + qq) ^ (rr & 7)) * 16);
  auto lds16 = [](unsigned at) __attribute__((always_inline)) {
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const __attribute__((address_space(3))) pv4*>((uintptr_t)at));
  };

  // Phase `second` of stage g multiplies its k half in `cur` and reads the next phase's operands into `nxt`:
  // (A slot ca, W slot cw). Its barrier also frees the W slot, and in the second phase the A slot, that the operands
  // in `cur` came from. Loads: W half-stage 2 g + 4 (+ 1); A stage g + 3, its first half in the second
  // phase, its second half in the first phase of stage g + 1 (there it counts as stage g + 2 ahead).
  int g = 0, ca = 0, cw = 0;   // stage; slots of the operands read next
  auto phase = [&](auto steady, auto first, auto second, const Frags& cur, Frags& nxt, bool la,
                   bool lw) __attribute__((always_inline)) {
    constexpr bool ST = decltype(steady)::value, FIRST = decltype(first)::value, SUB1 = decltype(second)::value;
    cw = (cw + 1) & 3;
    if constexpr (SUB1) ca = ca + 1 == G_ASLOTS ? 0 : ca + 1;
    const unsigned wr = wread + cw * G_WBYTES, ar = (SUB1 ? aread0 : aread1) + ca * G_ABYTES;
    if constexpr (ST) ring_wait<16>();
    else ring_wait<0>();
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    unroll<64>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value, mb = j / 8, nb = j % 8;
      if constexpr (j % 2 == 0 && j < 16) nxt.w[j / 2] = lds16(wr + j * 512);
      if constexpr (j % 2 == 0 && j >= 16 && j < 32) nxt.x[j / 2 - 8] = lds16(ar + (j - 16) * 1024);
      if constexpr (j % 6 == 3 && j < 48) {
        constexpr int i = j / 12;
        if constexpr (j % 12 == 3) {
          if (ST || lw) issue_w(std::integral_constant<int, i>{});
        } else {
          if (ST || la) issue_a(std::integral_constant<int, i + (SUB1 ? 0 : 4)>{});
        }
      }
      if constexpr (j == 50) {
        if (ST || lw) bump_w();
      }
      if constexpr (j == 53 && !SUB1) {
        if (ST || la) bump_a();
      }
      if constexpr (j == 56) {
        if (ST || lw) next_w();
      }
      if constexpr (j == 59 && !SUB1) {
        if (ST || la) next_a();
      }
      if constexpr (FIRST) mfma_new(acc[mb][nb], cur.w[nb], cur.x[mb]);
      else mfma_acc(acc[mb][nb], cur.w[nb], cur.x[mb]);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto step = [&](auto steady, auto first) __attribute__((always_inline)) {
    phase(steady, first, std::false_type{}, f0, f1, g + 2 < G, g + 2 < G);
    phase(steady, std::false_type{}, std::true_type{}, f1, f0, g + 3 < G, g + 2 < G);
    ++g;
  };

  open_a();
  open_w();
  unroll<3>([&](auto sc) __attribute__((always_inline)) {   // A stages 0, 1 and half of 2; W half-stages 0 .. 3
    constexpr int s = decltype(sc)::value;
    if (s < G) {
      unroll<(s < 2 ? 8 : 4)>([&](auto i) __attribute__((always_inline)) { issue_a(i); });
      if constexpr (s < 2) {
        bump_a();
        next_a();
        unroll<2>([&](auto) __attribute__((always_inline)) {
          unroll<4>([&](auto i) __attribute__((always_inline)) { issue_w(i); });
          bump_w();
          next_w();
        });
      }
    }
  });
  ring_wait<0>();
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    f0.w[r] = lds16(wread + r * 1024);
    f0.x[r] = lds16(aread0 + r * 2048);
  }
  constexpr std::true_type yes;
  constexpr std::false_type no;
  for (int t = 0; t < mine; ++t) {
    const int steady = min(KB, G - 3 - g);
    if (steady > 0) step(yes, yes);
    else step(no, yes);
    int kb = 1;
    for (; kb < steady; ++kb) step(yes, no);
    for (; kb < KB; ++kb) step(no, no);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMA's results are in the AGPRs
    __builtin_amdgcn_sched_barrier(0);
    int m0, nt0;
    tile_at(t, m0, nt0);
    store_tiles<8, 8, EPI>(p, m0 + wm * 128, nt0 + wn * 8, lane, [&](int mb, int nb, int i) { return acc_read(acc[mb][nb][i]); });
  }
}

template <int BM, int BN, int WM, int WN, int SUB, int S, bool DIRECT = true>
int launch_tiles(PfGemmParams p, int epi, dim3 grid, hipStream_t stream) {
  p.mtiles = (p.M + BM - 1) / BM;
  p.ntiles = p.N / BN;
  constexpr int T = 64 * WM * WN;
  if (epi == PEPI_STORE) prompt_gemm_kernel<BM, BN, WM, WN, SUB, S, PEPI_STORE, DIRECT><<<grid, T, 0, stream>>>(p);
  else if (epi == PEPI_RES) prompt_gemm_kernel<BM, BN, WM, WN, SUB, S, PEPI_RES, DIRECT><<<grid, T, 0, stream>>>(p);
  else prompt_gemm_kernel<BM, BN, WM, WN, SUB, S, PEPI_SWIGLU, DIRECT><<<grid, T, 0, stream>>>(p);
  QWEN_RETURN_LAUNCH();
}

int launch_big(PfGemmParams p, int epi, dim3 grid, hipStream_t stream) {
  p.mtiles = (p.M + GM - 1) / GM;
  p.ntiles = p.N / GN;
  if (epi == PEPI_STORE) prompt_gemm_big_kernel<PEPI_STORE><<<grid, 256, 0, stream>>>(p);
  else if (epi == PEPI_RES) prompt_gemm_big_kernel<PEPI_RES><<<grid, 256, 0, stream>>>(p);
  else prompt_gemm_big_kernel<PEPI_SWIGLU><<<grid, 256, 0, stream>>>(p);
  QWEN_RETURN_LAUNCH();
}

// The tiles that qwen_gemm chooses from, with what one round of them (at most a tile on every CU) takes: `step` ns per
// 64 k and `fixed` ns for filling the ring and the epilogue, [0] where one round leaves a quarter of the CUs idle (they
// pull weights, and the others share less), [1] otherwise. Fitted on MI355X on the Qwen3-4B projections with cold
// weights, every tile at 16 to 1,551 rows (the two largest also at 2,048 to 16,384). Rounds times that, the least
// of it, picks the fastest or within 8 % of it. `span`: n-tiles past its first whose weights a wavefront addresses by
// 32-bit offsets from it.
struct TileCost {
  int bm, bn, sub, span;
  int step[2], fixed[2];
};
constexpr TileCost TILES[] = {
    {256, 256, 2, 15, {1009, 1050}, {14600, 5500}}, {256, 128, 2, 0, {585, 650}, {9400, 4300}},
    {128, 128, 2, 0, {410, 400}, {6400, 6000}},     {128, 64, 2, 0, {271, 314}, {5900, 4400}},
    {64, 128, 2, 0, {285, 383}, {6400, 2100}},      {64, 64, 4, 0, {172, 250}, {4500, 4200}},
    {32, 128, 4, 1, {250, 300}, {4300, 7400}},      {32, 64, 4, 0, {129, 195}, {5000, 4500}},
    {32, 32, 4, 0, {96, 118}, {5400, 4400}},
};

// The tile of a launch on slots x 8 CUs and the tiles per XCD's run; -1 where none fits.
int choose_tile(int M, int N, int K, int slots, long long* per_xcd) {
  int best = -1;
  long long least = 0;
  for (int i = 0; i < (int)(sizeof(TILES) / sizeof(TILES[0])); ++i) {
    const TileCost& t = TILES[i];
    if (N % t.bn || K % (32 * t.sub)) continue;
    if (((long long)t.span * (K / 32) + t.sub) * 1024 > 0xffffffffLL) continue;
    const long long tiles = (long long)((M + t.bm - 1) / t.bm) * (N / t.bn), run = (tiles + 7) / 8;
    if (tiles > 0x7fffff00LL) continue;
    const int full = run * 4 > slots * 3;
    const long long cost = (run + slots - 1) / slots * ((long long)(K / 64) * t.step[full] + t.fixed[full]);
    if (best < 0 || cost < least) best = i, least = cost, *per_xcd = run;
  }
  return best;
}

}  // namespace

extern "C" int qwen_gemm_tile(int M, int N, int K, int cus) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 128 || K % 64 || cus < 0 || (long long)M * K >= 0x7fffffffLL) return 0;
  long long run = 0;
  const int i = choose_tile(M, N, K, std::max(1, (cus ? cus : device_cu_count()) / 8), &run);
  return i < 0 ? 0 : TILES[i].bm << 16 | TILES[i].bn;
}

extern "C" int qwen_gemm(const void* a, const void* w_tiled, void* out, int M, int N, int K, int ld_out,
                         const void* residual, int epi, hipStream_t stream) {
  if (!a || !w_tiled || !out) return QWEN_ENULL;
  if (M < 0 || N <= 0 || K <= 0 || N % 128 || K % 64 || epi < PEPI_STORE || epi > PEPI_SWIGLU) return QWEN_EARG;
  const int ncols = epi == PEPI_SWIGLU ? N / 2 : N;
  if (ld_out < ncols || ld_out % 8) return QWEN_EARG;
  if (epi == PEPI_RES && !residual) return QWEN_ENULL;
  if (M == 0) return QWEN_OK;
  if ((long long)M * K >= 0x7fffffffLL) return QWEN_EARG;
  PfGemmParams p{};
  p.a = (const bf16_t*)a;
  p.w = (const bf16_t*)w_tiled;
  p.res = (const bf16_t*)residual;
  p.out = (bf16_t*)out;
  p.M = M; p.N = N; p.K = K; p.ldo = ld_out;
  const int slots = std::max(1, device_cu_count() / 8);   // workgroups per XCD
  // Direct loads want 16-byte aligned addresses; rows and tiles are multiples of 128 bytes, so the bases decide. All
  // other operands are staged through registers, in the larger tile where the smaller one takes more than a round (us,
  // smaller -> larger, N = 2688 and 2,048 rows: K = 2560 82 -> 53, K = 9728 311 -> 194). A load's latency shows in each
  // k step: 29 us at 23 rows and K = 2560, 8.6 from aligned operands; at 16,384 rows and K = 9728 1,209, aligned 737.
  if (((uintptr_t)a | (uintptr_t)w_tiled) & 15) {
    const bool large = (long long)((M + 127) / 128) * (N / 64) > 8LL * slots;
    const long long tiles = large ? (long long)((M + 255) / 256) * (N / 128) : (long long)((M + 127) / 128) * (N / 64);
    if (tiles > 0x7fffff00LL) return QWEN_EARG;
    const dim3 grid((unsigned)(8 * std::min<long long>((tiles + 7) / 8, slots)));
    return large ? launch_tiles<256, 128, 4, 2, 2, 3, false>(p, epi, grid, stream)
                 : launch_tiles<128, 64, 2, 2, 2, 6, false>(p, epi, grid, stream);
  }
  long long per_xcd = 0;
  const int best = choose_tile(M, N, K, slots, &per_xcd);
  if (best < 0) return QWEN_EARG;
  // Persistent: at most one workgroup per CU. Idle CUs pull weights where they are a quarter or more (fewer fall behind
  // and only add traffic: down at 96 rows, 240 tiles of 32 x 32, 49 us with them, 22 without) and up to 1,024 rows
  // (more do not wait for weights: down 77 -> 68 us at 1,000 rows, 75 -> 76 at 1,300, 97 -> 102 at 1,551). An n-tile's
  // bytes are a 32-bit number there.
  p.pull = best > 0 && M <= 1024 && per_xcd * 4 <= slots * 3 && K < 1 << 25;
  const dim3 grid((unsigned)(8 * (p.pull ? slots : std::min<long long>(per_xcd, slots))));
  switch (best) {
    case 0: return launch_big(p, epi, grid, stream);
    case 1: return launch_tiles<256, 128, 4, 2, 2, 3>(p, epi, grid, stream);
    case 2: return launch_tiles<128, 128, 2, 4, 2, 4>(p, epi, grid, stream);
    case 3: return launch_tiles<128, 64, 2, 2, 2, 6>(p, epi, grid, stream);
    case 4: return launch_tiles<64, 128, 2, 4, 2, 6>(p, epi, grid, stream);
    case 5: return launch_tiles<64, 64, 2, 2, 4, 4>(p, epi, grid, stream);
    case 6: return launch_tiles<32, 128, 1, 4, 4, 4>(p, epi, grid, stream);
    case 7: return launch_tiles<32, 64, 2, 2, 4, 6>(p, epi, grid, stream);
    default: return launch_tiles<32, 32, 2, 1, 4, 8>(p, epi, grid, stream);
  }
}

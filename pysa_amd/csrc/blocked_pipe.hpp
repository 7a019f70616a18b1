// The pipelined kernel of the MFMA form (a template over the coupling
// encoding, spin words per matrix wave, the visit order and the tiles per
// workgroup), instantiated one encoding per translation unit.
#pragma once
#include "blocked_dev.hpp"

namespace pysa {
namespace blk {

// ------------------------------------------------------- pipelined form --
// Eight waves per group of 32 NT replicas (NT tiles of 32), two per SIMD.
// One proposal wave per tile runs the proposals, two lanes per replica: lane l
// holds replica l % 32 of the tile and, of the block's 32 visits, those of
// the 4-visit groups with the parity h = l / 32 -- the layout in which the
// matrix cores deliver a product (row 8 (v / 4) + 4 h + v % 4 of column l % 32
// in register v).  Three matrix waves (SIMDs 1-3), a third of the K range
// each and every tile, compute the next block's fields over every K block
// except c (whose spins are changing) while the proposal waves sweep block c:
//     P_{c+1} = sum_{b != c} J[c+1, b] . S_b
// The missing product J[c+1, c] . S_c (one K block) a proposal wave takes itself
// at the start of block c+1, behind its reads of the partials and brackets,
// whose latency it covers (behind the chain of block c, before the barrier:
// 41.4 instead of 40.8 us a sweep at n = 512, 113.7 instead of 112.5 with two
// tiles at n = 1024).  The rows of every fragment are loaded in the visit
// order of their block (row k ^ mask at place k: an XOR of the lane's address),
// so the fields come out in visit order and nothing is permuted afterwards.
// The helper waves stage the next blocks' J block, h and row sums and compute
// the acceptance brackets, so the chain only compares, flips and updates.
// Shared state alternates between two buffers by the parity of a running
// block counter.
// K ranges of the pipelined kernel (one matrix wave each).
constexpr int kPipeMW = 3;
// What the pipelined kernel runs (its MODE).
constexpr int kModePT = 0, kModeBatched = 1, kModeAIS = 2;
// Waves 4..7 but the second tile's proposal wave are helpers.  Wave w runs on
// SIMD w % 4, so both proposal waves share SIMD 0 (with the second one on SIMD
// 1, beside a matrix wave, N = 1024 took 129 instead of 121 us a sweep).
constexpr int kPropWave1 = 4;

// The least float t > x for x < 0 (so x < d, d a float, is t <= d).
__device__ __forceinline__ float float_above(double x) {
  const float f = (float)x;
  return (double)f > x ? f : __uint_as_float(__float_as_uint(f) - 1u);
}
__device__ __forceinline__ void swap2(float& a, float& b) {
  const float t = a;
  a = b;
  b = t;
}
constexpr int kHL = 36;
// Place of visit v in a row of the staged J block: the visits of either lane
// half together, in the order of its field registers.
__device__ __forceinline__ int half_slot(int v) {
  return ((v >> 2) & 1) * 16 + (v >> 3) * 4 + (v & 3);
}
// Counts every element of x as used here (no instruction).
__device__ __forceinline__ void use_whole(const float4& x) {
  asm volatile("" ::"v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w));
}
// The value of lane l % 32 (HI = 0) or 32 + l % 32 (HI = 1) in lane l.
template <int HI>
__device__ __forceinline__ uint32_t half_bcast(uint32_t x) {
  const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return HI ? r[1] : r[0];
}
template <int HI>
__device__ __forceinline__ float half_bcast(float x) {
  return __uint_as_float(half_bcast<HI>(__float_as_uint(x)));
}
template <int HI>
__device__ __forceinline__ double half_bcast(double x) {
  const uint64_t u = as_u64(x);
  return as_double(((uint64_t)half_bcast<HI>((uint32_t)(u >> 32)) << 32) |
                   half_bcast<HI>((uint32_t)u));
}
// NI: instances per workgroup (the batched form keeps one J block and h per
// tile).
template <int MW, int NI, int NT>
struct __align__(16) PipeLds {
  // [parity][matrix wave][tile][register group v / 4][lane]: partial fields
  float4 part[2][MW][NT][4][64];
  // visit i's couplings to the later visits v, else 0: at 32 i + half_slot(v), or
  // (MFMA updates) those of later 4-visit groups at 32 i + v and those of its
  // own group in ji at 4 i + v % 4
  float jb[2][NI][kB * kB];
  float ji[2][NI][kB * 4];
  float hb[2][NI][kB];        // in visit order
  float rsb[2][kB];
  // acceptance brackets [parity][replica][visit index], rows padded to
  // kHL floats so that 16-byte reads of consecutive replicas hit distinct banks
  float lo[2][32 * NT][kHL];
  float hi[2][32 * NT][kHL];
  uint32_t bb[2][64];         // block spins before the block (bit k = row k ^ the visit mask)
  uint32_t bnew[2][64];       // block spins after the block (by block parity)
  float sfp[32 * NT * 33];    // exact rerun staging
  // visit schedule by pass parity: block at step t | its in-block XOR mask << 8
  uint16_t sch[2][64];
  double ds[64];  // a replica's energy change over the sweep (dry pass: its energy)
  uint32_t nacc[64];  // its accepted flips
  float E[64];
  float rb[64];
  float bet[64];  // the ladder by slot (batched: tile t's instance's at 32 t)
  // by slot a (the exchange with slot a - 1): the energy of the replica in slot
  // a - 1, beta[a] - beta[a - 1], the exchange's log-uniform
  // (behind four entries that are only read ahead)
  float4 wl[4 + 64];
  int bso[64];    // the ladder's ascending order (log-omega)
  int bi[64];
  int flag[64];
  int src[64];
  float lu[64];  // by slot a: the least float above the log-uniform of its exchange with a - 1
};

// BR: block-random visit order (schedule tables in LDS); otherwise blocks are
// visited in order with no in-block shuffle, and every schedule entry is
// plain arithmetic on the step.
// BAT: the batched form.  Each workgroup runs two tiles (its entry of
// p.bat), each up to 32 chains of one instance of a batch, the two instances
// with the same number of blocks; couplings are scale * S (S int8), the
// fields kept as the exact integer counts S s, and the field of a spin is the
// f32 value scale * c + h, rounded twice like the batched chain of the
// oracle; the energy changes are summed in f64 in visit order.
// MODE: kModePT (Metropolis sweeps with parallel tempering), kModeBatched
// (BAT), kModeAIS (AIS: annealed importance sampling with the uniform
// reference; no exchanges, no best tracking; every chain at the schedule's
// beta of the sweep, its energy tracked in f64 and its log-weight updated
// after every sweep, pysa/simulation.py:293-317).
template <int NP, bool I8, int NW, int MW, bool BR, int NT, int MODE = kModePT>
__global__ __launch_bounds__(128 * (MW + 1)) void blocked_pipe_kernel(BParams p0) {
  constexpr bool BAT = MODE == kModeBatched, AIS = MODE == kModeAIS;
  // a local copy (the register allocation of the block loops was found to be
  // sensitive to this; the copy keeps it as measured)
  BParams p = p0;
  static_assert(!BAT || (I8 && NP == 1), "the batched form multiplies int8 couplings");
  constexpr int NI = BAT ? NT : 1;  // instances per workgroup (coupling sets)
  // How the proposal waves update the fields of later visits.  One tile per
  // workgroup is bound by the latency of its one proposal wave, and the f32
  // MFMA form shortens it (n = 512, us per sweep of 16 blocks: 43.8 against
  // 45.5); two tiles are bound by instruction issue, shared by two proposal
  // waves on SIMD 0, where the VALU form is better (n = 1024, 32 blocks: 119
  // against 125).
  constexpr bool MU = NT == 1;
  __shared__ PipeLds<MW, NI, NT> L;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int read0 = blockIdx.x * p.rpw;
  const int R = p.R, n = p.n;
  const int nblk = BAT ? p.bat[blockIdx.x].nblk : p.nblk;
  const int kb = BAT ? p.bat[blockIdx.x].kb : p.kb;
  // batched: tile tt's instance and reads, read once at the start (before
  // any store, so they are scalar loads kept in registers; a load later in
  // the kernel could not be proven unclobbered and would be a vector load)
  BatTile bt[NI];
  if constexpr (BAT) {
#pragma unroll
    for (int tt = 0; tt < NI; ++tt) bt[tt] = p.bat[blockIdx.x].t[tt];
  }
  auto tile = [&](int tt) -> const BatTile& { return bt[tt]; };
  auto n_of = [&](int tt) { return BAT ? tile(tt).n : n; };
  const int h = lane >> 5;
  // Two waves per SIMD (SIMD w & 3).  Waves 0 and (two tiles) kPropWave1 run
  // the proposals of a tile each; matrix wave w = 1..MW computes the products
  // of K range m = w - 1 for both tiles of 32 replicas (each coupling fragment
  // is loaded once for both); the helper waves stage the next blocks' J block,
  // h and row sums and compute the acceptance brackets, wave 7 also the
  // visit schedule and the exchange uniforms.  Wave 0 also ends the sweeps.
  static_assert(MW == 3, "eight waves: up to two proposal waves, three matrix waves, helpers");
  const bool mw = w >= 1 && w <= MW;                          // a matrix wave
  const bool pw = w == 0 || (NT == 2 && w == kPropWave1);     // a proposal wave
  const bool hw = !mw && !pw;                                 // a helper wave
  const int m = mw ? w - 1 : 0;
  constexpr int NH = NT == 2 ? 3 : 4;  // helpers
  // helper index
  const int hx = !hw ? 0 : w - (8 - NH);
  const int hl = hw ? hx * 64 + lane : -1;  // helper-lane index 0..64 NH - 1
  // Operand role (matrix waves): replica qtt[tt] of tile tt.
  static_assert(NT == 1 || NT == 2, "one or two tiles of 32 replicas");
  // gtt: its read within the workgroup (recomputed where needed: kept in
  // registers across the block loop they would add to its pressure)
  int qtt[NT], gtt[NT];
  bool actt[NT];
  size_t base_t[NT];
  auto rtt_of = [&](int tt) {  // its replica within the read
    return BAT ? (lane & 31) % R : qtt[tt] - gtt[tt] * R;
  };
  auto rdt_of = [&](int tt) {  // the read's global index
    return BAT ? tile(tt).read0 + (lane & 31) / R : read0 + gtt[tt];
  };
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) {
    qtt[tt] = tt * 32 + (lane & 31);
    if constexpr (BAT) {  // tile tt: p.rpw reads of its own instance
      const int gl = (lane & 31) / R;
      gtt[tt] = tt * p.rpw + gl;
      actt[tt] = mw && gl < p.rpw && rdt_of(tt) < tile(tt).read_end;
      base_t[tt] = actt[tt] ? (size_t)(tile(tt).spin_adj +
                                       ((int64_t)rdt_of(tt) * R + rtt_of(tt)) * tile(tt).n)
                            : 0;
    } else {  // p.rpw reads over the tiles
      gtt[tt] = qtt[tt] / R;
      actt[tt] = mw && (gtt[tt] < p.rpw) && (read0 + gtt[tt] < p.reads);
      base_t[tt] = actt[tt] ? ((size_t)(read0 + gtt[tt]) * R + (qtt[tt] - gtt[tt] * R)) * n : 0;
    }
  }
  // the best state of tile tt's read (operand role)
  auto best_of = [&](int tt) -> int8_t* {
    if constexpr (BAT) return p.best_state + (tile(tt).best_adj + (int64_t)rdt_of(tt) * tile(tt).n);
    return p.best_state + (size_t)(read0 + gtt[tt]) * n;
  };
  // Replica role (every wave): lane = replica q of the group; g its read
  // within the workgroup, tq its tile in the batched form (whose instance's
  // size, scale and ladder the lane uses).
  const int q = lane;
  const int tq = BAT && NT == 2 ? (q >> 5) : 0;
  const int gl = BAT ? (q & 31) / R : 0;  // batched: its read within the tile
  const int g = BAT ? tq * p.rpw + gl : q / R;
  const int rr = BAT ? (q & 31) - gl * R : q - g * R;
  const int read = BAT ? (tq ? tile(NI - 1).read0 : tile(0).read0) + gl : read0 + g;
  const bool act = BAT ? (NT == 2 || q < 32) && gl < p.rpw &&
                             read < (tq ? tile(NI - 1).read_end : tile(0).read_end)
                       : (g < p.rpw) && (read < p.reads);
  const int nq = BAT ? (tq ? tile(NI - 1).n : tile(0).n) : n;
  const float* betas_q =
      BAT ? p.betas + (size_t)(tq ? tile(NI - 1).inst : tile(0).inst) * R : p.betas;
  const uint64_t cid = (uint64_t)read * R + rr;
  // the same of replica qx of a workgroup with one tile
  auto chain_of = [&](int qx) -> uint64_t {
    return (uint64_t)(BAT ? tile(0).read0 : read0) * R + qx;
  };
  auto act_of = [&](int qx) {
    return qx < p.rpw * R && (BAT ? tile(0).read0 : read0) + qx / R < (BAT ? tile(0).read_end : p.reads);
  };
  const int c0 = mw ? m * kb : 0;
  const int jn = mw ? max(0, min(kb, nblk - c0)) : 0;

  Bits<NW> sa[NT];  // this wave's K range of each tile's spins, operand layout
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) {
    sa[tt].w = 0;
    for (int j = 0; j < jn; ++j) {
      const int c = c0 + j;
      const uint32_t va =
          actt[tt] ? load_half<I8>(p.spins + base_t[tt], c, h, n_of(tt)) : 0u;
      set_half<NW>(sa[tt], j, va);
    }
  }
  float E = 0.f, bestE = 0.f, gE = 0.f;
  int gsw = 0, gimp = 0;
  unsigned long long acc = 0;
  double Ed = 0.0, lw = 0.0, bold = 0.0;  // AIS: f64 energy, log-weight, previous beta
  if (AIS && w == 0) {
    Ed = act ? p.ais_e[read] : 0.0;  // R = 1: chain = read
    L.bi[q] = 0;
    const float t0 = p.temps[0];
    L.rb[q] = act ? t0 : 0.f;
    // ordering 1: the weight of sweep 0 before it (bold = 0)
    if (p.ordering == 1 && act) lw = lw + ((-(double)t0 * Ed) - (-bold * Ed));
  }
  if (!AIS && w == 0) {
    E = act ? p.energies[(size_t)read * R + rr] : 0.f;
    L.bi[q] = act ? rr : 0;  // beta_idx = arange(R) (sa.py:325)
    L.rb[q] = act ? betas_q[rr] : 0.f;
    // the ladder in LDS for the exchanges (read serially by the read leaders)
    const int kq = BAT ? (q & 31) : q;
    L.bet[q] = kq < R ? betas_q[kq] : 0.f;
    L.bso[q] = (kq < R && p.logw && p.bsort) ? p.bsort[kq] : 0;
    bestE = E;
    gE = E;  // simulation.py:205 (meaningful on read leaders, rr == 0)
    if (p.best_sem == 0 && act) {
      p.best_rep_e[(size_t)read * R + rr] = E;
      p.best_rep_sw[(size_t)read * R + rr] = 0;
    }
  }
  // fragment stages in flight per matrix wave (slot ring), within the registers
  // (two tiles, N = 1024, us a sweep of 200: two pieces 121 with 3, 127 with 5; three
  // pieces 151 with 2, 160 with 3, which spills)
  constexpr int PF = I8 || NP == 1 ? 6 : NT == 1 ? (NP == 2 ? 6 : 4) : NP == 2 ? 3 : 2;
  const uint32_t emul = p.ptype == 0 ? 0xFEu : 1u;
  const uint32_t exr = p.ptype == 0 ? 0xFFFFFFFFu : 0u;
  // operand-expansion constants in vector registers (see spins_bf16_r)
  uint32_t vmask = 0x80008000u, vone = 0x3F803F80u;
  asm volatile("" : "+v"(vmask), "+v"(vone));
  constexpr int NST = I8 ? 1 : 2;
  constexpr int NHL = 64 * NH;  // helper lanes, NHL / 32 rows of the J block at a time
  constexpr int NJB = (kB * 32 + NHL - 1) / NHL;
  typedef typename std::conditional<I8, i32x4, bf16x8>::type Frag;
  Frag ring[NI][PF][NST][NP];  // by instance (tile in the batched form)
  float jb_reg[NI][NJB], h_reg[NI] = {}, rs_reg = 0.f;
  uint32_t jb_ok[NI] = {};  // bit e2: jb_reg[.][e2] is a coupling; bit 31: h_reg / rs_reg are
  // the coupling fragments of instance ti
  auto frag_base = [&](int ti) -> const Frag* {
    if constexpr (BAT)
      return reinterpret_cast<const Frag*>(reinterpret_cast<const int8_t*>(p.frag) + tile(ti).frag);
    return reinterpret_cast<const Frag*>(p.frag);
  };
  auto frag_ptr = [&](int ti, int c, int j, int st, int pc) -> const Frag* {
    if (I8) return frag_base(ti) + ((size_t)c * nblk + c0 + j) * 64;
    return frag_base(ti) + (((size_t)c * (2 * nblk) + 2 * (c0 + j) + st) * NP + pc) * 64;
  };
  // Stage j of this wave's K range; stages past the range reload the
  // range's last K block (recently read, so a cache hit), so every path
  // issues the same loads and the wait counts stay exact (a skipped load
  // would make the compiler wait for all of them).
  // One K block of fragments: NST * NP * 64 of them, consecutive.
  constexpr int kStage = NST * NP * 64;
  // lx: the lane, its row (low five bits) XORed by the row block's visit mask.
  auto load_stage = [&](int c, int lx, int j, Frag (&dst)[NST][NP], int ti) {
    // jn passes through an empty asm so that the per-stage offsets are
    // recomputed (a few scalar ops) rather than hoisted out of the block
    // loop into registers that would spill
    int jnl = __builtin_amdgcn_readfirstlane(jn);
    asm volatile("" : "+s"(jnl));
    const int jc = jnl > 0 ? min(j, jnl - 1) : nblk - 1 - c0;
    // wave-uniform base of the stage, then a per-lane 16-byte offset
    const Frag* base = frag_ptr(ti, c, 0, 0, 0) + (size_t)jc * kStage;
#pragma unroll
    for (int st = 0; st < NST; ++st)
#pragma unroll
      for (int pc = 0; pc < NP; ++pc) dst[st][pc] = base[(st * NP + pc) * 64 + lx];
  };
  // Request row block c (visit mask xm): the first PF fragment stages of this
  // wave's K range (matrix waves).
  auto prefetch_frags = [&](int c, uint32_t xm) {
    const int lx = lane ^ (int)xm;
#pragma unroll
    for (int u = 0; u < PF; ++u)
#pragma unroll
      for (int ti = 0; ti < NI; ++ti) load_stage(c, lx, u, ring[ti][u], ti);
  };
  // Request row block c, visited with in-block mask xm, spread over the
  // helper lanes: J[blk][blk] in visit order, h and row sums.  Lane hl takes
  // visit column v = hl % 32 of the visit rows hl / 32 + e2 NHL / 32.
  const int jv = hl & 31, ji0 = hl >> 5;
  auto prefetch_jb = [&](int c, uint32_t xm) {
    const int pos0 = 32 * c;
    // Every lane loads (an in-bounds address when its element is padding)
    // and publish_block zeroes the padding: no register is written here
    // except by these loads, which keeps them from waiting on older loads.
#pragma unroll
    for (int ti = 0; ti < NI; ++ti) {
      const int ni = n_of(ti);
      const int col = pos0 + (jv ^ (int)xm);
      const bool cok = hl >= 0 && col < ni;
      jb_ok[ti] = 0;
#pragma unroll
      for (int e2 = 0; e2 < NJB; ++e2) {
        const int i = ji0 + e2 * (NHL / 32);  // visit row
        const int row = pos0 + (i ^ (int)xm);
        const bool ok = cok && i < jv && row < ni;  // i < jv <= 31: later visits only
        jb_ok[ti] |= (uint32_t)ok << e2;
        if constexpr (BAT)  // S symmetric: S^T = S
          jb_reg[ti][e2] = (float)(p.sgn + tile(ti).sgn)[ok ? (size_t)row * tile(ti).ld + col : 0];
        else
          jb_reg[ti][e2] = p.Jt[ok ? (size_t)row * ni + col : 0];
      }
      const bool hok = cok && hl < kB;
      jb_ok[ti] |= (uint32_t)hok << 31;
      if constexpr (BAT) {  // no row sums with int8
        const int64_t ho = tile(ti).h;
        h_reg[ti] = ho >= 0 ? p.h[ho + (hok ? col : 0)] : 0.f;
      } else {
        h_reg[ti] = p.h[hok ? col : 0];
        if (!I8 && p.rowsum) rs_reg = p.rowsum[hok ? col : 0];
      }
    }
  };
  auto publish_block = [&](int pb) {
#pragma unroll
    for (int ti = 0; ti < NI; ++ti)
#pragma unroll
      for (int e2 = 0; e2 < NJB; ++e2) {
        const int i = ji0 + e2 * (NHL / 32);
        if (hl >= 0 && i < kB) {
          const float x = ((jb_ok[ti] >> e2) & 1u) ? jb_reg[ti][e2] : 0.f;
          if constexpr (MU) {
            const bool own = (i >> 2) == (jv >> 2);
            L.jb[pb][ti][hl + e2 * NHL] = own ? 0.f : x;
            if (own) L.ji[pb][ti][4 * i + (jv & 3)] = x;
          } else {
            L.jb[pb][ti][32 * i + half_slot(jv)] = x;
          }
        }
      }
    if (hl >= 0 && hl < kB) {
#pragma unroll
      for (int ti = 0; ti < NI; ++ti) L.hb[pb][ti][hl] = ((jb_ok[ti] >> 31) & 1u) ? h_reg[ti] : 0.f;
      L.rsb[pb][hl] = (((jb_ok[0] >> 31) & 1u) && !I8 && p.rowsum) ? rs_reg : 0.f;
    }
  };
  // Products of K step j (fragments fa) with this tile's spins hx.
  auto mfma_step = [&](const Frag (&fa)[NST][NP], uint32_t hx, f32x16& acc, i32x16& iacc) {
    if (I8) {
      uint32_t d[4];
      spins_i8(hx, emul, exr, d);
      i32x4 bv;
#pragma unroll
      for (int e = 0; e < 4; ++e) bv[e] = (int)d[e];
      const i32x4 a8 = __builtin_bit_cast(i32x4, fa[0][0]);
      iacc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a8, bv, iacc, 0, 0, 0);
    } else {
      const uint32_t nz = spins_nz(hx);
#pragma unroll
      for (int st = 0; st < NST; ++st) {
        uint32_t d[4];
        if (st == 0)
          spins_bf16_r<0>(nz, vmask, vone, d);
        else
          spins_bf16_r<1>(nz, vmask, vone, d);
        u32x4v ud = {d[0], d[1], d[2], d[3]};
        const bf16x8 bv = __builtin_bit_cast(bf16x8, ud);
#pragma unroll
        for (int pc = 0; pc < NP; ++pc)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[st][pc]), bv,
                                                        acc, 0, 0, 0);
      }
    }
  };
  // Partial fields of row block cr over this wave's K range, skipping K block
  // ex (its product is added by the proposal wave once the block's spins are
  // final), into the buffers of parity pb; ring holds the first PF stages of
  // row block cr (visit mask xm) on entry.
  auto compute_part = [&](int cr, uint32_t xm, int ex, int pb) {
    const int lx = lane ^ (int)xm;
    f32x16 acc[NT] = {};
    i32x16 iacc[NT] = {};
    const int jx = ex - c0;  // the skipped stage, if it is in this wave's range
    constexpr int kUnrollJ = NW <= 8 ? (2 * NW + PF - 1) / PF : 1;
#pragma unroll kUnrollJ
    for (int jb0 = 0; jb0 < 2 * NW; jb0 += PF) {
      if (jb0 >= jn) break;
      // stages left from this chunk on, recomputed per chunk (a scalar
      // compare a slot instead of per-slot lane masks kept across the loop)
      int jrem = __builtin_amdgcn_readfirstlane(jn - jb0);
      asm volatile("" : "+s"(jrem));
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int j = jb0 + u;
        // consume slot u, then refill it with stage j + PF (no copy of the
        // fragments: the load is issued after the products that read them);
        // slots past the 2 NW spin halves exist only when PF does not divide
        // 2 NW and are never live
        if (j < 2 * NW && u < jrem && j != jx) {
#pragma unroll
          for (int tt = 0; tt < NT; ++tt)
            mfma_step(ring[BAT ? tt : 0][u], get_half<NW>(sa[tt], j), acc[tt], iacc[tt]);
        }
#pragma unroll
        for (int ti = 0; ti < NI; ++ti) load_stage(cr, lx, j + PF, ring[ti][u], ti);
      }
    }
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        float4 x;
        if (I8)
          x = make_float4((float)iacc[tt][4 * g4], (float)iacc[tt][4 * g4 + 1],
                          (float)iacc[tt][4 * g4 + 2], (float)iacc[tt][4 * g4 + 3]);
        else
          x = make_float4(acc[tt][4 * g4], acc[tt][4 * g4 + 1], acc[tt][4 * g4 + 2],
                          acc[tt][4 * g4 + 3]);
        L.part[pb][m][tt][g4][lane] = x;
      }
  };
  // Acceptance brackets of row block cr (in-block mask xm) for sweep counter
  // sw, stored by visit index: groups of 4 rows (one Philox block each) dealt
  // over the helpers, beta from L.rb.  Two tiles: lane = replica; one tile:
  // lanes l and l + 32 hold replica l and take groups 2 hx and 2 hx + 1.
  const int qb = NT == 2 ? q : (lane & 31);
  const uint64_t cidb = NT == 2 ? cid : chain_of(qb);
  const bool actb = NT == 2 ? act : act_of(qb);
  const SweepStream stream(cidb, p.k0, p.k1);
  const bool idle_any = __ballot(!actb) != 0;
  float cb = 0.f, cz = 0.f;  // of the pass (sweep_factors)
  auto sweep_factors = [&]() { bracket_factors(L.rb[qb], cb, cz); };
  // a lane's groups side by side (their Philox rounds are one dependent chain
  // each); with two tiles the third helper's last one repeats its first
  constexpr int NG = NT == 2 ? 3 : 1;
  static_assert(NT == 2 ? NH == 3 : NH == 4, "8 groups over the helpers");
  auto group_of = [&](int i) {
    const int g4 = NT == 2 ? hx + 3 * i : 2 * hx + h;
    return g4 < kB / 4 ? g4 : hx;
  };
  // the logarithms (base 2) of row block cr's uniforms, which need no beta
  auto draw = [&](int cr, uint64_t sw, float (&lg)[NG][4]) {
    const auto sws = stream.sweep(sw);
    u32x4 blk[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) blk[i] = stream.block(sws, (uint32_t)(8 * cr + group_of(i)));
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      lg[i][0] = accept_log2(blk[i].x), lg[i][1] = accept_log2(blk[i].y);
      lg[i][2] = accept_log2(blk[i].z), lg[i][3] = accept_log2(blk[i].w);
    }
  };
  auto finish = [&](int cr, uint32_t xm, const float (&lg)[NG][4], int pb) {
    const int pos0 = 32 * cr;
    const bool partial = pos0 + kB > (BAT ? min(tile(0).n, tile(NI - 1).n) : n);
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const int g4 = group_of(i);
      float lo[4], hi[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) accept_bounds_l(lg[i][e], cb, cz, lo[e], hi[e]);
      if (partial || idle_any) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (pos0 + 4 * g4 + e >= nq || !actb) lo[e] = hi[e] = INFINITY;  // padding, idle lanes
      }
      // rows 4 g4 + e are visits 4 (g4 ^ xm / 4) + (e ^ xm % 4): one 16-byte
      // store each, its entries exchanged by the uniform low bits of xm
      if (xm & 1u) {
        swap2(lo[0], lo[1]), swap2(lo[2], lo[3]);
        swap2(hi[0], hi[1]), swap2(hi[2], hi[3]);
      }
      if (xm & 2u) {
        swap2(lo[0], lo[2]), swap2(lo[1], lo[3]);
        swap2(hi[0], hi[2]), swap2(hi[1], hi[3]);
      }
      const int v4 = 4 * (g4 ^ (int)(xm >> 2));
      *reinterpret_cast<float4*>(&L.lo[pb][qb][v4]) = make_float4(lo[0], lo[1], lo[2], lo[3]);
      *reinterpret_cast<float4*>(&L.hi[pb][qb][v4]) = make_float4(hi[0], hi[1], hi[2], hi[3]);
    }
  };
  float lgn[NG][4];  // drawn for the next pass's first block during this pass's last
  auto brackets = [&](int cr, uint32_t xm, uint64_t sw, int pb) {
    float lg[NG][4];
    draw(cr, sw, lg);
    finish(cr, xm, lg, pb);
  };
  auto owner_of = [&](int c) { return 1 + c / kb; };  // matrix wave owning K block c
  // by the owner of block c, in the visit order of its next visit (mask xm),
  // so that the proposal chain starts without a permute of its own
  auto publish_bits = [&](int c, int pb, uint32_t xm) {
    const int j = c - c0;
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      const uint32_t mine = get_half<NW>(sa[tt], j);
      const uint32_t got = (uint32_t)__shfl_xor((int)mine, 32, 64);  // the other half
      const uint32_t bits = block_of<I8>(mine, got);
      if (lane < 32) L.bb[pb][qtt[tt]] = BR ? xor_permute_bits(bits, xm) : bits;
    }
  };

  // Visit schedule of sweep counter swn into parity par (wave 7, one lane
  // per step): the block visited at step t and that block's in-block mask.
  auto fill_sched = [&](int par, uint64_t swn, bool dry) {
    if (lane < nblk) {
      int bo = lane;
      uint32_t mk = 0;
      if (p.order == kBlockRandom && !dry) {
        const FeistelKey fk = block_order_key((uint32_t)nblk, swn, p.k0, p.k1);
        bo = (int)feistel_perm(fk, (uint32_t)lane);
        mk = block_mask(swn, (uint32_t)bo, p.k0, p.k1);
      }
      L.sch[par][lane] = (uint16_t)(bo | (mk << 8));
    }
  };
  // The entry of a step: block (low byte) and mask, one LDS read for both.
  // Reads are volatile so that each use reloads the entry (a short LDS read)
  // instead of keeping it live in scalar registers across the block's work.
  auto sched_entry = [&](int par, int step) -> uint32_t {
    if (!BR) return (uint32_t)step;
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)*(volatile uint16_t*)&L.sch[par][step]);
  };
  auto entry_block = [](uint32_t e) { return BR ? (int)(e & 0xffu) : (int)e; };
  auto entry_mask = [](uint32_t e) { return BR ? e >> 8 : 0u; };

  // Passes over the blocks.  Every `refresh` sweeps (p.refresh > 0 and
  // S > refresh) a dry pass recomputes the energy: the tracked energy adds
  // each sweep's accepted changes (simulation.py:157-158), and each change
  // carries the f32 rounding of the matrix-product fields, which
  // random-walks over millions of flips (the reference recomputes each field
  // from its coupling row).  A dry pass runs the pipeline over every block
  // with the proposals switched off, so each block's fields are the full
  // products F = J s of the current state (with the couplings the products
  // use); wave 0 sums E = s.(F/2 + h) in f64 and resets the tracked energy
  // to it plus the offset the caller's initial energy had from the dry pass
  // before the first sweep (zero unless the caller passed other energies).
  // Integer couplings are exact either way.  Passes: a dry pass, then
  // `refresh` sweeps and a dry pass, repeated; no dry pass after the last
  // sweep.  pass_info gives a pass's kind and its sweep (for a dry pass the
  // sweep that follows it).
  const int kre = p.refresh;
  const bool rec = kre > 0 && p.S > kre;
  const int npass = rec ? p.S + 1 + (p.S - 1) / kre : p.S;
  auto pass_info = [&](int ps, int& s_out) -> bool {
    if (!rec) {
      s_out = ps;
      return false;
    }
    if (ps == 0) {
      s_out = 0;
      return true;
    }
    const int qq = ps - 1, bq = qq / (kre + 1), rq = qq - bq * (kre + 1);
    if (rq == kre) {
      s_out = (bq + 1) * kre;
      return true;
    }
    s_out = bq * kre + rq;
    return false;
  };

  // ---- prologue: the fields of the first block in full, its brackets and spins
  {
    int s0;
    const bool dry0 = pass_info(0, s0);
    if (BR && w == 7) fill_sched(0, (uint64_t)s0 + p.sweep_offset, dry0);
  }
  __syncthreads();  // wave 0's betas (L.rb) and the schedule are visible
  {
    int s0;
    (void)pass_info(0, s0);
    const uint64_t sw0 = (uint64_t)s0 + p.sweep_offset;
    const uint32_t ef = sched_entry(0, 0), es = sched_entry(0, 1);
    const int cf = entry_block(ef), cs = entry_block(es);
    const uint32_t mf = entry_mask(ef), ms = entry_mask(es);
    if (mw) {
      prefetch_frags(cf, mf);
      compute_part(cf, mf, -1, 0);
      prefetch_frags(cs, ms);
      if (w == owner_of(cf)) publish_bits(cf, 0, mf);
    }
    if (hw) {
      prefetch_jb(cf, mf);
      publish_block(0);
      prefetch_jb(cs, ms);
      sweep_factors();
      brackets(cf, mf, sw0, 0);
    }
  }
  __syncthreads();

  const float cu = (p.ptype == 0) ? 2.f : 1.f;  // |dn / (F + h)|
  // F = fsc * (sum of the partial products + rsb) + h: QUBO with bf16
  // operands used +-1 spins, F = (J.s + J.1) / 2 with the row sums J.1 in
  // rsb (zero otherwise); fsc is a power of two, so the fma rounds like the add
  const bool qsum = !I8 && p.ptype == 1;
  const float fsc = qsum ? 0.5f : 1.f;
  // batched: field = bsc * count + h, the scale of the proposal wave's instance
  const float bsc = BAT ? (w == 0 ? tile(0).scale : tile(NI - 1).scale) : 1.f;
  double eoff = 0.0;  // wave 0: caller's initial energy minus its recomputation

  // The correction J[c1, c] . S_c of the next block c1 by a proposal wave,
  // once block c's spins are final: the A fragments of row block c1, K block
  // c (rows in the visit order of c1, lx as in load_stage) were loaded into fa
  // at the block's start, and the product stays in its registers.
  typedef Frag FragSet[NST][NP];
  auto load_corr_frags = [&](int c1, int c, int lx, int ti, FragSet& fa) {
    const Frag* fb = frag_base(ti);
#pragma unroll
    for (int st = 0; st < NST; ++st)
#pragma unroll
      for (int pc = 0; pc < NP; ++pc) {
        const size_t f = I8 ? (size_t)c1 * nblk + c
                            : ((size_t)c1 * (2 * nblk) + 2 * c + st) * NP + pc;
        fa[st][pc] = fb[f * 64 + lx];
      }
  };

  uint32_t t = 0;                               // running block counter
  // The roles run separate copies of the block loop (so that each keeps only
  // its own state in registers); all pass the same barriers: one after the
  // block's work (B), and at the end of a pass one more (three after a sweep).
  if (pw) {
    // schedule entries of this step and the next; the one after is read each
    // block and made wave-uniform at the block's end
    const uint32_t e0 = sched_entry(0, 0), e1 = sched_entry(0, 1);
    int c = entry_block(e0), c1 = entry_block(e1);
    uint32_t xm = entry_mask(e0), xm1 = entry_mask(e1);
    const int tw = w == 0 ? 0 : NT - 1;    // the wave's tile
    const int ti = BAT ? tw : 0;           // its instance
    const int qp = 32 * tw + (lane & 31);  // the lane's replica of the group
    const int np = n_of(ti);
    // the block before: its fragments of J[c, c_prev] and its final spins (block
    // rows); their product, the correction, is taken while the partials are read
    FragSet fcorr;
#pragma unroll
    for (int st = 0; st < NST; ++st)
#pragma unroll
      for (int pc = 0; pc < NP; ++pc) fcorr[st][pc] = Frag{};
    uint32_t mbr = 0;
    for (int ps = 0; ps < npass; ++ps) {
      int s;
      const bool dry = pass_info(ps, s);
      const uint64_t sw = (uint64_t)s + p.sweep_offset;
      const int sp = ps & 1;
      double dsum = 0.0, eacc = 0.0;
      uint32_t nacc = 0;
      for (int tb = 0; tb < nblk; ++tb, ++t) {
        const int pb = t & 1;
        // block c of this step, its visit k being block row k ^ xm; c1 the next
        const int pos0 = 32 * c;
        const bool lastb = tb + 1 == nblk;
        const int p2 = tb + 2 < nblk ? sp : sp ^ 1, i2 = tb + 2 < nblk ? tb + 2 : tb + 2 - nblk;
        const uint32_t raw2 = BR ? (uint32_t)*(volatile uint16_t*)&L.sch[p2][i2] : (uint32_t)i2;
        // the spins of the block's visits, in either half of the wave
        uint32_t mb = L.bb[pb][qp];
        // the partial fields and the brackets of the lane's visits (slot 4 m + e
        // is visit 8 m + 4 h + e)
        float hib[16], lob[16];
        float4 x[4][MW];
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4)
#pragma unroll
          for (int mm = 0; mm < MW; ++mm) x[g4][mm] = L.part[pb][mm][tw][g4][lane];
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const float4 a = *reinterpret_cast<const float4*>(&L.hi[pb][qp][8 * g4 + 4 * h]);
          const float4 b = *reinterpret_cast<const float4*>(&L.lo[pb][qp][8 * g4 + 4 * h]);
          hib[4 * g4] = a.x, hib[4 * g4 + 1] = a.y, hib[4 * g4 + 2] = a.z, hib[4 * g4 + 3] = a.w;
          lob[4 * g4] = b.x, lob[4 * g4 + 1] = b.y, lob[4 * g4 + 2] = b.z, lob[4 * g4 + 3] = b.w;
        }
        __builtin_amdgcn_sched_barrier(0);  // the reads first: the product covers their latency
        float corr[16];
        {
          f32x16 a = {};
          i32x16 ia = {};
          mfma_step(fcorr, half_of<I8>(mbr, h), a, ia);
#pragma unroll
          for (int v = 0; v < 16; ++v) corr[v] = I8 ? (float)ia[v] : a[v];
        }
        load_corr_frags(c1, c, lane ^ (int)xm1, ti, fcorr);
        if (dry) {
          // ---- dry pass: f64 energy of the block's rows from its full fields
          // (a dry pass visits every block with mask 0: visits are rows), the
          // rows' terms added in order, passed between the lane halves
          static_for<kB / 4>([&](auto gc) __attribute__((always_inline)) {
            constexpr int gr = decltype(gc)::value, g4 = gr >> 1;
            for (int e = 0; e < 4; ++e) {
              const int i = 4 * gr + e;
              if (pos0 + i < np) {
                auto el = [&](const float4& y) { return e == 0 ? y.x : e == 1 ? y.y : e == 2 ? y.z : y.w; };
                double f = (double)el(x[g4][0]);
#pragma unroll
                for (int mm = 1; mm < MW; ++mm) f += (double)el(x[g4][mm]);
                f += (double)(e == 0   ? corr[4 * g4]
                              : e == 1 ? corr[4 * g4 + 1]
                              : e == 2 ? corr[4 * g4 + 2]
                                       : corr[4 * g4 + 3]);
                if (qsum) f = 0.5 * (f + (double)L.rsb[pb][i]);
                if (BAT) f *= (double)bsc;
                const double si = ((mb >> i) & 1u) ? 1.0 : (p.ptype == 0 ? -1.0 : 0.0);
                eacc += si * (0.5 * f + (double)L.hb[pb][ti][i]);
              }
            }
            eacc = half_bcast<gr & 1>(eacc);
          });
        } else {
          // ---- proposals of block c
          // fields: the partials in order, the correction, (QUBO with bf16
          // operands) the row sums, then h (batched: the integer counts, with
          // h in hk)
          f32x16 fp;
          float hk[16];
          {
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
              float4 sm = x[g4][0];
#pragma unroll
              for (int mm = 1; mm < MW; ++mm) {
                sm.x = sm.x + x[g4][mm].x;
                sm.y = sm.y + x[g4][mm].y;
                sm.z = sm.z + x[g4][mm].z;
                sm.w = sm.w + x[g4][mm].w;
              }
              fp[4 * g4] = sm.x + corr[4 * g4];
              fp[4 * g4 + 1] = sm.y + corr[4 * g4 + 1];
              fp[4 * g4 + 2] = sm.z + corr[4 * g4 + 2];
              fp[4 * g4 + 3] = sm.w + corr[4 * g4 + 3];
            }
            if (qsum) {
#pragma unroll
              for (int g4 = 0; g4 < 4; ++g4) {
                const float4 r = *reinterpret_cast<const float4*>(&L.rsb[pb][8 * g4 + 4 * h]);
                fp[4 * g4] += r.x, fp[4 * g4 + 1] += r.y, fp[4 * g4 + 2] += r.z, fp[4 * g4 + 3] += r.w;
              }
            }
            // every h zero: adding +0 would only turn a -0 into +0, which no
            // decision or sum distinguishes
            if (BAT || qsum || !p.hzero) {
#pragma unroll
              for (int g4 = 0; g4 < 4; ++g4) {
                const float4 r = *reinterpret_cast<const float4*>(&L.hb[pb][ti][8 * g4 + 4 * h]);
                const float hv[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  if constexpr (BAT)
                    hk[4 * g4 + e] = hv[e];
                  else
                    fp[4 * g4 + e] = __builtin_fmaf(fsc, fp[4 * g4 + e], hv[e]);
                }
              }
            }
          }
          const uint32_t mb0 = mb;
          // accepted flips and decisions not below their bracket, step k at bit
          // 31 - k: one add with carry each per step (tn: only the bits of the
          // lane's own visits mean anything)
          uint32_t tk = 0, tn = 0;
          // bit k of mb is only changed at step k, so every step reads its
          // spin from the block's initial bits: sign bit = !spin, magnitude cu
          const uint32_t nmb = ~mb0, cub = __float_as_uint(cu);
          uint32_t vsgn = 0x80000000u;  // kept in a register (not a literal operand)
          asm volatile("" : "+v"(vsgn));
          float dpart = 0.f;
          const double dsum0 = dsum;  // batched: the sum before the block (for a rerun)
          // The field updates of the later visits, one of two ways (MU):
          // * VALU: every decision updates the lane's later slots, rows of
          //   J[blk][blk] streaming from LDS through a ring JR rows ahead, from
          //   the first slot group a lane of either half needs.
          // * MFMA: within a 4-visit group each decision updates the fields
          //   behind it on the VALU (ff); the later groups take two visits at a
          //   time as one f32 MFMA: row v of A = J[visits][v], B = the two spin
          //   changes per replica, C = the fields, which lie in this layout
          //   already.  The instruction adds its two products one after the
          //   other, each as an fma (checked on the device against both orders
          //   and against one rounding), and the products are exact (changes
          //   are 0, +-1 or +-2), so the fields round as with one VALU update
          //   per visit.
          constexpr int JR = 2;
          const float4* jb4 = reinterpret_cast<const float4*>(L.jb[pb][ti]) + 4 * h;
          float4 jring[JR][4];
          auto load_j = [&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            // k = 8 m + 7 is done with slot group m
            if constexpr (!MU && k + 1 < kB)
              static_for<4>([&](auto mc) __attribute__((always_inline)) {
                constexpr int m4 = decltype(mc)::value;
                if constexpr (m4 >= (k + 1) >> 3) jring[k % JR][m4] = jb4[k * (kB / 4) + m4];
              });
          };
          static_for<JR>([&](auto dc) __attribute__((always_inline)) { load_j(dc); });
          const float* ja = &L.jb[pb][ti][lane];
          const float4* jg = reinterpret_cast<const float4*>(L.ji[pb][ti]);
          float a_rg[2][2];  // one group ahead of the chain
          float4 j_rg[2][3];
          auto load_group = [&](auto gc) __attribute__((always_inline)) {
            constexpr int g = decltype(gc)::value;
            if constexpr (MU && g < kB / 4) {
              if constexpr (g + 1 < kB / 4) {
                a_rg[g & 1][0] = ja[(4 * g) * kB];
                a_rg[g & 1][1] = ja[(4 * g + 2) * kB];
              }
              j_rg[g & 1][0] = jg[4 * g];
              j_rg[g & 1][1] = jg[4 * g + 1];
              j_rg[g & 1][2] = jg[4 * g + 2];
            }
          };
          load_group(std::integral_constant<int, 0>{});
          // sg = 2 s or 2x - 1 of visit k: one bit insert
          auto sign_of = [&](int k) __attribute__((always_inline)) {
            const uint32_t shk = nmb << (31 - k);
            return __uint_as_float((shk & vsgn) | (cub & ~vsgn));
          };
          static_for<kB / 4>([&](auto gc) __attribute__((always_inline)) {
            constexpr int g = decltype(gc)::value;
            constexpr int H = g & 1, j0 = 4 * (g >> 1);  // the half that holds the group, its first slot
            load_group(std::integral_constant<int, g + 1>{});
            float ff[4] = {fp[j0], fp[j0 + 1], fp[j0 + 2], fp[j0 + 3]}, dS[4];
            static_for<4>([&](auto ec) __attribute__((always_inline)) {
              constexpr int e = decltype(ec)::value, k = 4 * g + e;
              const float f = MU ? ff[e] : fp[j0 + e];
              // batched: scale * c + h of the count, a product, then a sum
              const float fk = BAT ? f * bsc + hk[j0 + e] : f;
              const float sg = sign_of(k);
              // dn = 2 s (F + h) (ising) or (2x - 1)(F + h) (qubo), exact in f32
              const float dn = fk * sg;
              // The half without visit k compares another slot; only the
              // other's word counts.  Idle lanes and padding rows have lo = hi
              // = +inf (and finite dn): never taken, never inside their bracket.
              const uint64_t tb64 = __builtin_amdgcn_ballot_w64(dn > hib[j0 + e]);
              const uint64_t ib64 = __builtin_amdgcn_ballot_w64(!(dn < lob[j0 + e]));
              const uint32_t tm = H ? (uint32_t)(tb64 >> 32) : (uint32_t)tb64;
              // the decisions as the lane mask of both halves (the vector type
              // keeps it to one scalar move)
              typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
              const uint64_t tmm = __builtin_bit_cast(uint64_t, (u32x2){tm, tm});
              // taken ? -sg : 0
              asm("v_cndmask_b32_e64 %0, 0, -%1, %2" : "=v"(dS[e]) : "v"(sg), "s"(tmm));
              if constexpr (MU) {
                if constexpr (e < 3) {
                  const float4 j4 = j_rg[g & 1][e];
                  const float jv4[4] = {j4.x, j4.y, j4.z, j4.w};
                  static_for<4>([&](auto rc) __attribute__((always_inline)) {
                    constexpr int r = decltype(rc)::value;
                    if constexpr (r > e) ff[r] = __builtin_fmaf(jv4[r], dS[e], ff[r]);
                  });
                }
                if constexpr (g + 1 < kB / 4 && (e & 1) == 1) {
                  const float b = h ? dS[e] : dS[e - 1];
                  fp = __builtin_amdgcn_mfma_f32_32x32x2f32(a_rg[g & 1][e >> 1], b, fp, 0, 0, 0);
                }
              } else {
                // every element of the row's loads counts as used, or the
                // compiler splits them into narrow ones
                static_for<4>([&](auto mc) __attribute__((always_inline)) {
                  constexpr int m4 = decltype(mc)::value;
                  if constexpr (k + 1 < kB && m4 >= (k + 1) >> 3) use_whole(jring[k % JR][m4]);
                });
                static_for<16>([&](auto rc) __attribute__((always_inline)) {
                  constexpr int r = decltype(rc)::value;
                  // slot r is a later visit in one half at least (the high
                  // one's visit is the later)
                  if constexpr (8 * (r >> 2) + 4 + (r & 3) > k) {
                    const float4 j4 = jring[k % JR][r >> 2];
                    const float jv4[4] = {j4.x, j4.y, j4.z, j4.w};
                    fp[r] = __builtin_fmaf(jv4[r & 3], dS[e], fp[r]);
                  }
                });
                load_j(std::integral_constant<int, k + JR>{});
              }
              {
                uint64_t co;  // tk = 2 tk + taken (the mask as carry-in)
                asm("v_addc_co_u32_e64 %0, %1, %2, %2, %3"
                    : "=v"(tk), "=s"(co)
                    : "v"(tk), "s"(tmm));
                asm("v_addc_co_u32_e64 %0, %1, %2, %2, %3"
                    : "=v"(tn), "=s"(co)
                    : "v"(tn), "s"(ib64));
                (void)co;
              }
              // dS * fk is exactly -dn or 0, so this rounds like dpart - dn
              // (batched: summed in f64 in visit order, as the oracle sums)
              if constexpr (BAT)
                dsum += (double)(dS[e] * fk);
              else
                dpart = __builtin_fmaf(dS[e], fk, dpart);
            });
            // the sum so far goes to the half of the next group's visits
            if constexpr (BAT)
              dsum = half_bcast<H>(dsum);
            else
              dpart = half_bcast<H>(dpart);
          });
          // a decision not below its bracket and not taken is inside; bits of the
          // lane's own visits (k / 4 even or odd, bit 31 - k)
          const uint32_t own = h ? 0x0F0F0F0Fu : 0xF0F0F0F0u;
          const bool inside = __builtin_amdgcn_ballot_w64(((tn & ~tk) & own) != 0) != 0;
          mb = mb0 ^ __builtin_bitreverse32(tk);
          if (__builtin_expect(inside, 0)) {
            // A decision fell inside its bracket: rerun the block, taking the
            // exact test for the decisions inside their brackets (rolled loop,
            // fields staged in LDS; both lanes of a replica do the same).
            float* sf = &L.sfp[qp * 33];
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
              float4 v = L.part[pb][0][tw][g4][lane];
#pragma unroll
              for (int mm = 1; mm < MW; ++mm) {
                const float4 y = L.part[pb][mm][tw][g4][lane];
                v.x = v.x + y.x, v.y = v.y + y.y, v.z = v.z + y.z, v.w = v.w + y.w;
              }
              const float vs[4] = {v.x + corr[4 * g4], v.y + corr[4 * g4 + 1], v.z + corr[4 * g4 + 2],
                                   v.w + corr[4 * g4 + 3]};
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int r = 8 * g4 + 4 * h + e;
                sf[r] = BAT ? vs[e] : __builtin_fmaf(fsc, vs[e] + L.rsb[pb][r], L.hb[pb][ti][r]);
              }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const float beta = L.rb[qp];
            const int glp = BAT ? (lane & 31) / R : qp / R;  // its read of the tile / group
            const int rdp = BAT ? tile(ti).read0 + glp : read0 + glp;
            const bool actp = glp < p.rpw && rdp < (BAT ? tile(ti).read_end : p.reads);
            const uint64_t cidp = (uint64_t)rdp * R + (BAT ? (lane & 31) - glp * R : qp - glp * R);
            mb = mb0;
            dpart = 0.f;
            if constexpr (BAT) dsum = dsum0;
            for (int k = 0; k < kB; ++k) {
              const bool up = (mb >> k) & 1u;
              const float sg = up ? cu : -cu;
              const float fk = BAT ? sf[k] * bsc + L.hb[pb][ti][k] : sf[k];
              const float dn = fk * sg;
              // idle lanes and padding rows have lo = hi = +inf: never taken
              bool take = actp & (dn > L.hi[pb][qp][k]);
              if (actp && !take && !(dn < L.lo[pb][qp][k])) {
                const uint32_t pk = (uint32_t)(pos0 + (k ^ (int)xm));
                const uint32_t wd = pick_word(sweep_block(cidp, sw, pk, p.k0, p.k1), pk & 3u);
                take = accept_exact(wd, beta, dn);
              }
              mb ^= (uint32_t)take << k;
              if constexpr (BAT)
                dsum += take ? (double)(-dn) : 0.0;
              else
                dpart += take ? -dn : 0.f;
              const float dS = take ? -sg : 0.f;
              for (int r = k + 1; r < kB; ++r)
                sf[r] = __builtin_fmaf(!MU                    ? L.jb[pb][ti][k * kB + half_slot(r)]
                                       : (r >> 2) == (k >> 2) ? L.ji[pb][ti][4 * k + (r & 3)]
                                                              : L.jb[pb][ti][k * kB + r],
                                       dS, sf[r]);
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
          }
          if constexpr (!BAT) dsum += (double)dpart;
          nacc += (uint32_t)__builtin_popcount(mb ^ mb0);
        }
        mbr = BR ? xor_permute_bits(mb, xm) : mb;  // back to block-row order
        if (lane < 32) {
          L.bnew[pb][qp] = mbr;
          // the same block next (at a pass boundary): its spins are these, in
          // its next visit order (the owners, whose copy is older, skip it)
          if (c1 == c) L.bb[pb ^ 1][qp] = BR ? xor_permute_bits(mbr, xm1) : mbr;
        }
        // the next step's block and the one after it
        c = c1, xm = xm1;
        const uint32_t e2 = BR ? (uint32_t)__builtin_amdgcn_readfirstlane((int)raw2) : raw2;
        c1 = entry_block(e2), xm1 = entry_mask(e2);
        if (lastb && lane < 32) {
          L.ds[qp] = dry ? eacc : dsum;
          L.nacc[qp] = nacc;
        }
        if (dry) {
          __syncthreads();  // B
          if (lastb) {
            if (w == 0 && act) {
              if constexpr (AIS) {
                if (ps == 0)
                  eoff = Ed - L.ds[q];
                else
                  Ed = L.ds[q] + eoff;
              } else {
                if (ps == 0)
                  eoff = (double)E - L.ds[q];
                else
                  E = (float)(L.ds[q] + eoff);
              }
            }
            __syncthreads();  // the next pass's first brackets
          }
          continue;
        }
        __syncthreads();  // B
        if (AIS && lastb) {
          if (w != 0) {
            __syncthreads();
            __syncthreads();
            __syncthreads();
            continue;
          }
          // ---- end of an AIS step (simulation.py:305-316 with the uniform
          // reference: its log-density is 0): the energy after the sweep, the
          // weight of this step (ordering 0) or of the next one before its
          // sweep (ordering 1), and the next step's beta for every chain
          acc += L.nacc[q];
          Ed = Ed + L.ds[q];
          const double bt = (double)p.temps[s];
          if (act && p.ordering == 0) lw = lw + ((-bt * Ed) - (-bold * Ed));
          bold = bt;
          const bool more = s + 1 < p.S;
          const float tn = more ? p.temps[s + 1] : 0.f;
          if (act && p.ordering == 1 && more) lw = lw + ((-(double)tn * Ed) - (-bold * Ed));
          L.rb[q] = act ? tn : 0.f;
          __syncthreads();
          __syncthreads();
          __syncthreads();  // the next pass's first brackets
        } else if (lastb) {
          if (w != 0) {
            __syncthreads();
            __syncthreads();
            __syncthreads();
            continue;
          }
          // ---- end of sweep: energy (simulation.py:157-158), best states, PT
          // (lane = replica)
          acc += L.nacc[q];
          E = (float)((double)E + L.ds[q]);
          L.E[q] = E;
          if (p.best_sem == 0) {  // simulation.py:161-164
            const bool imp = act && (E < bestE);
            if (imp) {
              bestE = E;
              p.best_rep_e[(size_t)read * R + rr] = E;
              p.best_rep_sw[(size_t)read * R + rr] = s;
            }
            L.flag[q] = imp ? 1 : 0;
          }
          __syncthreads();
          // lane b0 + k: the energy of the replica in slot k (the walk below
          // reads the slots in order; the replicas' energies do not change).
          // The lane offsets are derived here from an opaque copy of the lane
          // index: hoisted to the kernel start they were kept in scratch.
          int qx = q;
          asm volatile("" : "+v"(qx));
          const int tx = BAT && NT == 2 ? (qx >> 5) : 0;
          const int b0 = BAT ? 32 * tx + ((qx & 31) / R) * R : (qx / R) * R;  // the read's first lane
          const int slot = qx - b0;
          const float* bet = &L.bet[32 * tx];
          int occ = L.bi[qx];  // the replica in the lane's slot
          if (p.best_sem == 1 && act && rr == 0) {  // simulation.py:222-225 in replica order
            int src = -1;
            float cur = gE;
            float en = L.E[b0];
            for (int k = 0; k < R; ++k) {
              const float ek = en;
              if (k + 1 < R) en = L.E[b0 + k + 1];  // the next one, read ahead
              if (ek < cur) {
                cur = ek;
                src = k;
              }
            }
            if (src >= 0) {
              gE = cur;
              gsw = s;
              gimp = 1;
            }
            L.src[g] = src;
          }
          if (p.use_pt && R > 1) {  // utils.py:44-58
            // Hot end first: at slot a the carried replica (at first slot R - 1's)
            // meets the occupant of slot a - 1 from before the walk; exchanged,
            // it is carried on to a - 1, otherwise it stays in a and that
            // occupant becomes the carried one.  Which replica is carried at a
            // slot is serial, but not how far each would be carried if it
            // were: every lane walks its slot's replica to where it would
            // stay (to), four slots at a time, and then the carried ones are
            // read off from the hot end, S = slots where one is picked up (a
            // read's last one leads on to the read below it; idle lanes stay
            // where they are).  R = 32: 6.6 -> 2.3 k cycles a sweep (one lane
            // per read walking all slots before).
            const int below = L.bi[max(qx - 1, 0)];  // of the slot below
            const float es = L.E[b0 + occ];
            // (a read's last slot and idle lanes: no exchange)
            L.wl[4 + qx] = make_float4(L.E[lane_below(b0, below)], bet[slot] - bet[max(slot - 1, 0)],
                                       act && slot > 0 ? L.lu[qx] : __builtin_nanf(""), 0.f);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            int to = qx;
            uint64_t go = ~0ull;  // lanes still carried, kept as a mask: no branches inside
            do {
              float4 y[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) y[i] = L.wl[4 + to - i];
              int d = 0;
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float dd = (es - y[i].x) * y[i].y;
                go &= __builtin_amdgcn_ballot_w64(dd >= y[i].z);  // dd >= 0 or log u < dd (log u < 0)
                uint64_t co;
                asm("v_addc_co_u32_e64 %0, %1, 0, %2, %3" : "=v"(d), "=s"(co) : "v"(d), "s"(go));
                (void)co;
              }
              to -= d;
            } while (go != 0);
            // S starts as every slot; a replica carried down takes out the ones
            // it passes
            uint64_t S = ~0ull, mv = __builtin_amdgcn_ballot_w64(to != qx);
            while (mv != 0) {
              const int c = 63 - __builtin_clzll(mv), d = __builtin_amdgcn_readlane(to, c);
              S &= ~((1ull << c) - (1ull << d));
              mv &= (1ull << d) - 1ull;
            }
            // the slot below one that is picked up (or below none) ends a walk
            const bool end = qx == 0 || ((S >> (qx - 1)) & 1ull) != 0;
            const int from = L.bi[qx + (int)__builtin_ctzll(S >> qx)];
            occ = end ? from : below;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (act) L.bi[qx] = occ;
          }
          // every slot's new beta to the replica now in it
          if (act) L.rb[b0 + occ] = bet[slot];
          if (p.logw && p.log_omegas) {  // ais.py:99-112 over the ascending ladder
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            // lane r: its term, then the leader adds them in order
            if (act && slot > 0) {
              const int k = L.bso[slot];
              const float en = L.E[b0 + L.bi[b0 + k]];
              const float a = -bet[k] * en;
              const double bold = slot > 1 ? (double)bet[L.bso[slot - 1]] : 0.0;
              L.ds[qx] = (double)a - (-bold * (double)en);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (act && rr == 0) {
              double lw = 0.0;
#pragma unroll 4
              for (int r = 1; r < R; ++r) lw += L.ds[b0 + r];
              p.log_omegas[(size_t)read * p.S + s] = lw;
            }
          }
          __syncthreads();
          __syncthreads();  // the next pass's first brackets
        }
      }
    }
  } else {
    // schedule entries carried from block to block: c (this step), c1 (the
    // next) and its mask; c2 (the one after) is read each block
    const uint32_t e1 = sched_entry(0, 1);
    int c = entry_block(sched_entry(0, 0)), c1 = entry_block(e1);
    uint32_t m1 = entry_mask(e1);
    for (int ps = 0; ps < npass; ++ps) {
      int s, s_next;
      const bool dry = pass_info(ps, s);
      const bool dry_next = pass_info(ps + 1, s_next);
      const uint64_t sw = (uint64_t)s + p.sweep_offset;
      const uint64_t sw_next = (uint64_t)s_next + p.sweep_offset;
      const int sp = ps & 1;
      for (int tb = 0; tb < nblk; ++tb, ++t) {
        const int pb = t & 1, pn = pb ^ 1;
        // the schedule of the next pass, needed from step nblk - 2 on
        if (BR && w == 7 && tb == 0) fill_sched(sp ^ 1, sw_next, dry_next);
        const bool last = tb + 1 == nblk;
        const int p2 = tb + 2 < nblk ? sp : sp ^ 1, i2 = tb + 2 < nblk ? tb + 2 : tb + 2 - nblk;
        // The entry two steps ahead is read here and made wave-uniform where
        // it is first needed (the prefetches at the end of the step), so the
        // step's work does not wait for the LDS read.
        const uint32_t raw2 = BR ? (uint32_t)*(volatile uint16_t*)&L.sch[p2][i2] : (uint32_t)i2;
        auto entry2 = [&]() {
          return BR ? (uint32_t)__builtin_amdgcn_readfirstlane((int)raw2) : raw2;
        };
        int c2 = 0;
        uint32_t m2 = 0;
        // ---- meanwhile: block c1's spins, fields except K block c, J / h and brackets
        if (mw) {
          // c1's spins have not changed since its last visit unless c1 == c
          // (a pass boundary), which the proposal wave publishes itself
          if (w == owner_of(c1) && c1 != c) publish_bits(c1, pn, m1);
          compute_part(c1, m1, c, pn);
          const uint32_t en2 = entry2();
          c2 = entry_block(en2);
          m2 = entry_mask(en2);
          prefetch_frags(c2, m2);
        }
        if (hw) {
          publish_block(pn);
          if (!last) {
            if (!dry) brackets(c1, m1, sw, pn);
          } else if (!dry_next) {
            draw(c1, sw_next, lgn);
          }
          const uint32_t en2 = entry2();
          c2 = entry_block(en2);
          m2 = entry_mask(en2);
          prefetch_jb(c2, m2);
          // the sweep's exchange uniforms (utils.py:57), by a helper that has
          // no brackets to compute during the last block
          if (w == 7 && last && !dry && p.use_pt && act && rr < R - 1)
            L.lu[q + R - 1 - 2 * rr] = float_above(log_u32(pick_word(  // pair rr: slot R - 1 - rr
                pt_block((uint64_t)read, sw, (uint32_t)rr, p.k0, p.k1), (uint32_t)rr & 3u)));
        }
        __syncthreads();  // B
        // ---- the owners of block c take its new spins
        if (mw && w == owner_of(c)) {
#pragma unroll
          for (int tt = 0; tt < NT; ++tt)
            set_half<NW>(sa[tt], c - c0, half_of<I8>(L.bnew[pb][qtt[tt]], h));
        }
        if (last) {
          if (!dry) {
            __syncthreads();
#pragma unroll
            for (int tt = 0; tt < NT; ++tt)
              if (!AIS && mw && p.best_sem == 0 && actt[tt] && L.flag[qtt[tt]])
                store_range<NW, I8>(sa[tt], c0, kb, nblk, n_of(tt), p.ptype,
                                    p.best_rep + base_t[tt]);
            __syncthreads();
            // owners copy their part of a new global best
#pragma unroll
            for (int tt = 0; tt < NT; ++tt)
              if (!AIS && mw && p.best_sem == 1 && actt[tt] && L.src[gtt[tt]] == rtt_of(tt))
                store_range<NW, I8>(sa[tt], c0, kb, nblk, n_of(tt), p.ptype, best_of(tt));
          }
          // the next pass's first block (after the exchanges: new betas)
          if (hw && !dry_next) {
            sweep_factors();
            finish(c1, m1, lgn, pn);
          }
          __syncthreads();
        }
        c = c1;
        c1 = c2;
        m1 = m2;
      }
    }
  }

  // ---- outputs
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
    if (actt[tt]) store_range<NW, I8>(sa[tt], c0, kb, nblk, n_of(tt), p.ptype, p.spins + base_t[tt]);
  if (AIS && w == 0 && act) {
    if (p.accepted) atomicAdd(p.accepted + read, acc);
    p.ais_e[read] = Ed;
    p.ais_w[read] = lw;
  }
  if (!AIS && w == 0 && act) {
    if (p.accepted) atomicAdd(p.accepted + read, acc);
    p.energies[(size_t)read * R + rr] = E;
    p.beta_idx[(size_t)read * R + rr] = L.bi[q];
    if (rr == 0 && p.best_sem == 1) {
      p.best_energy[read] = gE;
      p.best_sweeps[read] = gsw;
      L.src[g] = gimp;
    }
  }
  if (!AIS && p.best_sem == 1) {
    // never improved: best_state is still the view of states[0] (simulation.py:204)
    __syncthreads();
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
      if (actt[tt] && rtt_of(tt) == 0 && !L.src[gtt[tt]])
        store_range<NW, I8>(sa[tt], c0, kb, nblk, n_of(tt), p.ptype, best_of(tt));
  }
}

template <int NP, bool I8, bool BR, int NT, int MODE = kModePT>
hipError_t launch_pipe_o(const BParams& p, int nw, int groups, hipStream_t st) {
  // (batched: the sizes are checked where the workgroups' table is built)
  if (MODE != kModeBatched && !pipe_takes(BR ? kBlockRandom : kSequential, p.nblk))
    return hipErrorInvalidValue;
  dim3 grid(groups), block(128 * (kPipeMW + 1));
  switch (nw) {
    case 4: hipLaunchKernelGGL((blocked_pipe_kernel<NP, I8, 4, kPipeMW, BR, NT, MODE>), grid, block, 0, st, p); break;
    case 8: hipLaunchKernelGGL((blocked_pipe_kernel<NP, I8, 8, kPipeMW, BR, NT, MODE>), grid, block, 0, st, p); break;
    case 16: hipLaunchKernelGGL((blocked_pipe_kernel<NP, I8, 16, kPipeMW, BR, NT, MODE>), grid, block, 0, st, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Launch of one coupling encoding: nw spin words per matrix wave, nt tiles of
// 32 replicas per workgroup, the order from p.
template <int NP, bool I8>
hipError_t launch_pipe_enc(const BParams& p, int nw, int nt, int groups, hipStream_t st) {
  if (nt != 1 && nt != 2) return hipErrorInvalidValue;
  if (p.order == kBlockRandom)
    return nt == 2 ? launch_pipe_o<NP, I8, true, 2>(p, nw, groups, st)
                   : launch_pipe_o<NP, I8, true, 1>(p, nw, groups, st);
  return nt == 2 ? launch_pipe_o<NP, I8, false, 2>(p, nw, groups, st)
                 : launch_pipe_o<NP, I8, false, 1>(p, nw, groups, st);
}

// AIS (kModeAIS) with one coupling encoding: nt tiles of 32 chains per
// workgroup, the order from p.
template <int NP, bool I8>
hipError_t launch_pipe_ais_enc(const BParams& p, int nw, int nt, int groups, hipStream_t st) {
  if (p.order == kBlockRandom)
    return nt == 2 ? launch_pipe_o<NP, I8, true, 2, kModeAIS>(p, nw, groups, st)
                   : launch_pipe_o<NP, I8, true, 1, kModeAIS>(p, nw, groups, st);
  return nt == 2 ? launch_pipe_o<NP, I8, false, 2, kModeAIS>(p, nw, groups, st)
                 : launch_pipe_o<NP, I8, false, 1, kModeAIS>(p, nw, groups, st);
}

// One per translation unit (blocked_pipe_i8.hip, blocked_pipe_bf16_{1,2,3}.hip).
hipError_t launch_pipe_i8(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_bf16_1(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_bf16_2(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_bf16_3(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_ais_i8(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_ais_bf16_1(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_ais_bf16_2(const BParams& p, int nw, int nt, int groups, hipStream_t st);
hipError_t launch_pipe_ais_bf16_3(const BParams& p, int nw, int nt, int groups, hipStream_t st);
// The batched form (blocked_pipe_bat.hip): one workgroup per entry of p.bat.
hipError_t launch_pipe_bat(const BParams& p, int nw, int nt, int groups, hipStream_t st);

}  // namespace blk
}  // namespace pysa

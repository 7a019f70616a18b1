// Batched form: many independent dense instances of different sizes, all
// reads of all of them in one persistent launch.
//
// PySA has no batching across instances; a batch of problems is a Python
// loop over Solver objects, each running its reads one after another
// (pysa/sa.py:425-427 inside a caller's loop).  Per instance the chain is the
// one of pysa/simulation.py:123-236 (sweeps :41-76, update_spin
// pysa/ising.py:40-63 / pysa/qubo.py:40-63, exchange pysa/utils.py:26-58).
//
// Couplings are J = scale * S with S a symmetric zero-diagonal int8 matrix
// (+-1 signs for Sherrington-Kirkpatrick instances).  Local fields are kept
// as exact integers c = S s, so the field of spin i is scale*c_i + h_i,
// rounded once in float32 -- the correctly rounded value of the reference's
// float32 row dot J_i . s (which rounds at every partial sum in an order set
// by BLAS) -- and the fields never drift.
//
// Layout.  One workgroup per (instance, read), one wave per replica (R <= 16
// waves).  A replica's integer fields stay in VGPRs for the whole run, with
// element i in lane (i>>2)&63, slot ((i>>8)<<2)|(i&3), so an accepted flip
// adds one int8 coupling row, 4 bytes per lane per 256 elements, to every
// field.  A sweep takes its visits 64 at a time, one per lane: all decide at
// once, the first accepted one flips and passes its row through LDS to the
// visits behind it, which decide again, so a window takes as many steps as it
// has accepted flips.  Batches of at most 64 spins (what the MFMA form leaves)
// keep the couplings in LDS and the fields in visit order for the whole sweep.
// Workgroups are issued largest instance first so the tail of the launch holds
// the short ones.
#include <stdint.h>

#include "engine.hpp"
#include "rng.hpp"
#include "wave_dev.hpp"

namespace pysa {
namespace {

__device__ __forceinline__ int elem_of(int lane, int g) {
  return ((g >> 2) << 8) + (lane << 2) + (g & 3);
}

// Integer fields and spin bits of one replica (G <= 32 slots per lane).
template <int G>
struct IChain {
  int f[G];
  uint32_t bits;  // bit g: element elem_of(lane, g) is up (+1 / 1)

  // f += d * row (row: int8, zero beyond n, 16-byte aligned rows)
  __device__ __forceinline__ static void load_row(int (&x)[G / 4], const int8_t* __restrict__ row,
                                                  int n) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int g4 = 0; g4 < G / 4; ++g4) {
      const int i0 = (g4 << 8) + (lane << 2);
      x[g4] = (i0 < n) ? *reinterpret_cast<const int*>(row + i0) : 0;
    }
  }
  __device__ __forceinline__ void add_row(const int (&x)[G / 4], int d) {
#pragma unroll
    for (int g4 = 0; g4 < G / 4; ++g4)
#pragma unroll
      for (int q = 0; q < 4; ++q) f[4 * g4 + q] += d * ((x[g4] << (24 - 8 * q)) >> 24);
  }
};

// SMALL: every instance has at most 64 spins (one window of visits); the
// couplings are staged in LDS and an accepted flip updates the fields of all
// visits, so the rows are never added to the element order: the fields go to
// visit order at the start of a sweep and back at its end.
// Bound: latency, an LDS read and an f64 comparison per accepted flip (SMALL),
// one row from L2 (else).  Before, each visit picked its field by a select tree
// and waited for the last flip's row: 500 sweeps of the instances below 65
// spins of a 256-instance batch 11.8 -> 3.1 ms.
template <int G, bool SMALL>
__global__ __launch_bounds__(G >= 32 ? 512 : 1024) void batched_pt_kernel(BatchParams p) {
  const int item = p.order_map ? p.order_map[blockIdx.x] : (int)blockIdx.x;
  const int inst = item / p.reads, rd = item - inst * p.reads;
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int R = p.R, n = p.inst_n[inst], ld = p.ld[inst];
  const float sc = p.scale[inst];
  const int8_t* __restrict__ S = p.signs + p.j_off[inst];
  const int64_t so = p.s_off[inst];                      // states of this instance
  const int64_t gread = (int64_t)inst * p.reads + rd;     // global read index
  int8_t* spins = p.states + so + (int64_t)rd * R * n;
  int8_t* brep = p.best_rep + so + (int64_t)rd * R * n;
  int8_t* bstate = p.best_state + so / R + (int64_t)rd * n;
  const float* betas = p.betas + (int64_t)inst * R;

  extern __shared__ __align__(16) int s_buf[];  // 64 G per wave
  __shared__ float s_h[SMALL ? 64 : kBatchedMaxN];
  __shared__ int8_t s_S[SMALL ? 64 * 64 : 1];
  __shared__ float s_E[16], s_beta[16], s_bs[16], s_bE[16];
  __shared__ int s_bi[16];
  __shared__ double s_lu[16];
  __shared__ int s_bsw[16], s_src, s_gsw, s_imp;
  __shared__ float s_gE;
  int* buf = s_buf + r * 64 * G;
  for (int i = tid; i < n; i += blockDim.x) s_h[i] = p.h ? p.h[p.h_off[inst] + i] : 0.f;
  if constexpr (SMALL)
    for (int i = tid; i < 64 * 64; i += blockDim.x) {
      const int row = i >> 6, col = i & 63;
      s_S[i] = row < n && col < n ? S[(int64_t)row * ld + col] : (int8_t)0;
    }
  if (tid < R) {
    s_E[tid] = p.energies[gread * R + tid];
    s_bE[tid] = s_E[tid];
    s_bsw[tid] = 0;
    s_bi[tid] = tid;  // beta_idx = arange(R) (sa.py:325)
    s_beta[tid] = betas[tid];
  }
  if (tid == 0) {
    s_gE = p.energies[gread * R];  // simulation.py:205
    s_gsw = 0;
    s_imp = 0;
  }

  // Load the spins and build the exact integer fields c = S s.
  IChain<G> ch;
  ch.bits = 0;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    ch.f[g] = 0;
    const int i = elem_of(lane, g);
    if (i < n && spins[(int64_t)r * n + i] == 1) ch.bits |= 1u << g;
  }
  for (int j = 0; j < n; ++j) {
    const int sj = spins[(int64_t)r * n + j];
    if (sj != 0) {
      int x[G / 4];
      ch.load_row(x, S + (int64_t)j * ld, n);
      ch.add_row(x, sj);
    }
  }
  if (p.best_sem == 0)
    for (int i = lane; i < n; i += 64) brep[(int64_t)r * n + i] = spins[(int64_t)r * n + i];
  __syncthreads();

  const uint64_t cid = (uint64_t)gread * R + r;
  unsigned long long acc = 0;
  for (int s = 0; s < p.S; ++s) {
    const uint64_t sw = (uint64_t)s + p.sweep_offset;
    if (tid < R) s_bs[s_bi[tid]] = s_beta[tid];  // simulation.py:151-152
    if (p.use_pt && tid < R - 1)
      s_lu[tid] = log_u32(pick_word(pt_block((uint64_t)gread, sw, (uint32_t)tid, p.k0, p.k1),
                                    (uint32_t)tid & 3u));
    __syncthreads();
    // ---- one sweep of replica r (simulation.py:41-76)
    const double bd = (double)s_bs[r];
    FeistelKey fk;
    const bool brand = p.order == kBlockRandom;
    const int nv = brand ? kOrderBlock * ((n + kOrderBlock - 1) / kOrderBlock) : n;
    if (brand)
      fk = block_order_key((uint32_t)((n + kOrderBlock - 1) / kOrderBlock), sw, p.k0, p.k1);
    else if (p.order != kSequential)
      fk = feistel_make((uint32_t)n, perm_keys(p.order == kRandomShared ? 0ull : cid, sw,
                                               p.order == kRandomShared ? kStreamShared
                                                                        : kStreamPerm,
                                               p.k0, p.k1));
    double sum = 0.0;
    for (int w = 0; w < nv; w += 64) {
      const int vi = w + lane;
      int pos_l = -1;
      double lr_l = 0.0;
      if (vi < nv) {
        if (brand)
          pos_l = block_random_pos(fk, sw, (uint32_t)vi, n, p.k0, p.k1);
        else
          pos_l = (p.order == kSequential) ? vi : (int)feistel_perm(fk, (uint32_t)vi);
        if (pos_l >= 0)
          lr_l = log_u32(pick_word(sweep_block(cid, sw, (uint32_t)pos_l, p.k0, p.k1),
                                   (uint32_t)pos_l & 3u));
      }
      const int pc = max(pos_l, 0);
      const uint64_t valid = __ballot(pos_l >= 0);
      const float hl = s_h[pc];
      // counts and spins of the visits
#pragma unroll
      for (int g4 = 0; g4 < G / 4; ++g4)
        reinterpret_cast<int4*>(buf)[(g4 << 6) + lane] =
            make_int4(ch.f[4 * g4], ch.f[4 * g4 + 1], ch.f[4 * g4 + 2], ch.f[4 * g4 + 3]);
      wave_sync();
      int c = buf[pc];
      const bool up =
          ((uint32_t)__shfl((int)ch.bits, (pc >> 2) & 63, 64) >> (((pc >> 8) << 2) | (pc & 3))) & 1u;
      const uint64_t upm = __ballot(up);
      wave_sync();
      // dn = 2 s (F + h) (ising.py:48-49) or (2x - 1)(F + h) (qubo.py:48-49)
      const double sg = p.ptype == 0 ? (up ? 2.0 : -2.0) : (up ? 1.0 : -1.0);
      double dn;
      auto decisions = [&]() __attribute__((always_inline)) {  // ising.py:52
        const float fh = (float)c * sc + hl;
        dn = sg * (double)fh;
        return __builtin_amdgcn_ballot_w64(dn >= 0.0) | __builtin_amdgcn_ballot_w64(lr_l < bd * dn);
      };
      uint64_t m = decisions() & valid, taken = 0;
      while (m) {
        const int t = __builtin_ctzll(m);
        const int pos = rl(pos_l, t);
        const bool upt = (upm >> t) & 1;
        const int d = p.ptype == 0 ? (upt ? -2 : 2) : (upt ? -1 : 1);
        const double dnt = rl(dn, t);
        taken |= 1ull << t;
        if constexpr (SMALL) {
          c += d * (int)s_S[pos * 64 + pc];
        } else {
          int x[G / 4];
          ch.load_row(x, S + (int64_t)pos * ld, n);
#pragma unroll
          for (int g4 = 0; g4 < G / 4; ++g4) buf[(g4 << 6) + lane] = x[g4];  // byte i: coupling i
          wave_sync();
          c += d * (int)reinterpret_cast<const int8_t*>(buf)[pc];
          ch.add_row(x, d);
          wave_sync();
          if (lane == ((pos >> 2) & 63)) ch.bits ^= 1u << (((pos >> 8) << 2) | (pos & 3));
        }
        m = decisions() & valid & (~1ull << t);
        sum += -dnt;
      }
      acc += (unsigned long long)__builtin_popcountll(taken);
      if constexpr (SMALL) {  // one window: counts and spins back to element order
        if (pos_l >= 0) {
          buf[pos_l] = c;
          buf[64 + pos_l] = (int)(up != (bool)((taken >> lane) & 1));
        }
        wave_sync();
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int i = elem_of(lane, g);
          if (i < n) {
            ch.f[g] = buf[i];
            ch.bits = (ch.bits & ~(1u << g)) | ((uint32_t)buf[64 + i] << g);
          }
        }
        wave_sync();
      }
    }
    const float en = (float)((double)s_E[r] + sum);  // simulation.py:157-158
    if (p.best_sem == 0 && en < s_bE[r]) {  // simulation.py:161-164
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int i = elem_of(lane, g);
        if (i < n)
          brep[(int64_t)r * n + i] = ((ch.bits >> g) & 1u) ? 1 : (p.ptype == 0 ? -1 : 0);
      }
      if (lane == 0) {
        s_bE[r] = en;
        s_bsw[r] = s;
      }
    }
    if (lane == 0) s_E[r] = en;
    __syncthreads();
    if (r == 0) {
      if (p.best_sem == 1 && lane == 0) {  // simulation.py:222-225 in replica order
        int src = -1;
        float cur = s_gE;
        for (int k = 0; k < R; ++k)
          if (s_E[k] < cur) {
            cur = s_E[k];
            src = k;
          }
        if (src >= 0) {
          s_gE = cur;
          s_gsw = s;
          s_imp = 1;
        }
        s_src = src;
      }
      if (p.use_pt) exchange_wave<float, int>(R, s_E, s_beta, s_lu, s_bi);
    }
    __syncthreads();
    if (p.best_sem == 1 && s_src == r) {  // the improving replica copies itself
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int i = elem_of(lane, g);
        if (i < n) bstate[i] = ((ch.bits >> g) & 1u) ? 1 : (p.ptype == 0 ? -1 : 0);
      }
    }
  }

  // Outputs.
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int i = elem_of(lane, g);
    if (i < n) spins[(int64_t)r * n + i] = ((ch.bits >> g) & 1u) ? 1 : (p.ptype == 0 ? -1 : 0);
  }
  if (p.accepted && lane == 0) atomicAdd(p.accepted + gread, acc);
  __syncthreads();
  if (tid < R) {
    p.beta_idx[gread * R + tid] = s_bi[tid];
    p.energies[gread * R + tid] = s_E[tid];
  }
  if (tid == 0) {
    if (p.best_sem == 0) {  // simulation.py:174-177, first minimum wins
      int bp = 0;
      for (int k = 1; k < R; ++k)
        if (s_bE[k] < s_bE[bp]) bp = k;
      s_src = bp;
      p.best_energy[gread] = s_bE[bp];
      p.best_sweeps[gread] = s_bsw[bp];
    } else {
      s_src = s_imp ? -1 : 0;  // not improved: best_state is the view of states[0] (:204)
      p.best_energy[gread] = s_gE;
      p.best_sweeps[gread] = s_gsw;
    }
  }
  __syncthreads();
  if (s_src >= 0) {
    const int8_t* src = (p.best_sem == 0 ? brep : spins) + (int64_t)s_src * n;
    for (int i = tid; i < n; i += blockDim.x) bstate[i] = src[i];
  }
}

}  // namespace

int batched_regs_for(int max_n) {
  int g = 4;
  while (64 * g < max_n) g *= 2;
  return g;
}

hipError_t launch_batched(const BatchParams& p, int items, int max_n, hipStream_t st) {
  if (items < 1) return hipSuccess;
  if (max_n < 1 || max_n > kBatchedMaxN || p.R < 1 || p.R > 16) return hipErrorInvalidValue;
  if (batched_regs_for(max_n) >= 32 && p.R > 8) return hipErrorInvalidValue;
  const dim3 grid((unsigned)items), block((unsigned)(64 * p.R));
  const int G = batched_regs_for(max_n);
  const size_t lds = (size_t)p.R * 64 * G * sizeof(int);
  if (max_n <= 64)
    hipLaunchKernelGGL((batched_pt_kernel<4, true>), grid, block, lds, st, p);
  else
    switch (G) {
      case 4: hipLaunchKernelGGL((batched_pt_kernel<4, false>), grid, block, lds, st, p); break;
      case 8: hipLaunchKernelGGL((batched_pt_kernel<8, false>), grid, block, lds, st, p); break;
      case 16: hipLaunchKernelGGL((batched_pt_kernel<16, false>), grid, block, lds, st, p); break;
      case 32: hipLaunchKernelGGL((batched_pt_kernel<32, false>), grid, block, lds, st, p); break;
      default: return hipErrorInvalidValue;
    }
  return hipGetLastError();
}

}  // namespace pysa

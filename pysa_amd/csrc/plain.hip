// Plain form of the engine: the drop-in for PySA's Metropolis sweep.
//
// Reference path (what these kernels replace):
//   pysa/simulation.py:123-236  simulation_parallel / simulation_sequential
//   pysa/simulation.py:41-76    random_sweep / sequential_sweep
//   pysa/ising.py:40-63, pysa/qubo.py:40-63  update_spin
//   pysa/utils.py:26-58         pt
//   pysa/ais.py:79-112          get_log_omega
//   pysa/simulation.py:266-317  ais_simulation_parallel / ais_sample
//
// Layout.  A wave carries one chain at a time.  A chain's local fields F = J s
// live in VGPRs: element i sits in lane (i>>2)&63, register slot
// ((i>>8)<<2)|(i&3), so four consecutive slots of a lane hold four consecutive
// elements and a coupling row moves as 16-byte vectors.  Spins are one bit per
// slot.
//
// A sweep takes its visits 64 at a time, one per lane (sweep_dense): every
// lane holds the field of its visit and decides at once; the first accepted
// visit flips, its coupling row updates the fields of the visits behind it,
// and they decide again.  So rejected proposals cost nothing by themselves,
// and a window takes as many steps as it has accepted flips.  The additions
// to every field happen in the order of the flips, as one visit after another
// would make them, so the results equal that to the bit.
//
// Where the chains run (plan_plain): one workgroup per read that carries all
// replicas through the whole run and meets at a barrier once per sweep, or,
// when that leaves most of the device idle, one workgroup per chain with the
// exchanges in a launch of their own after every sweep.
#include <type_traits>

#include "engine.hpp"
#include "rng.hpp"
#include "wave_dev.hpp"

namespace pysa {
namespace {

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Element <-> (lane, slot) map of the field layout.
__device__ __forceinline__ int elem_of(int lane, int g) {
  return ((g >> 2) << 8) + (lane << 2) + (g & 3);
}
__device__ __forceinline__ int lane_of(int i) { return (i >> 2) & 63; }
__device__ __forceinline__ int slot_of(int i) { return ((i >> 8) << 2) | (i & 3); }

__device__ __forceinline__ uint32_t shfl_bits(uint32_t w, int src) {
  return (uint32_t)__shfl((int)w, src, 64);
}
__device__ __forceinline__ uint64_t shfl_bits(uint64_t w, int src) {
  const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)w, src, 64);
  const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(w >> 32), src, 64);
  return ((uint64_t)hi << 32) | lo;
}

// x dS + f for dS a power of two: rounds like the product and the sum.
__device__ __forceinline__ float fma_t(float x, float dS, float f) { return __builtin_fmaf(x, dS, f); }
__device__ __forceinline__ double fma_t(double x, double dS, double f) { return __builtin_fma(x, dS, f); }

template <typename T>
struct alignas(4 * sizeof(T)) T4 {
  T v[4];
};

// One chain: G field registers per lane (G a multiple of 4, n <= 64*G).
template <int G>
struct BitsFor {
  using type = uint64_t;
};
template <>
struct BitsFor<4> {
  using type = uint32_t;
};
template <>
struct BitsFor<8> {
  using type = uint32_t;
};
template <>
struct BitsFor<16> {
  using type = uint32_t;
};
template <>
struct BitsFor<32> {
  using type = uint32_t;
};

template <typename T, int G>
struct Chain {
  using B = typename BitsFor<G>::type;
  T f[G];
  B bits;  // bit g: the spin of element elem_of(lane, g) is up (+1 / 1)

  __device__ void load_spins(const int8_t* s, int n) {
    const int lane = threadIdx.x & 63;
    bits = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int i = elem_of(lane, g);
      f[g] = T(0);
      if (i < n && s[i] == 1) bits |= (B(1) << g);
    }
  }
  __device__ void load(const T* F, const int8_t* s, int n) {
    const int lane = threadIdx.x & 63;
    load_spins(s, n);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int i = elem_of(lane, g);
      if (i < n) f[g] = F[i];
    }
  }
  __device__ void store(T* F, int8_t* s, int n, int ptype) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int i = elem_of(lane, g);
      if (i < n) {
        F[i] = f[g];
        s[i] = ((bits >> g) & 1) ? int8_t(1) : (ptype == 0 ? int8_t(-1) : int8_t(0));
      }
    }
  }
  __device__ void store_spins(int8_t* s, int n, int ptype) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int i = elem_of(lane, g);
      if (i < n) s[i] = ((bits >> g) & 1) ? int8_t(1) : (ptype == 0 ? int8_t(-1) : int8_t(0));
    }
  }
  __device__ bool up_at(int pos) const { return (rl(bits, lane_of(pos)) >> slot_of(pos)) & 1; }

  // f[g] for a wave-uniform slot g, as a select tree on g's bits: register
  // indices stay compile-time constants, so the fields never leave VGPRs.
  __device__ __forceinline__ T pick(int g) const {
    T v[G];
#pragma unroll
    for (int k = 0; k < G; ++k) v[k] = f[k];
#pragma unroll
    for (int half = G / 2; half >= 1; half >>= 1) {
      const bool hi = (g & half) != 0;
#pragma unroll
      for (int k = 0; k < half; ++k) v[k] = hi ? v[k + half] : v[k];
    }
    return v[0];
  }

  // F = J s accumulated in f64 and rounded once to T; returns
  // E = s.(F/2 + h) in f64 (the periodic recomputation that bounds drift).
  // Rows of J^T padded with zeros to ldp, eight in flight.
  __device__ double refresh(const T* __restrict__ Jp, int ldp, const T* h, int n, int ptype) {
    const int lane = threadIdx.x & 63;
    double e = 0.0;
#pragma unroll
    for (int g4 = 0; g4 < G / 4; ++g4) {
      double a[4] = {0.0, 0.0, 0.0, 0.0};
      const int i0 = (g4 << 8) + (lane << 2);
      if ((g4 << 8) < ldp) {
        for (int j0 = 0; j0 < n; j0 += 8) {
          T4<T> x[8];
#pragma unroll
          for (int u = 0; u < 8; ++u)
            x[u] = *reinterpret_cast<const T4<T>*>(Jp + (size_t)min(j0 + u, n - 1) * ldp + i0);
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            if (j0 + u >= n) break;
            const bool upj = up_at(j0 + u);
            if (ptype == 1 && !upj) continue;
            const double sj = upj ? 1.0 : -1.0;
#pragma unroll
            for (int q = 0; q < 4; ++q) a[q] += (double)x[u].v[q] * sj;
          }
        }
      }
      e = put_fields(g4, a, h, n, ptype, e);
    }
    return wave_sum(e);
  }
  // Slots 4 g4 .. 4 g4 + 3 from their f64 sums; returns e plus their terms of
  // the energy, in slot order.
  __device__ __forceinline__ double put_fields(int g4, const double (&a)[4], const T* h, int n,
                                               int ptype, double e) {
    const int i0 = (g4 << 8) + ((threadIdx.x & 63) << 2);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int g = 4 * g4 + q;
      f[g] = (T)a[q];
      if (i0 + q < n) {
        const double si = ((bits >> g) & 1) ? 1.0 : (ptype == 0 ? -1.0 : 0.0);
        e += si * (0.5 * a[q] + (double)h[i0 + q]);
      }
    }
    return e;
  }

  // The same from the nonzeros of a symmetric J (sparse form): row i's
  // entries in ascending column order, so the f64 sums equal the dense
  // ones term for term (a zero coupling adds exactly nothing).
  __device__ double refresh_ell(const int* __restrict__ cols, const T* __restrict__ vals, int D,
                                const T* h, int n, int ptype) {
    const int lane = threadIdx.x & 63;
    double e = 0.0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int i = elem_of(lane, g);
      double a = 0.0;
      for (int k = 0; k < D; ++k) {
        const int j = (i < n) ? cols[(size_t)i * D + k] : -1;
        // every lane takes part in the exchange (a disabled source lane reads as zero)
        const B w = shfl_bits(bits, lane_of(j < 0 ? 0 : j));
        if (j < 0) continue;
        const bool upj = (w >> slot_of(j)) & 1;
        if (ptype == 1 && !upj) continue;
        a += (double)vals[(size_t)i * D + k] * (upj ? 1.0 : -1.0);
      }
      f[g] = (T)a;
      if (i < n) {
        const double si = ((bits >> g) & 1) ? 1.0 : (ptype == 0 ? -1.0 : 0.0);
        e += si * (0.5 * a + (double)h[i]);
      }
    }
    return wave_sum(e);
  }

  // Add m to f[g] for a wave-uniform slot g (a scalar branch tree on g's
  // bits, so the register index stays a compile-time constant).
  template <int LO, int HI>
  __device__ __forceinline__ void add_at(int g, T m) {
    if constexpr (HI - LO == 1) {
      f[LO] += m;
    } else {
      constexpr int MID = (LO + HI) / 2;
      if (g < MID)
        add_at<LO, MID>(g, m);
      else
        add_at<MID, HI>(g, m);
    }
  }
  // Add dS times row p of a symmetric sparse J (its ELL row: d <= 64
  // entries, column -1 past the row's nonzeros): lane k loads entry k (one
  // load latency for the whole row), then each nonzero's owner lane updates
  // its register; the other lanes add zero, as the dense row would.
  __device__ __forceinline__ void add_ell(const int* __restrict__ cols,
                                          const T* __restrict__ vals, int d, T dS) {
    const int lane = threadIdx.x & 63;
    const int kl = lane < d ? lane : 0;
    const int cl = cols[kl];
    const T vl = vals[kl];
    for (int k = 0; k < d; ++k) {
      const int j = rl(cl, k);
      if (j < 0) break;
      add_at<0, G>(slot_of(j), lane == lane_of(j) ? rl(vl, k) * dS : T(0));
    }
  }

  __device__ int count_up(int n) const {
    const int lane = threadIdx.x & 63;
    int c = 0;
#pragma unroll
    for (int g = 0; g < G; ++g)
      if (elem_of(lane, g) < n) c += (int)((bits >> g) & 1);
    return wave_sum(c);
  }

  // Row pos of the couplings padded with zeros to ldp elements (a multiple of
  // 256, at most 64 G, 16-byte aligned): a 256-element chunk is loaded whole
  // or, beyond ldp, not at all (a wave-uniform test; the chunks up to G = 8 and
  // the first half above always exist, because G is the least power of two).
  __device__ __forceinline__ static void load_row(T4<T> (&x)[G / 4], const T* __restrict__ Jp,
                                                  int pos, int ldp) {
    const uint32_t row = (uint32_t)pos * (uint32_t)ldp;  // at most 4096 x 4096
    const T4<T>* r4 = reinterpret_cast<const T4<T>*>(Jp + row);
    const uint32_t lane = threadIdx.x & 63;
    constexpr int HALF = G <= 8 ? G / 4 : G / 8;
#pragma unroll
    for (int g4 = 0; g4 < HALF; ++g4) x[g4] = r4[(g4 << 6) + lane];
    if (HALF == G / 4 || ldp == 64 * G) {
#pragma unroll
      for (int g4 = HALF; g4 < G / 4; ++g4) x[g4] = r4[(g4 << 6) + lane];
    } else {
#pragma unroll
      for (int g4 = HALF; g4 < G / 4; ++g4)
        x[g4] = ((g4 << 8) < ldp) ? r4[(g4 << 6) + lane] : T4<T>{{T(0), T(0), T(0), T(0)}};
    }
  }
  __device__ __forceinline__ void add_row(const T4<T> (&x)[G / 4], T dS) {
#pragma unroll
    for (int g4 = 0; g4 < G / 4; ++g4)
#pragma unroll
      for (int q = 0; q < 4; ++q) f[4 * g4 + q] = fma_t(x[g4].v[q], dS, f[4 * g4 + q]);
  }
  __device__ __forceinline__ void flip(int pos) {
    bits ^= (int)(threadIdx.x & 63) == lane_of(pos) ? B(1) << slot_of(pos) : B(0);
  }
};

// Decision for one proposal (ising.py:48-52 / qubo.py:48-52; with AIS the
// reference-distribution term of update_spin_ref, ising.py:75-83).
template <typename T, bool AIS>
__device__ __forceinline__ bool decide(int ptype, bool up, T fh, double lr, double bd, int ref,
                                       double lratio, double& dn) {
  dn = (ptype == 0) ? 2.0 * (up ? 1.0 : -1.0) * (double)fh
                    : (2.0 * (up ? 1.0 : 0.0) - 1.0) * (double)fh;
  if (AIS) {
    const double refd = (ref == 1) ? (up ? lratio : -lratio) : 0.0;
    const double full = bd * dn + (1.0 - bd) * refd;
    return full >= 0 || lr < full;
  }
  return dn >= 0 || lr < bd * dn;
}

// Log-uniform of (chain, position) from replay or Philox.
__device__ __forceinline__ double log_uniform(const double* rep, uint64_t chain, uint64_t sw,
                                              int pos, uint32_t k0, uint32_t k1) {
  if (rep) return rep[pos];
  return log_u32(pick_word(sweep_block(chain, sw, (uint32_t)pos, k0, k1), (uint32_t)pos & 3u));
}

constexpr int kMaxR = 1024;

// How a chain's sweep runs (the sweep variant of a kernel).
//   kWide   many chains: the rows of accepted flips pass through a wave's LDS
//           buffer of n elements to the lanes whose visits need them
//   kBlock  few chains: the 64 x 64 couplings between the visits of a window
//           are staged in LDS first, so a decision waits for LDS only, and the
//           rows are added afterwards, several in flight
//   kSparse one visit after another, an accepted flip updating the nonzeros of
//           its ELL row
constexpr int kWide = 0, kBlock = 1, kSparse = 2;

// Waves per workgroup for `regs` VGPRs of fields per lane, keeping fields and
// working registers inside the VGPR budget.
constexpr int waves_of(int regs) { return regs <= 16 ? 16 : regs <= 32 ? 8 : 4; }
template <typename T, int G>
constexpr int kernel_waves() {
  return waves_of(G * (int)(sizeof(T) / 4));
}
// The sparse update and refresh need more registers per lane (half the waves).
template <typename T, int G, int V>
constexpr int pt_waves() {
  return V == kSparse && kernel_waves<T, G>() > 4 ? kernel_waves<T, G>() / 2 : kernel_waves<T, G>();
}
// A wave's LDS buffer, in elements.
template <int G, int V>
constexpr int wave_buf() {
  return V == kSparse ? 0 : V == kBlock ? 64 * 64 : 64 * G;
}

struct SweepCtx {
  int n, ptype, order, ref;
  uint32_t k0, k1;
  uint64_t sw;
  double lratio;
  // sparse form: ELL rows of J (ell_d > 0), else the dense padded rows
  const int* ell_cols = nullptr;
  const void* ell_vals = nullptr;
  int ell_d = 0;
};

// The visits of one sweep (simulation.py:41-76): visit vi of a chain in the
// sequential order, a Feistel permutation (per chain, or shared by all chains
// of the sweep), the block-random order or a replayed order.
struct Visits {
  int nv;  // visit slots: n, or 32 per block in the block-random order
  bool brand;
  FeistelKey fk;
  __device__ Visits(const SweepCtx& c, uint64_t cid, bool replay) {
    brand = c.order == kBlockRandom && !replay;
    const int nb = (c.n + kOrderBlock - 1) / kOrderBlock;
    nv = brand ? kOrderBlock * nb : c.n;
    if (brand)
      fk = block_order_key((uint32_t)nb, c.sw, c.k0, c.k1);
    else if (c.order != kSequential && !replay)
      fk = feistel_make((uint32_t)c.n,
                        perm_keys(c.order == kRandomShared ? 0ull : cid, c.sw,
                                  c.order == kRandomShared ? kStreamShared : kStreamPerm, c.k0,
                                  c.k1));
  }
  // The position (-1: a padding slot of the last block) and its log-uniform.
  __device__ void at(int vi, const SweepCtx& c, uint64_t cid, const double* rep_lr,
                     const int* rep_perm, int& pos, double& lr) const {
    pos = -1;
    lr = 0.0;
    if (vi < nv) {
      if (rep_perm)
        pos = rep_perm[vi];
      else if (brand)
        pos = block_random_pos(fk, c.sw, (uint32_t)vi, c.n, c.k0, c.k1);
      else
        pos = (c.order == kSequential) ? vi : (int)feistel_perm(fk, (uint32_t)vi);
      if (pos >= 0) lr = log_uniform(rep_lr, cid, c.sw, pos, c.k0, c.k1);
    }
  }
};

// One sweep of one chain, one visit after another (sparse form).
template <typename T, int G>
__device__ double sweep_sparse(Chain<T, G>& ch, const T* hs, const SweepCtx& c, T beta,
                               uint64_t cid, const double* rep_lr, const int* rep_perm,
                               unsigned long long& acc) {
  const int lane = threadIdx.x & 63;
  const Visits vs(c, cid, rep_perm != nullptr);
  double sum = 0.0;
  for (int w = 0; w < vs.nv; w += 64) {
    int pos_l;
    double lr_l;
    vs.at(w + lane, c, cid, rep_lr, rep_perm, pos_l, lr_l);
    const T h_l = (pos_l >= 0) ? hs[pos_l] : T(0);
    const int cnt = min(64, vs.nv - w);
    for (int t = 0; t < cnt; ++t) {
      const int pos = rl(pos_l, t);
      if (pos < 0) continue;  // padding slot (wave-uniform)
      const double lr = rl(lr_l, t);
      const int pl = lane_of(pos), ps = slot_of(pos);
      const bool up = (rl(ch.bits, pl) >> ps) & 1;
      const T fh = rl(ch.pick(ps), pl) + rl(h_l, t);
      double dn;
      if (decide<T, false>(c.ptype, up, fh, lr, (double)beta, c.ref, c.lratio, dn)) {
        sum += -dn;
        ++acc;
        ch.flip(pos);
        const T dS = (c.ptype == 0) ? (up ? T(-2) : T(2)) : (up ? T(-1) : T(1));
        ch.add_ell(c.ell_cols + (size_t)pos * c.ell_d,
                   static_cast<const T*>(c.ell_vals) + (size_t)pos * c.ell_d, c.ell_d, dS);
      }
    }
  }
  return sum;
}

// The spin change of a flip, -+2 (ising) or -+1 (qubo), in scalar registers.
__device__ __forceinline__ float spin_change(int ptype, bool up, float) {
  return __uint_as_float((ptype == 0 ? 0x40000000u : 0x3F800000u) | ((uint32_t)up << 31));
}
__device__ __forceinline__ double spin_change(int ptype, bool up, double) {
  return as_double((uint64_t)((ptype == 0 ? 0x40000000u : 0x3FF00000u) | ((uint32_t)up << 31))
                   << 32);
}

// One sweep of one chain with dense rows (see the top of the file), buf the
// wave's LDS buffer.
// Bound: kWide by the L1 / L2 traffic of one row per accepted flip and the
// issue of its additions; kBlock by latency, a chain of an LDS read and an f64
// comparison per accepted flip, then the rows' loads.  Before, every visit
// picked its field from the registers by a select tree (~100 VALU slots a
// proposal) and waited for the row of the last flip: 512 reads of 32 replicas
// of 1024 spins x 40 sweeps, random order, 118.0 -> 55.9 ms (kWide); 8 reads
// of 16 replicas of 300 spins in f64 x 100 sweeps 17.8 -> 3.4 ms, one read of
// 100 replicas of 3072 spins x 2 sweeps 944 -> 2.4 ms (kBlock, a workgroup per
// chain; before, one workgroup for the read).
template <typename T, int G, bool AIS, int V>
__device__ double sweep_dense(Chain<T, G>& ch, const T* hs, const SweepCtx& c,
                              const T* __restrict__ Jp, int ldp, T beta, uint64_t cid,
                              const double* rep_lr, const int* rep_perm, unsigned long long& acc,
                              int& od, T* buf) {
  const int lane = threadIdx.x & 63;
  const double bd = (double)beta;
  const Visits vs(c, cid, rep_perm != nullptr);
  od = 0;
  double sum = 0.0;
  for (int w = 0, cnt; w < vs.nv; w += cnt) {
    int pos_l;
    double lr_l;
    vs.at(w + lane, c, cid, rep_lr, rep_perm, pos_l, lr_l);
    cnt = min(64, vs.nv - w);
    if (rep_perm) {  // a replayed order may repeat a position: the window ends before it
      bool again = false;
      for (int t = 0; t < cnt; ++t) again = again || (t < lane && pos_l == rl(pos_l, t));
      const uint64_t dup = __ballot(again && lane < cnt);
      if (dup) cnt = __builtin_ctzll(dup);
      if (lane >= cnt) pos_l = -1;
    }
    const int pc = max(pos_l, 0);
    const uint64_t valid = __ballot(pos_l >= 0);
    const T h_l = hs[pc];
    // the fields of the visits, through LDS (element i at buf[i]), and their spins
#pragma unroll
    for (int g4 = 0; g4 < G / 4; ++g4) {
      T4<T> v;
#pragma unroll
      for (int q = 0; q < 4; ++q) v.v[q] = ch.f[4 * g4 + q];
      reinterpret_cast<T4<T>*>(buf)[(g4 << 6) + lane] = v;
    }
    wave_sync();
    T fv = buf[pc];
    const bool up = (shfl_bits(ch.bits, lane_of(pc)) >> slot_of(pc)) & 1;
    const uint64_t upm = __ballot(up);
    wave_sync();
    if constexpr (V == kBlock) {  // row t: the couplings of visit t to every visit
      for (int t0 = 0; t0 < cnt; t0 += 16) {
        T v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u)
          v[u] = Jp[(uint32_t)max(rl(pos_l, t0 + u), 0) * (uint32_t)ldp + (uint32_t)pc];
#pragma unroll
        for (int u = 0; u < 16; ++u) buf[(t0 + u) * 64 + lane] = v[u];
      }
      wave_sync();
    }
    // dn = 2 s (F + h) (ising.py:48-49) or (2x - 1)(F + h) (qubo.py:48-49)
    const double sg = c.ptype == 0 ? (up ? 2.0 : -2.0) : (up ? 1.0 : -1.0);
    const double refd = (AIS && c.ref == 1) ? (up ? c.lratio : -c.lratio) : 0.0;
    const double cref = (1.0 - bd) * refd;
    double dn;
    auto decisions = [&]() __attribute__((always_inline)) {  // ising.py:52 / :75-83
      dn = sg * (double)(fv + h_l);
      const double x = bd * dn, y = AIS ? x + cref : dn, z = AIS ? y : x;
      return __builtin_amdgcn_ballot_w64(y >= 0) | __builtin_amdgcn_ballot_w64(lr_l < z);
    };
    uint64_t m = decisions() & valid, taken = 0;
    while (m) {  // the first accepted visit t of those not yet passed
      const int t = __builtin_ctzll(m);
      const T dS = spin_change(c.ptype, (upm >> t) & 1, T(0));
      const double dnt = rl(dn, t);
      taken |= 1ull << t;
      if constexpr (V == kBlock) {
        fv = fma_t(buf[t * 64 + lane], dS, fv);
      } else {
        const int pos = rl(pos_l, t);
        T4<T> x[G / 4];
        ch.load_row(x, Jp, pos, ldp);
        ch.flip(pos);
#pragma unroll
        for (int g4 = 0; g4 < G / 4; ++g4) reinterpret_cast<T4<T>*>(buf)[(g4 << 6) + lane] = x[g4];
        wave_sync();
        fv = fma_t(buf[pc], dS, fv);
        ch.add_row(x, dS);
        wave_sync();
      }
      m = decisions() & valid & (~1ull << t);
      sum += -dnt;
    }
    acc += (unsigned long long)__builtin_popcountll(taken);
    od += __builtin_popcountll(taken & ~upm) - __builtin_popcountll(taken & upm);
    if constexpr (V == kBlock) {
      // the accepted rows in order, NB in flight; loads past the last one
      // repeat it, so that every path issues the same loads
      constexpr int REG = G * (int)(sizeof(T) / 4);
      constexpr int NB = REG >= 32 ? 2 : REG >= 16 ? 4 : 8;
      if (taken) {
        T4<T> x[NB][G / 4];
        uint64_t ql = taken;  // rows to load
        int last = 0;
        auto load_next = [&](T4<T> (&d)[G / 4]) __attribute__((always_inline)) {
          last = ql ? rl(pos_l, __builtin_ctzll(ql)) : last;
          ql &= ql - 1;
          ch.load_row(d, Jp, last, ldp);
        };
#pragma unroll
        for (int b = 0; b < NB; ++b) load_next(x[b]);
        while (taken) {
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            if (taken) {
              const int t = __builtin_ctzll(taken);
              taken &= taken - 1;
              ch.flip(rl(pos_l, t));
              ch.add_row(x[b], spin_change(c.ptype, (upm >> t) & 1, T(0)));
            }
            load_next(x[b]);
          }
        }
      }
    }
  }
  return sum;
}

// PT log-uniform of one pair (utils.py:57): replayed or drawn.
template <typename T>
__device__ __forceinline__ double pt_log_uniform(const PTParams<T>& p, int read, int s, int k) {
  if (p.rep_pt) return p.rep_pt[((size_t)read * p.S + s) * (p.R - 1) + k];
  return log_u32(pick_word(pt_block((uint64_t)read, (uint64_t)s + p.sweep_offset, (uint32_t)k,
                                    p.k0, p.k1),
                           (uint32_t)k & 3u));
}

// log-omega of one sweep (ais.py:99-112) over the ascending ladder.
template <typename T, typename I>
__device__ double log_omega_of(int R, const int* bsort, const T* beta, const T* E, const I* bi) {
  double lw = 0.0, bold = 0.0;
  for (int r = 1; r < R; ++r) {
    const int q = bsort[r];
    const T be = beta[q];
    const T en = E[bi[q]];
    const T a = -be * en;
    lw += (double)a - (-bold * (double)en);
    bold = (double)be;
  }
  return lw;
}

template <typename T>
__device__ SweepCtx sweep_ctx(const PTParams<T>& p) {
  SweepCtx c;
  c.n = p.n;
  c.ptype = p.ptype;
  c.order = p.order;
  c.ref = 0;
  c.k0 = p.k0;
  c.k1 = p.k1;
  c.lratio = 0.0;
  c.ell_cols = p.ell_cols;
  c.ell_vals = p.ell_vals;
  c.ell_d = p.ell_d;
  return c;
}

// LDS of plain_pt_kernel (dynamic): the wave buffers, h, and the read's
// replicas.
template <typename T>
struct PTLds {
  T *buf, *h, *bs, *beta, *E, *bE;
  double *lu, *eoff;
  int *bi, *bsw;
  __host__ __device__ static size_t bytes(int buf_elems, int n, int R) {
    return (size_t)(buf_elems + ((n + 1) & ~1) + 4 * ((R + 1) & ~1)) * sizeof(T) +
           (size_t)R * (2 * sizeof(double) + 2 * sizeof(int));
  }
  __device__ PTLds(char* base, int buf_elems, int n, int R) {
    const int Re = (R + 1) & ~1;  // every array 8-byte aligned
    buf = reinterpret_cast<T*>(base);
    h = buf + buf_elems;
    bs = h + ((n + 1) & ~1);
    beta = bs + Re;
    E = beta + Re;
    bE = E + Re;
    lu = reinterpret_cast<double*>(bE + Re);
    eoff = lu + R;
    bi = reinterpret_cast<int*>(eoff + R);
    bsw = bi + R;
  }
};

// All sweeps of one read: W waves carry its R replicas (each wave its own for
// the whole run when R <= W, else one after another through global memory)
// and meet after every sweep for the exchanges.
template <typename T, int G, int V>
__global__ __launch_bounds__((64 * pt_waves<T, G, V>())) void plain_pt_kernel(PTParams<T> p) {
  const int read = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, W = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int R = p.R, n = p.n;
  extern __shared__ __align__(16) char lds[];
  const PTLds<T> L(lds, W * wave_buf<G, V>(), n, R);
  __shared__ int s_src;
  __shared__ T s_gE;
  __shared__ int s_gsw, s_improved;
  T* buf = L.buf + wave * wave_buf<G, V>();

  for (int i = tid; i < n; i += blockDim.x) L.h[i] = p.h[i];
  for (int k = tid; k < R; k += blockDim.x) {
    L.bi[k] = k;  // beta_idx = arange(R) (sa.py:325)
    L.E[k] = p.energies[(size_t)read * R + k];
    L.bE[k] = L.E[k];  // simulation.py:143-145
    L.bsw[k] = 0;
    L.beta[k] = p.betas[k];
  }
  if (tid == 0) {
    s_gE = p.energies[(size_t)read * R];  // simulation.py:205
    s_gsw = 0;
    s_improved = 0;
  }
  __syncthreads();
  SweepCtx c = sweep_ctx(p);
  unsigned long long acc = 0;
  const bool own = R <= W;  // the wave's replica stays in registers
  Chain<T, G> ch;
  if (own && wave < R) {
    const size_t off = ((size_t)read * R + wave) * n;
    ch.load_spins(p.spins + off, n);
  }
  for (int s = 0; s < p.S; ++s) {
    c.sw = (uint64_t)s + p.sweep_offset;
    // Local fields F = J s recomputed in f64 (rounded once) at the start and
    // every `refresh` sweeps, which bounds the drift of float couplings.  The
    // reference recomputes every field from its coupling row
    // (ising.py:48), so its energy changes carry no drift; here the tracked
    // energy is reset with the fields to the f64 energy plus the offset the
    // caller's initial energy had from it (zero unless the caller passed
    // other energies), so the drift of incrementally updated fields does not
    // accumulate.  Integer couplings are exact either way: the reset then
    // leaves the value unchanged.
    const bool fresh = s == 0 || (p.refresh > 0 && s % p.refresh == 0);
    for (int k = tid; k < R; k += blockDim.x) L.bs[L.bi[k]] = L.beta[k];  // simulation.py:151-152
    // PT log-uniforms, one per pair, drawn in parallel ahead of the serial walk.
    if (p.use_pt)
      for (int k = tid; k < R - 1; k += blockDim.x) L.lu[k] = pt_log_uniform(p, read, s, k);
    __syncthreads();
    for (int r = wave; r < R; r += W) {  // replicas of this read (simulation.py:154-164)
      const size_t off = ((size_t)read * R + r) * n;
      if (!own) {
        if (s == 0)
          ch.load_spins(p.spins + off, n);
        else
          ch.load(p.fields + off, p.spins + off, n);
      }
      if (fresh) {
        double ex;
        if constexpr (V == kSparse)
          ex = ch.refresh_ell(p.ell_cols, p.ell_vals, p.ell_d, L.h, n, p.ptype);
        else
          ex = ch.refresh(p.Jp, p.ldp, L.h, n, p.ptype);
        if (lane == 0) {
          if (s == 0)
            L.eoff[r] = (double)L.E[r] - ex;
          else
            L.E[r] = (T)(ex + L.eoff[r]);
        }
        wave_sync();
      }
      const size_t rb = (((size_t)read * p.S + s) * R + r) * (size_t)n;
      const uint64_t cid = (uint64_t)read * R + r;
      const double* rlr = p.rep_lr ? p.rep_lr + rb : nullptr;
      const int* rpm = p.rep_perm ? p.rep_perm + rb : nullptr;
      double d;
      int od;
      if constexpr (V == kSparse)
        d = sweep_sparse<T, G>(ch, L.h, c, L.bs[r], cid, rlr, rpm, acc);
      else
        d = sweep_dense<T, G, false, V>(ch, L.h, c, p.Jp, p.ldp, L.bs[r], cid, rlr, rpm, acc, od,
                                        buf);
      if (!own || s + 1 == p.S || p.best_sem == 1) ch.store(p.fields + off, p.spins + off, n, p.ptype);
      const T en = (T)((double)L.E[r] + d);  // simulation.py:157-158
      if (p.best_sem == 0 && en < L.bE[r]) {  // simulation.py:161-164
        ch.store_spins(p.best_rep + off, n, p.ptype);
        if (lane == 0) {
          L.bE[r] = en;
          L.bsw[r] = s;
        }
      }
      if (lane == 0) L.E[r] = en;
    }
    __syncthreads();
    if (wave == 0) {
      if (p.best_sem == 1 && lane == 0) {  // simulation.py:222-225 in replica order
        int src = -1;
        T cur = s_gE;
        for (int k = 0; k < R; ++k)
          if (L.E[k] < cur) {
            cur = L.E[k];
            src = k;
          }
        if (src >= 0) {
          s_gE = cur;
          s_gsw = s;
          s_improved = 1;
        }
        s_src = src;
      }
      if (p.use_pt) exchange_wave<T, int>(R, L.E, L.beta, L.lu, L.bi);
      if (p.logw && p.log_omegas) {
        wave_sync();
        if (lane == 0)
          p.log_omegas[(size_t)read * p.S + s] = log_omega_of<T, int>(R, p.bsort, L.beta, L.E, L.bi);
      }
    }
    __syncthreads();
    if (p.best_sem == 1 && s_src >= 0) {
      const int8_t* src = p.spins + ((size_t)read * R + s_src) * n;
      for (int i = tid; i < n; i += blockDim.x) p.best_state[(size_t)read * n + i] = src[i];
    }
  }

  // Outputs.
  for (int k = tid; k < R; k += blockDim.x) {
    p.beta_idx[(size_t)read * R + k] = L.bi[k];
    p.energies[(size_t)read * R + k] = L.E[k];
  }
  if (lane == 0 && p.accepted) atomicAdd(p.accepted + read, acc);
  __syncthreads();
  if (p.best_sem == 0) {  // simulation.py:174-177, first minimum wins
    if (tid == 0) {
      int bp = 0;
      for (int k = 1; k < R; ++k)
        if (L.bE[k] < L.bE[bp]) bp = k;
      s_src = bp;
      p.best_energy[read] = L.bE[bp];
      p.best_sweeps[read] = L.bsw[bp];
    }
    __syncthreads();
    const int8_t* src = p.best_rep + ((size_t)read * R + s_src) * n;
    for (int i = tid; i < n; i += blockDim.x) p.best_state[(size_t)read * n + i] = src[i];
  } else {
    if (tid == 0) {
      p.best_energy[read] = s_gE;
      p.best_sweeps[read] = s_gsw;
    }
    if (!s_improved) {  // best_state is still the view of states[0] (simulation.py:204)
      const int8_t* src = p.spins + (size_t)read * R * n;
      for (int i = tid; i < n; i += blockDim.x) p.best_state[(size_t)read * n + i] = src[i];
    }
  }
}

// ---- one workgroup (one wave) per chain ----

// F = J s and the energy of the chains from c0 on from their f64 sums
// (chain_sums_kernel), as Chain::refresh makes them; s: the sweep before which
// this happens.
template <typename T, int G>
__global__ __launch_bounds__(64) void chain_refresh_kernel(PTParams<T> p, int s, int c0) {
  const size_t chain = (size_t)c0 + blockIdx.x;
  const int lane = threadIdx.x, n = p.n;
  Chain<T, G> ch;
  ch.load_spins(p.spins + chain * n, n);
  const double* sums = p.sums + (size_t)blockIdx.x * n;
  double e = 0.0;
#pragma unroll
  for (int g4 = 0; g4 < G / 4; ++g4) {
    double a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = (g4 << 8) + (lane << 2) + q;
      a[q] = i < n ? sums[i] : 0.0;
    }
    e = ch.put_fields(g4, a, p.h, n, p.ptype, e);
  }
  e = wave_sum(e);
  ch.store(p.fields + chain * n, p.spins + chain * n, n, p.ptype);
  if (lane == 0) {
    if (s == 0)
      p.eoff[chain] = (double)p.energies[chain] - e;
    else
      p.energies[chain] = (T)(e + p.eoff[chain]);
  }
}

// Sweeps [s0, s1) of one chain (several only when nothing of a sweep's end
// concerns other chains).
template <typename T, int G>
__global__ __launch_bounds__(64) void chain_sweep_kernel(PTParams<T> p, int s0, int s1) {
  __shared__ T buf[64 * 64];
  const int chain = blockIdx.x, lane = threadIdx.x, n = p.n;
  const size_t off = (size_t)chain * n;
  Chain<T, G> ch;
  ch.load(p.fields + off, p.spins + off, n);
  SweepCtx c = sweep_ctx(p);
  const T beta = p.chain_beta[chain];
  T E = p.energies[chain], bE = p.best_rep_e[chain];
  const int read = chain / p.R, r = chain - read * p.R;
  unsigned long long acc = 0;
  for (int s = s0; s < s1; ++s) {
    c.sw = (uint64_t)s + p.sweep_offset;
    const size_t rb = (((size_t)read * p.S + s) * p.R + r) * (size_t)n;
    int od;
    const double d = sweep_dense<T, G, false, kBlock>(
        ch, p.h, c, p.Jp, p.ldp, beta, (uint64_t)chain, p.rep_lr ? p.rep_lr + rb : nullptr,
        p.rep_perm ? p.rep_perm + rb : nullptr, acc, od, buf);
    E = (T)((double)E + d);  // simulation.py:157-158
    if (p.best_sem == 0 && E < bE) {  // simulation.py:161-164
      bE = E;
      ch.store_spins(p.best_rep + off, n, p.ptype);
      if (lane == 0) {
        p.best_rep_e[chain] = E;
        p.best_rep_sw[chain] = s;
      }
    }
  }
  ch.store(p.fields + off, p.spins + off, n, p.ptype);
  if (lane == 0) {
    p.energies[chain] = E;
    if (p.accepted) atomicAdd(p.accepted + read, acc);
  }
}

// The end of sweep s of a read whose chains run in workgroups of their own
// (s < 0: before the first sweep, which only takes the betas): best state in
// replica order, exchanges, log-omega and the chains' new betas, as in
// plain_pt_kernel.
template <typename T>
__global__ __launch_bounds__(256) void chain_exchange_kernel(PTParams<T> p, int s) {
  __shared__ T s_E[kMaxR], s_beta[kMaxR];
  __shared__ int s_bi[kMaxR];
  __shared__ double s_lu[kMaxR];
  __shared__ int s_src;
  const int read = blockIdx.x, tid = threadIdx.x, R = p.R, n = p.n;
  const size_t c0 = (size_t)read * R;
  for (int k = tid; k < R; k += 256) {
    s_E[k] = p.energies[c0 + k];
    s_beta[k] = p.betas[k];
    s_bi[k] = s < 0 ? k : (int)p.beta_idx[c0 + k];
    if (s >= 0 && p.use_pt && k < R - 1) s_lu[k] = pt_log_uniform(p, read, s, k);
  }
  __syncthreads();
  if (tid < 64) {
    if (tid == 0 && p.best_sem == 1) {  // simulation.py:222-225 in replica order
      T cur = s < 0 ? s_E[0] : p.best_energy[read];
      int src = -1;
      if (s >= 0)
        for (int k = 0; k < R; ++k)
          if (s_E[k] < cur) {
            cur = s_E[k];
            src = k;
          }
      if (s < 0 || src >= 0) {
        p.best_energy[read] = cur;
        p.best_sweeps[read] = s < 0 ? 0 : s;
        if (src >= 0) p.best_rep_sw[c0] = 1;  // a state has been copied
      }
      s_src = src;
    }
    if (s >= 0) {
      if (p.use_pt) exchange_wave<T, int>(R, s_E, s_beta, s_lu, s_bi);
      wave_sync();
      if (p.logw && p.log_omegas && tid == 0)
        p.log_omegas[(size_t)read * p.S + s] = log_omega_of<T, int>(R, p.bsort, s_beta, s_E, s_bi);
    }
  }
  __syncthreads();
  if (p.best_sem == 1 && s_src >= 0) {
    const int8_t* src = p.spins + (c0 + s_src) * n;
    for (int i = tid; i < n; i += 256) p.best_state[(size_t)read * n + i] = src[i];
  }
  for (int k = tid; k < R; k += 256) {
    p.beta_idx[c0 + k] = s_bi[k];
    p.chain_beta[c0 + s_bi[k]] = s_beta[k];  // simulation.py:151-152
  }
}

// The best of a read after the last sweep.
template <typename T>
__global__ __launch_bounds__(256) void chain_best_kernel(PTParams<T> p) {
  const int read = blockIdx.x, n = p.n, R = p.R;
  const size_t c0 = (size_t)read * R;
  int bp = 0;
  const int8_t* from = p.spins;  // never improved: the view of states[0] (simulation.py:204)
  if (p.best_sem == 0) {  // simulation.py:174-177, first minimum wins
    for (int k = 1; k < R; ++k)
      if (p.best_rep_e[c0 + k] < p.best_rep_e[c0 + bp]) bp = k;
    if (threadIdx.x == 0) {
      p.best_energy[read] = p.best_rep_e[c0 + bp];
      p.best_sweeps[read] = p.best_rep_sw[c0 + bp];
    }
    from = p.best_rep;
  } else if (p.best_rep_sw[c0]) {
    return;
  }
  for (int i = threadIdx.x; i < n; i += 256)
    p.best_state[(size_t)read * n + i] = from[(c0 + bp) * n + i];
}

// AIS: each wave carries one chain through the whole beta schedule
// (simulation.py:266-317); chains are independent, so there are no barriers
// after h is staged.
template <typename T, int G, int V>
__global__ __launch_bounds__(64 * (V == kBlock ? 1 : kernel_waves<T, G>())) void plain_ais_kernel(
    AISParams<T> p) {
  __shared__ T s_h[64 * G];
  __shared__ T s_buf[(V == kBlock ? 1 : kernel_waves<T, G>()) * wave_buf<G, V>()];
  const int tid = threadIdx.x, lane = tid & 63, W = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = p.n;
  for (int i = tid; i < n; i += blockDim.x) s_h[i] = p.h[i];
  __syncthreads();
  const int chain = blockIdx.x * W + wave;
  if (chain >= p.chains) return;
  T* buf = s_buf + wave * wave_buf<G, V>();
  Chain<T, G> ch;
  ch.load_spins(p.spins + (size_t)chain * n, n);
  double E = ch.refresh(p.Jp, p.ldp, s_h, n, p.ptype);
  int ones = ch.count_up(n);
  SweepCtx c;
  c.n = n;
  c.ptype = p.ptype;
  c.order = p.order;
  c.ref = p.ref;
  c.k0 = p.k0;
  c.k1 = p.k1;
  c.lratio = p.lp - p.l1p;
  double bold = 0.0, lw = 0.0;
  unsigned long long acc = 0;
  for (int t = 0; t < p.nt; ++t) {
    c.sw = (uint64_t)t;
    const T beta = p.temps[t];
    const double bd = (double)beta;
    // The reference recomputes the energy after every step
    // (simulation.py:309); here fields and energy are recomputed in f64
    // every `refresh` steps and updated by the accepted changes in between,
    // which bounds the drift of float couplings.
    if (t > 0 && p.refresh > 0 && t % p.refresh == 0)
      E = ch.refresh(p.Jp, p.ldp, s_h, n, p.ptype);
    if (p.ordering == 1) {  // Neal's ordering: weight before the transition
      const double refE = (p.ref == 1) ? -((double)(n - ones) * p.lp + (double)ones * p.l1p) : 0.0;
      lw += (-bd * E - (1.0 - bd) * refE) - (-bold * E - (1.0 - bold) * refE);
    }
    const size_t rb = ((size_t)chain * p.nt + t) * (size_t)n;
    int od;
    const double d = sweep_dense<T, G, true, V>(ch, p.h, c, p.Jp, p.ldp, beta, (uint64_t)chain,
                                                p.rep_lr ? p.rep_lr + rb : nullptr,
                                                p.rep_perm ? p.rep_perm + rb : nullptr, acc, od,
                                                buf);
    E += d;
    ones += od;
    if (p.ordering == 0) {  // simulation.py:309-314, after the transition
      const double refE = (p.ref == 1) ? -((double)(n - ones) * p.lp + (double)ones * p.l1p) : 0.0;
      lw += (-bd * E - (1.0 - bd) * refE) - (-bold * E - (1.0 - bold) * refE);
    }
    bold = bd;
  }
  ch.store(p.fields + (size_t)chain * n, p.spins + (size_t)chain * n, n, p.ptype);
  if (lane == 0) {
    p.energy[chain] = E;
    p.logw[chain] = lw;
  }
}

// J s in f64 for SB states per workgroup: thread t owns the elements
// i = i0 + t, i0 + 256 + t, ... (I of them), and every coupling it loads (from
// rows of J^T, coalesced across threads) serves all SB states.  A state's
// spins of 64 columns j are one bit per lane, read back one column at a time,
// so the factor of a product (1 for a set bit, else the double with the high
// word `low`: -1 or 0) is a scalar operand.  GEN: spins of any int8 value, read
// one by one.  Every sum runs over j in ascending order in f64, whatever SB
// and I are, and each product J s is exact, so the results do not depend on
// the tiling.
template <typename T, int SB, int I, bool GEN>
__device__ __forceinline__ void field_sums(const T* __restrict__ Jt,
                                           const int8_t* __restrict__ spins, int n, int count,
                                           int s0, int i0, uint32_t low, double (&f)[SB][I]) {
  const int lane = threadIdx.x & 63;
  // byte offsets within a row (the row's base is uniform), clamped: a thread
  // past n repeats the last element (unused)
  uint32_t ic[I];
#pragma unroll
  for (int k = 0; k < I; ++k)
    ic[k] = (uint32_t)min(i0 + 256 * k + (int)threadIdx.x, n - 1) * (uint32_t)sizeof(T);
#pragma unroll
  for (int b = 0; b < SB; ++b)
#pragma unroll
    for (int k = 0; k < I; ++k) f[b][k] = 0.0;
  constexpr int U = GEN ? 1 : SB * I >= 32 ? 2 : 16;  // columns whose loads are in flight together
  for (int j0 = 0; j0 < n; j0 += 64) {
    uint32_t up = 0;
    if constexpr (!GEN) {
      const int jl = min(j0 + lane, n - 1);
#pragma unroll
      for (int b = 0; b < SB; ++b)
        up |= (uint32_t)(spins[(size_t)min(s0 + b, count - 1) * n + jl] == 1) << b;
    }
    for (int jj = 0; jj < 64 && j0 + jj < n; jj += U) {
      T x[U][I];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // past the last column: its values again, as zeros
        const bool in = j0 + jj + u < n;
        const char* row =
            reinterpret_cast<const char*>(Jt + (size_t)(in ? j0 + jj + u : n - 1) * n);
#pragma unroll
        for (int k = 0; k < I; ++k) {
          const T v = *reinterpret_cast<const T*>(row + ic[k]);
          x[u][k] = U == 1 || in ? v : T(0);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t w = GEN ? 0u : rl(up, jj + u);
#pragma unroll
        for (int b = 0; b < SB; ++b) {
          const double sv =
              GEN ? (double)spins[(size_t)min(s0 + b, count - 1) * n + j0 + jj]
                  : as_double((uint64_t)(((w >> b) & 1u) ? 0x3FF00000u : low) << 32);
#pragma unroll
          for (int k = 0; k < I; ++k) f[b][k] = dfma((double)x[u][k], sv, f[b][k]);
        }
      }
    }
  }
}

// E = s.(J s / 2 + h) in f64 (ising.py:32-37), SB states per workgroup.  Thread
// t adds its elements t, t + 256, ... in this order, then the wave and the
// workgroup add theirs.  With one workgroup per group of states (gridDim.y =
// 1) the energies go to out; otherwise workgroup y writes the terms of its
// 256 I elements and energy_sum_kernel adds them in the same order.
template <typename T, int SB, int I, bool GEN>
__device__ __forceinline__ void energy_body(const T* __restrict__ Jt, const T* __restrict__ h,
                                            const int8_t* __restrict__ spins, double* out,
                                            double* terms, int n, int count, uint32_t low,
                                            double (&red)[SB][4]) {
  const int s0 = blockIdx.x * SB;
  double e[SB];
#pragma unroll
  for (int b = 0; b < SB; ++b) e[b] = 0.0;
  for (int c = blockIdx.y; c * 256 * I < n; c += gridDim.y) {
    double f[SB][I];
    field_sums<T, SB, I, GEN>(Jt, spins, n, count, s0, c * 256 * I, low, f);
#pragma unroll
    for (int k = 0; k < I; ++k) {
      const int i = (c * I + k) * 256 + threadIdx.x;
      const int il = min(i, n - 1);
      const double hi = (double)h[il];
#pragma unroll
      for (int b = 0; b < SB; ++b) {
        const double t =
            (double)spins[(size_t)min(s0 + b, count - 1) * n + il] * (0.5 * f[b][k] + hi);
        if (terms) {
          if (i < n && s0 + b < count) terms[(size_t)(s0 + b) * n + i] = t;
        } else {
          e[b] = i < n ? e[b] + t : e[b];
        }
      }
    }
  }
  if (terms) return;
#pragma unroll
  for (int b = 0; b < SB; ++b) {
    const double t = wave_sum(e[b]);
    if ((threadIdx.x & 63) == 0) red[b][threadIdx.x >> 6] = t;
  }
  __syncthreads();
  if (threadIdx.x < SB && s0 + (int)threadIdx.x < count) {
    double t = 0.0;
    for (int w = 0; w < 4; ++w) t += red[threadIdx.x][w];
    out[s0 + threadIdx.x] = t;
  }
}

// Bound: f64 fma issue (SB I per coupling loaded and converted).  16384 states
// of 1024 spins: 8.49 ms with one state per workgroup, where every product
// loaded its own coupling from L2, 1.17 ms with SB = 16, I = 4 (0.44 ms
// is 2^34 f64 fma at the vector peak).
template <typename T, int SB, int I>
__global__ __launch_bounds__(256, SB* I >= 32 ? 2 : 4) void energy_f64_kernel(
    const T* __restrict__ Jt, const T* __restrict__ h, const int8_t* __restrict__ spins,
    double* out, double* terms, int n, int count) {
  __shared__ double red[SB][4];
  // the values these states hold: +-1, 0 / 1, or others (the entry point takes any int8)
  const int s0 = blockIdx.x * SB;
  bool pm = true, zo = true;
  const size_t lo = (size_t)s0 * n, hi = (size_t)min(s0 + SB, count) * n;
  for (size_t i = lo + threadIdx.x; i < hi; i += 256) {
    const int v = spins[i];
    pm = pm && (v == 1 || v == -1);
    zo = zo && (v == 1 || v == 0);
  }
  pm = __syncthreads_and(pm);
  zo = __syncthreads_and(zo);
  if (pm || zo)
    energy_body<T, SB, I, false>(Jt, h, spins, out, terms, n, count, pm ? 0xBFF00000u : 0u, red);
  else
    energy_body<T, SB, I, true>(Jt, h, spins, out, terms, n, count, 0u, red);
}

__global__ __launch_bounds__(256) void energy_sum_kernel(const double* __restrict__ terms,
                                                         double* out, int n) {
  __shared__ double red[4];
  double e = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) e += terms[(size_t)blockIdx.x * n + i];
  e = wave_sum(e);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < 4; ++w) t += red[w];
    out[blockIdx.x] = t;
  }
}

// Field registers per lane for n spins: a power of two from 4 to 64 with
// 64 * G >= n.
int regs_for(int n) {
  int g = 4;
  while (64 * g < n) g *= 2;
  return g;
}

// J s in f64 of every chain (the input of chain_refresh_kernel).  The tiling
// multiplies by an unset QUBO spin, which makes NaN of an infinite coupling where
// Chain::refresh adds nothing; no other sum is NaN without one of its terms being
// so, and those that are, are taken again over the set spins.  (Leaving unset
// spins out of every sum cost the RBM step 0.13 of 3.73 ms.)
template <typename T>
__global__ __launch_bounds__(256) void chain_sums_kernel(const T* __restrict__ Jt,
                                                         const int8_t* __restrict__ spins, int n,
                                                         int count, int ptype, double* sums) {
  double f[4][1];
  const int s0 = blockIdx.x * 4, i = blockIdx.y * 256 + threadIdx.x;
  field_sums<T, 4, 1, false>(Jt, spins, n, count, s0, blockIdx.y * 256,
                             ptype == 0 ? 0xBFF00000u : 0u, f);
  if (i >= n) return;
#pragma unroll
  for (int b = 0; b < 4; ++b)
    if (s0 + b < count) {
      double x = f[b][0];
      if (ptype == 1 && x != x) {
        const int8_t* s = spins + (size_t)(s0 + b) * n;
        x = 0.0;
        for (int j = 0; j < n; ++j)
          if (s[j] == 1) x += (double)Jt[(size_t)j * n + i];
      }
      sums[(size_t)(s0 + b) * n + i] = x;
    }
}

template <typename T, int G, int V>
hipError_t launch_pt_read(const PTParams<T>& p, hipStream_t st) {
  const int W = min(p.R, pt_waves<T, G, V>());
  const size_t lds = PTLds<T>::bytes(W * wave_buf<G, V>(), p.n, p.R);
  hipLaunchKernelGGL((plain_pt_kernel<T, G, V>), dim3(p.reads), dim3(64 * W), lds, st, p);
  return hipGetLastError();
}

template <typename T, int G>
hipError_t launch_pt_chains(const PTParams<T>& p, hipStream_t st) {
  const int chains = p.reads * p.R;
  const bool coupled = p.coupled();
  hipLaunchKernelGGL((chain_exchange_kernel<T>), dim3(p.reads), dim3(256), 0, st, p, -1);
  for (int s = 0; s < p.S;) {
    if (s == 0 || (p.refresh > 0 && s % p.refresh == 0))
      for (int c0 = 0; c0 < chains; c0 += p.sums_chains) {
        const int cnt = min(p.sums_chains, chains - c0);
        hipLaunchKernelGGL((chain_sums_kernel<T>), dim3((cnt + 3) / 4, (p.n + 255) / 256),
                           dim3(256), 0, st, p.Jt, p.spins + (size_t)c0 * p.n, p.n, cnt, p.ptype,
                           p.sums);
        hipLaunchKernelGGL((chain_refresh_kernel<T, G>), dim3(cnt), dim3(64), 0, st, p, s, c0);
      }
    int e = coupled ? s + 1 : p.S;
    if (p.refresh > 0) e = min(e, s + p.refresh - s % p.refresh);
    hipLaunchKernelGGL((chain_sweep_kernel<T, G>), dim3(chains), dim3(64), 0, st, p, s, e);
    if (coupled) hipLaunchKernelGGL((chain_exchange_kernel<T>), dim3(p.reads), dim3(256), 0, st, p, s);
    s = e;
    const hipError_t le = hipGetLastError();
    if (le != hipSuccess) return le;
  }
  hipLaunchKernelGGL((chain_best_kernel<T>), dim3(p.reads), dim3(256), 0, st, p);
  return hipGetLastError();
}

template <typename T, int G>
hipError_t launch_pt_shape(const PTParams<T>& p, hipStream_t st) {
  if (p.ell_d > 0) return launch_pt_read<T, G, kSparse>(p, st);
  if (p.plan == kPlanChains) return launch_pt_chains<T, G>(p, st);
  return launch_pt_read<T, G, kWide>(p, st);
}

// AIS chains are independent: a workgroup each with staged windows while two
// fit a compute unit, else kWide waves spread evenly over the device.
template <typename T, int G>
hipError_t launch_ais_shape(const AISParams<T>& p, hipStream_t st) {
  const int cus = device_cus();
  if (p.chains <= 2 * cus) {
    hipLaunchKernelGGL((plain_ais_kernel<T, G, kBlock>), dim3(p.chains), dim3(64), 0, st, p);
  } else {
    const int W = min(kernel_waves<T, G>(), (p.chains + cus - 1) / cus);
    hipLaunchKernelGGL((plain_ais_kernel<T, G, kWide>), dim3((p.chains + W - 1) / W), dim3(64 * W),
                       0, st, p);
  }
  return hipGetLastError();
}

}  // namespace

// A workgroup per chain or per read.  A chain alone on its compute unit, with
// staged windows, takes a time that hardly depends on the replicas, plus about 8
// us for the two launches of a sweep when its end couples the chains (coupled).
// A read's time grows with its rounds of replicas and, within a round, with how
// far its waves crowd the rows of one compute unit.  So (us a sweep, per read /
// per chain):
// * More rounds of a read over its waves than of the chains over the device (8
//   chains a compute unit, 4 in f64, before they slow each other down): per
//   chain.  n = 200, 1 read of 32: 55 / 41; n = 1024, 64 reads of 32: 585 / 442;
//   n = 3072, 1 of 17: 26469 / 1260; n = 300, 1 of 17: 72 / 62.  Not where the
//   launches are a good part of a short sweep and the second round is at most
//   half full: n = 16, 1 of 17: 8.7 / 11.7; n = 64, 1 of 20: 15.0 / 18.2; n =
//   256, 1 of 17: 37 / 46; but n = 128, 1 of 24: 31 / 29.
// * Above 2048 spins a wave's fields leave few registers for rows in flight:
//   per chain while two fit a compute unit (n = 2500, 512 reads of 1: 2261 / 1248;
//   n = 4096, 1 of 1: 3383 / 1096).
// * Somewhat below, several replicas: per chain while each has a compute unit of
//   its own (n = 2048, 1 of 4: 775 / 627; n = 1284, 1 of 4: 357 / 401).
// * Else per chain where the read's waves crowd its compute unit, n R words 8000
//   or more (f64, n = 300, 8 of 16: 67 / 62; f64, n = 1024, 1 of 8: 383 / 339), of
//   sixteen waves with exchanges 9000 (n = 1024, 1 of 16: 198 / 192, of 8: 170 /
//   191; n = 512, 1 of 16: 77 / 92), and the chains are not two to a compute unit
//   with rows that are not short (f64, n = 1600, 128 of 4: 658 / 1055; f64, n =
//   300, 32 of 16: 70 / 68).
// The first fields take longer in a read's own waves, one row group after
// another, than spread over the device (n = 824, 1 of 10: 0.9 ms more), so the
// lines where a sweep is only a little faster per read ask for enough of them.
int plan_plain(int n, int reads, int R, int S, int elem, bool coupled) {
  const int64_t chains = (int64_t)reads * R;
  const int W = waves_of(regs_for(n) * (elem / 4));
  const int rounds = (R + W - 1) / W;
  const int cus = device_cus();
  const int64_t per = (int64_t)cus * (elem == 8 ? 4 : 8);
  const int64_t crounds = (chains + per - 1) / per;
  if (crounds < rounds) {
    const bool brief = n <= 256 && 2 * R <= 3 * W && (R - W) * n <= 320;
    return coupled && S >= 16 && brief ? kPlanReads : kPlanChains;
  }
  if (n > 2048) return chains <= 2 * cus ? kPlanChains : kPlanReads;
  if (n > 1800 && R > 1 && chains <= cus) return kPlanChains;
  const bool many = S >= 64;
  const bool crowded = (int64_t)n * R * (elem / 4) >= (coupled && many && W == 16 ? 9000 : 8000);
  return crowded && chains <= (many && n > 512 ? cus : 2 * cus) ? kPlanChains : kPlanReads;
}

template <typename T>
hipError_t launch_plain_pt(const PTParams<T>& p, hipStream_t st) {
  if (p.n < 1 || p.n > kPlainMaxN || p.R < 1 || p.R > kMaxR || p.reads < 1)
    return hipErrorInvalidValue;
  switch (regs_for(p.n)) {
    case 4: return launch_pt_shape<T, 4>(p, st);
    case 8: return launch_pt_shape<T, 8>(p, st);
    case 16: return launch_pt_shape<T, 16>(p, st);
    case 32: return launch_pt_shape<T, 32>(p, st);
    case 64:
      if constexpr (sizeof(T) == 4) return launch_pt_shape<T, 64>(p, st);
    default: return hipErrorInvalidValue;
  }
}

template <typename T>
hipError_t launch_plain_ais(const AISParams<T>& p, hipStream_t st) {
  if (p.n < 1 || p.n > kPlainMaxN || p.chains < 1) return hipErrorInvalidValue;
  switch (regs_for(p.n)) {
    case 4: return launch_ais_shape<T, 4>(p, st);
    case 8: return launch_ais_shape<T, 8>(p, st);
    case 16: return launch_ais_shape<T, 16>(p, st);
    case 32: return launch_ais_shape<T, 32>(p, st);
    case 64:
      if constexpr (sizeof(T) == 4) return launch_ais_shape<T, 64>(p, st);
    default: return hipErrorInvalidValue;
  }
}

// States whose f64 values per spin are in memory at a time: 16 MB of them, still
// 2000 workgroups of 4 states and 256 spins, so a launch fills the device.  (All
// at once, a problem kept 96 MB behind 4000 energies of 3000 spins.)
static int f64_piece(int n, long long count) {
  const long long fit = max(1ll, (16ll << 20) / (8ll * n) / 4) * 4;
  return (int)min(fit, count);
}

int chain_sums_chains(int n, long long chains) { return f64_piece(n, chains); }

// Tiling of the energy kernel: 16 states per workgroup once that fills the
// device, else 4 states and 256 elements each, the sums in a second launch
// (100 states of 3072 spins: 10.36 -> 0.37 ms).
constexpr int kEnergyWide = 16 * 256;

size_t energy_scratch_bytes(int n, long long count) {
  return count >= kEnergyWide || n <= 256 ? 0 : (size_t)f64_piece(n, count) * n * sizeof(double);
}

template <typename T>
hipError_t launch_energy_f64(const T* Jt, const T* h, const int8_t* spins, double* out, int n,
                             long long count, double* scratch, hipStream_t st) {
  if (count <= 0) return hipSuccess;
  if (count > 0x7fffffffLL) return hipErrorInvalidValue;
  if (count >= kEnergyWide) {
    hipLaunchKernelGGL((energy_f64_kernel<T, 16, 4>), dim3((unsigned)((count + 15) / 16)),
                       dim3(256), 0, st, Jt, h, spins, out, (double*)nullptr, n, (int)count);
    return hipGetLastError();
  }
  const unsigned chunks = (unsigned)((n + 255) / 256);
  if (chunks > 1 && !scratch) return hipErrorInvalidValue;
  const int piece = chunks > 1 ? f64_piece(n, count) : (int)count;
  for (long long s0 = 0; s0 < count; s0 += piece) {
    const int cnt = (int)min((long long)piece, count - s0);
    hipLaunchKernelGGL((energy_f64_kernel<T, 4, 1>), dim3((unsigned)((cnt + 3) / 4), chunks),
                       dim3(256), 0, st, Jt, h, spins + (size_t)s0 * n, out + s0,
                       chunks > 1 ? scratch : nullptr, n, cnt);
    if (chunks > 1)
      hipLaunchKernelGGL(energy_sum_kernel, dim3((unsigned)cnt), dim3(256), 0, st, scratch, out + s0,
                         n);
  }
  return hipGetLastError();
}

template hipError_t launch_plain_pt<float>(const PTParams<float>&, hipStream_t);
template hipError_t launch_plain_pt<double>(const PTParams<double>&, hipStream_t);
template hipError_t launch_plain_ais<float>(const AISParams<float>&, hipStream_t);
template hipError_t launch_plain_ais<double>(const AISParams<double>&, hipStream_t);
template hipError_t launch_energy_f64<float>(const float*, const float*, const int8_t*, double*, int,
                                             long long, double*, hipStream_t);
template hipError_t launch_energy_f64<double>(const double*, const double*, const int8_t*, double*,
                                              int, long long, double*, hipStream_t);

}  // namespace pysa

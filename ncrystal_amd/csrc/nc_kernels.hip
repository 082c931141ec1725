// Per-neutron kernels: cross sections and scatter sampling of a process
// composition (PowderBragg, incoherent elastic, S(alpha,beta)) with one lane
// per neutron and a Philox stream per neutron.
//
// Composition semantics: ncrystal_core/src/interfaces/NCProcImpl.cc:166-204
// (cumulative component xs), :353-362 (xs), :379-389 (component pick +
// sampling); batched layout: ncrystal_core/src/cinterface/ncrystal.cc:1107-1246.
#include "nc_kernels.hh"
#include "nc_sabstream.hh"
#include <algorithm>
#include <type_traits>

namespace ncamd {

// Neutrons and results of a batch that the last-level cache (256 MB) cannot hold
// pass by the caches, which are left to the tables: 3e7 neutrons, PowderBragg, 5000
// and 262k planes, cross sections 189 -> 177 and 250 -> 234 us, sampling 347 -> 326
// and 459 -> 430.  Smaller ones are often still there from the step that made
// them: 1e7 neutrons, past the caches against through them, cross sections 56 and
// 35 us (5000 planes), 76 and 58 (262k), sampling 104 and 64, 140 and 112.
// (A variant of the kernels: of a branch at run time the compiler makes one access.)
static inline bool past_caches(int64_t bytes) { return bytes > ((int64_t)256 << 20); }
template <bool Past>
NCD double load_stream(const double* __restrict__ p) {
  if constexpr (Past) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool Past>
NCD void store_stream(double x, double* __restrict__ p) {
  if constexpr (Past) __builtin_nontemporal_store(x, p);
  else *p = x;
}

// Variant kCompPBOnly: a single PowderBragg component (the same sum as
// comp_xs: 0 + scale * xs); kCompFG: FreeGas / absorption components
template <bool FP32PB, int Variant, bool Past>
__global__ void __launch_bounds__(256) k_xs_iso(CompView c, const double* __restrict__ ekin,
                                                int64_t n, int64_t repeat, double* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const double E = load_stream<Past>(ekin + i);
    double xs;
    if constexpr (Variant == kCompPBOnly) {
      xs = comp_outside(c, E) ? 0.0 : 0.0 + c.scale[0] * (pb_active(c.pb, E) ? pb_xs_sel<FP32PB>(c.pb, E) : 0.0);
    } else {
      xs = comp_xs<FP32PB, Variant == kCompFG>(c, E, nullptr);  // kCompFG: any composition with gas components
    }
    for (int64_t r = 0; r < repeat; ++r) store_stream<Past>(xs, out + r * n + i);
  }
}

template <int Variant, bool Past>
__global__ void __launch_bounds__(256) k_sample_iso(CompView c, const double* __restrict__ ekin,
                                                    int64_t n, int64_t total, uint64_t seed,
                                                    uint32_t stream, double* __restrict__ oE,
                                                    double* __restrict__ oMu,
                                                    unsigned long long* __restrict__ nerr) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += gstride) {
    const int64_t i = (total == n) ? k : (k % n);
    Rng rng;
    rng.init(seed, stream, (uint64_t)k);
    double Ef, mu;
    const int rc = comp_sample_iso<Variant>(c, rng, load_stream<Past>(ekin + i), Ef, mu);
    if (rc) { Ef = -1.0; mu = -999.0; atomicAdd(nerr, 1ull); }
    store_stream<Past>(Ef, oE + k);
    store_stream<Past>(mu, oMu + k);
  }
}

template <int Variant>
__global__ void __launch_bounds__(256) k_sample_dirs(CompView c, const double* __restrict__ ekin,
                                                     const double* __restrict__ dirs, int64_t n,
                                                     uint64_t seed, uint32_t stream,
                                                     double* __restrict__ oE, double* __restrict__ oD,
                                                     unsigned long long* __restrict__ nerr) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gstride) {
    Rng rng;
    rng.init(seed, stream, (uint64_t)k);
    double Ef, mu;
    const int rc = comp_sample_iso<Variant>(c, rng, ekin[k], Ef, mu);
    double ox = 0.0, oy = 0.0, oz = 0.0;
    if (rc) {
      Ef = -1.0;
      atomicAdd(nerr, 1ull);
    } else {
      rand_dir_given_mu(rng, mu, dirs[3 * k], dirs[3 * k + 1], dirs[3 * k + 2], ox, oy, oz);
    }
    oE[k] = Ef;
    oD[3 * k] = ox; oD[3 * k + 1] = oy; oD[3 * k + 2] = oz;
  }
}

// FreeGas (kKindFG) and 1/v absorption (kKindAbs) processes: cross section
// over the repeat layout, and FreeGas sampling (isotropic, or with a new
// direction from mu), one Philox stream per output slot.
__global__ void __launch_bounds__(256) k_simple_xs(int kind, FGView g, double abs_c, const double* __restrict__ ekin,
                                                   int64_t n, int64_t total, double* __restrict__ out) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += gstride) {
    const double E = ekin[(total == n) ? k : (k % n)];
    out[k] = kind == kKindFG ? fg_xs(g, E) : absoov_xs(abs_c, E);
  }
}
template <bool Dirs>
__global__ void __launch_bounds__(256) k_fg_sample(FGView g, const double* __restrict__ ekin,
                                                   const double* __restrict__ dirs, int64_t n, int64_t total,
                                                   uint64_t seed, uint32_t stream, double* __restrict__ oE,
                                                   double* __restrict__ oX, unsigned long long* __restrict__ nerr) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += gstride) {
    const int64_t i = (total == n) ? k : (k % n);
    Rng rng;
    rng.init(seed, stream, (uint64_t)k);
    double Ef, mu;
    const int rc = fg_sample_demu(g, rng, ekin[i], Ef, mu);
    if (rc) atomicAdd(nerr, 1ull);
    if constexpr (Dirs) {
      double ox = 0.0, oy = 0.0, oz = 0.0;
      if (rc) Ef = -1.0;
      else rand_dir_given_mu(rng, mu, dirs[3 * k], dirs[3 * k + 1], dirs[3 * k + 2], ox, oy, oz);
      oE[k] = Ef;
      oX[3 * k] = ox; oX[3 * k + 1] = oy; oX[3 * k + 2] = oz;
    } else {
      if (rc) { Ef = -1.0; mu = -999.0; }
      oE[k] = Ef;
      oX[k] = mu;
    }
  }
}

// Compositions with an S(alpha,beta) part, in stages so that no kernel
// carries every sampler: k_comp_pick samples PowderBragg / ElInc picks in
// place and queues the neutrons that pick S(alpha,beta), those below the
// table's Emax and those above it apart; k_comp_sab samples both.  The S(alpha,beta) stages restart
// the neutron's Philox stream and replay the pick's draw (`skip`), so every
// neutron gets what one kernel doing all of it would give.
// outputs of one neutron: (E', mu), or (E', direction) for the oriented call
// (random azimuth about the incoming direction, NCProcImpl.cc:29-37)
template <bool Dirs>
NCD void comp_store(int64_t k, int rc, double Ef, double mu, Rng& rng, const double* __restrict__ dirs,
                    double* __restrict__ oE, double* __restrict__ o2, unsigned long long* __restrict__ nerr) {
  if constexpr (Dirs) {
    double ox = 0.0, oy = 0.0, oz = 0.0;
    if (rc) { Ef = -1.0; atomicAdd(nerr, 1ull); }
    else rand_dir_given_mu(rng, mu, dirs[3 * k], dirs[3 * k + 1], dirs[3 * k + 2], ox, oy, oz);
    oE[k] = Ef;
    o2[3 * k] = ox; o2[3 * k + 1] = oy; o2[3 * k + 2] = oz;
  } else {
    if (rc) { Ef = -1.0; mu = -999.0; atomicAdd(nerr, 1ull); }
    oE[k] = Ef;
    o2[k] = mu;
  }
}

// Appends to one counter run one after the other, about 13 ns each whatever
// workgroup they come from, and paced this kernel (1e6 neutrons, two queues:
// 107 us with an append per queue and 256 neutrons): large workgroups, both ends
// of a queue by one atomic.
constexpr int kPickThreads = 1024;
template <bool Dirs, bool Gas>
__global__ void __launch_bounds__(kPickThreads) k_comp_pick(CompView c, const double* __restrict__ ekin,
                                                   const double* __restrict__ dirs, int64_t n, int64_t total,
                                                   uint64_t seed, uint32_t stream, double* __restrict__ oE,
                                                   double* __restrict__ o2, unsigned long long* __restrict__ nerr,
                                                   int64_t* __restrict__ sq, unsigned long long* __restrict__ sqc,
                                                   const double* __restrict__ ext, int64_t* __restrict__ cq,
                                                   unsigned long long* __restrict__ cqc) {
  constexpr int NW = kPickThreads / 64;
  __shared__ unsigned long long s_app[NW + 2];
  const bool packed = total < ((int64_t)1 << 32);
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  // workgroup-uniform loop: the queue appends synchronise the workgroup
  for (int64_t k0 = (int64_t)blockIdx.x * blockDim.x; k0 < total; k0 += gstride) {
    const int64_t k = k0 + threadIdx.x;
    const bool valid = k < total;
    Rng rng;
    double E = 0.0, Ef = 0.0, mu = 0.0;
    int slot = 0, rc = kCompToStage + kCompToSCB + 1;  // neither queue
    if (valid) {
      const int64_t i = (total == n) ? k : (k % n);
      E = ekin[i];
      rng.init(seed, stream, (uint64_t)k);
      rc = comp_pick_sample<Gas>(c, rng, E, Ef, mu, slot, ext ? ext[k] : 0.0);
    }
    // queue appends, one atomic per workgroup and queue: one queue per
    // staged component, and the SCBragg queue
    const bool staged = valid && rc == kCompToStage;
    // (a component's neutrons above its table's Emax from the back of its queue)
    for (int s = 0; s < c.nstaged; ++s) {
      const bool want = staged && slot == s;
      const bool high = want && c.kind[c.stage_comp[s]] == kKindSAB && !(E < c.sab[s].egrid[c.sab[s].ne - 1]);
      const int64_t pos = (int64_t)block_append2<NW>(&sqc[s], kMaxStaged, packed, want && !high, high, s_app);
      if (want) sq[(int64_t)s * total + (high ? total - 1 - pos : pos)] = k;
    }
    const bool to_scb = valid && rc == kCompToSCB;
    if (cqc) {
      const unsigned long long pos = block_append<NW>(cqc, to_scb, s_app);
      if (to_scb) cq[pos] = k;
    }
    if (valid && !staged && !to_scb) comp_store<Dirs>(k, rc, Ef, mu, rng, dirs, oE, o2, nerr);
  }
}

// entries at the front (0) or back (1) of a staged component's queue
NCD int64_t queue_count(const unsigned long long* __restrict__ count, int back, int64_t total) {
  if (total < ((int64_t)1 << 32)) return (int64_t)(back ? *count >> 32 : *count & 0xFFFFFFFFull);
  return (int64_t)count[back * kMaxStaged];
}
// One launch per component: workgroups from nhigh on stream their waves' shares
// of the queue's front (sab_stream), the first nhigh sample the neutrons above
// the table's Emax at its back (free-gas extender).  Together the two hide each
// other's latencies, and the pick has parted them: told apart here, each refill
// of a wave appended to the extender's queue by an atomic of its own.
template <bool Dirs, bool Lds>
__global__ void __launch_bounds__(256, 4) k_comp_sab(SABView s, const double* __restrict__ ekin,
                                                     const double* __restrict__ dirs, int64_t n, int64_t total,
                                                     uint64_t seed, uint32_t stream, int skip,
                                                     double* __restrict__ oE, double* __restrict__ o2,
                                                     unsigned long long* __restrict__ nerr,
                                                     const int64_t* __restrict__ q,
                                                     const unsigned long long* __restrict__ count, unsigned nhigh) {
  __shared__ double lds[Lds ? kSabLds : 1];
  if (blockIdx.x < nhigh) {
    const int64_t m = queue_count(count, 1, total);
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < m; j += (int64_t)nhigh * blockDim.x) {
      const int64_t k = q[total - 1 - j];
      Rng rng;
      rng.init(seed, stream, (uint64_t)k);
      if (skip) rng.gen();
      double Ef, mu;
      const int rc = sab_sample_iso(s, rng, ekin[(total == n) ? k : (k % n)], Ef, mu);
      comp_store<Dirs>(k, rc, Ef, mu, rng, dirs, oE, o2, nerr);
    }
    return;
  }
  const int64_t m = queue_count(count, 0, total);
  if (m == 0) return;
  const SabSmall<Lds> small(s, lds);
  const SabShare share(m, (blockIdx.x - nhigh) * 4 + (threadIdx.x >> 6), (gridDim.x - nhigh) * 4);
  sab_stream<Dirs>(
      s, small, seed, stream, skip, share,
      [&](int64_t i, int64_t& k, double& E) {
        k = q[share.at(i)];
        E = ekin[(total == n) ? k : (k % n)];
        return true;
      },
      [](bool) {},
      [&](int64_t k, int rc, double Ef, double mu) {
        if (rc) atomicAdd(nerr, 1ull);
        oE[k] = rc ? -1.0 : Ef;
        if constexpr (Dirs) {  // errors only
          o2[3 * k] = 0.0; o2[3 * k + 1] = 0.0; o2[3 * k + 2] = 0.0;
        } else {
          o2[k] = rc ? -999.0 : mu;
        }
      },
      [&](int64_t k, double Ef, double ox, double oy, double oz) {
        oE[k] = Ef;
        o2[3 * k] = ox; o2[3 * k + 1] = oy; o2[3 * k + 2] = oz;
      },
      [&](int64_t k, double& ix, double& iy, double& iz) {
        ix = dirs[3 * k]; iy = dirs[3 * k + 1]; iz = dirs[3 * k + 2];
      });
}

// stage kernel of a FreeGas component beside S(alpha,beta) components: the
// queued neutrons restart their stream, replay the pick's draw and sample
// the free-gas collision
template <bool Dirs>
__global__ void __launch_bounds__(256) k_comp_fg(FGView g, const double* __restrict__ ekin,
                                                 const double* __restrict__ dirs, int64_t n, int64_t total,
                                                 uint64_t seed, uint32_t stream, int skip, double* __restrict__ oE,
                                                 double* __restrict__ o2, unsigned long long* __restrict__ nerr,
                                                 const int64_t* __restrict__ inq,
                                                 const unsigned long long* __restrict__ inqc) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  const int64_t nq = queue_count(inqc, 0, total);
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nq; q += gstride) {
    const int64_t k = inq[q];
    Rng rng;
    rng.init(seed, stream, (uint64_t)k);
    if (skip) rng.gen();
    double Ef, mu;
    const int rc = fg_sample_demu(g, rng, ekin[(total == n) ? k : (k % n)], Ef, mu);
    comp_store<Dirs>(k, rc, Ef, mu, rng, dirs, oE, o2, nerr);
  }
}

// The stages of a composition within one workgroup: its `per` neutrons are
// picked, listed in LDS by component (below the table's Emax from the front of
// its list, above it from the back) and sampled there, without queues in memory,
// counters to clear or launches to wait for.  Such small batches are bound by
// the latency of their longest rejection (a step of sab_stream takes about 5 us
// on its own), so the neutrons are spread over the chip first, down to 16 a
// workgroup, and the lists over its waves.
template <bool Dirs, bool Gas, bool Lds>
__global__ void __launch_bounds__(256, 4) k_comp_local(CompView c, const double* __restrict__ ekin,
                                                       const double* __restrict__ dirs, int64_t n, int64_t total,
                                                       uint64_t seed, uint32_t stream, double* __restrict__ oE,
                                                       double* __restrict__ o2,
                                                       unsigned long long* __restrict__ nerr,
                                                       const double* __restrict__ ext, int64_t* __restrict__ cq,
                                                       unsigned long long* __restrict__ cqc, int per) {
  constexpr int kList = 256;
  __shared__ double lds[Lds ? kSabLds : 1];
  __shared__ unsigned char list[kMaxStaged][kList];
  __shared__ int count[2 * kMaxStaged];
  __shared__ unsigned long long s_app[5];
  const int tid = (int)threadIdx.x;
  if (tid < 2 * kMaxStaged) count[tid] = 0;
  __syncthreads();
  const int64_t k0 = (int64_t)blockIdx.x * per;
  {
    const int64_t k = k0 + tid;
    const bool valid = tid < per && k < total;
    Rng rng;
    double Ef = 0.0, mu = 0.0;
    int slot = 0, rc = kCompToStage + kCompToSCB + 1;  // neither list
    if (valid) {
      const double E = ekin[(total == n) ? k : (k % n)];
      rng.init(seed, stream, (uint64_t)k);
      rc = comp_pick_sample<Gas>(c, rng, E, Ef, mu, slot, ext ? ext[k] : 0.0);
      if (rc == kCompToStage) {
        const bool high = c.kind[c.stage_comp[slot]] == kKindSAB && !(E < c.sab[slot].egrid[c.sab[slot].ne - 1]);
        const int pos = atomicAdd(&count[high ? kMaxStaged + slot : slot], 1);
        list[slot][high ? kList - 1 - pos : pos] = (unsigned char)tid;
      }
    }
    const bool to_scb = valid && rc == kCompToSCB;
    if (cqc) {
      const unsigned long long pos = block_append<4>(cqc, to_scb, s_app);
      if (to_scb) cq[pos] = k;
    }
    if (valid && rc != kCompToStage && !to_scb) comp_store<Dirs>(k, rc, Ef, mu, rng, dirs, oE, o2, nerr);
  }
  __syncthreads();
  const int skip = c.n > 1 ? 1 : 0;
  for (int sl = 0; sl < c.nstaged; ++sl) {
    const int low = count[sl], high = count[kMaxStaged + sl];
    if (Gas && c.kind[c.stage_comp[sl]] == kKindFG) {
      for (int j = tid; j < low; j += 256) {
        const int64_t k = k0 + list[sl][j];
        Rng rng;
        rng.init(seed, stream, (uint64_t)k);
        if (skip) rng.gen();
        double Ef, mu;
        const int rc = fg_sample_demu(c.fg[c.stage_comp[sl]], rng, ekin[(total == n) ? k : (k % n)], Ef, mu);
        comp_store<Dirs>(k, rc, Ef, mu, rng, dirs, oE, o2, nerr);
      }
      continue;
    }
    const SABView& s = c.sab[sl];
    if (low > 0) {
      const SabSmall<Lds> small(s, lds);
      const SabRun share(low, tid >> 6, 4, 32);
      sab_stream<Dirs>(
          s, small, seed, stream, skip, share,
          [&](int64_t i, int64_t& k, double& E) {
            k = k0 + list[sl][share.at(i)];
            E = ekin[(total == n) ? k : (k % n)];
            return true;
          },
          [](bool) {},
          [&](int64_t k, int rc, double Ef, double mu) {
            if (rc) atomicAdd(nerr, 1ull);
            oE[k] = rc ? -1.0 : Ef;
            if constexpr (Dirs) {  // errors only
              o2[3 * k] = 0.0; o2[3 * k + 1] = 0.0; o2[3 * k + 2] = 0.0;
            } else {
              o2[k] = rc ? -999.0 : mu;
            }
          },
          [&](int64_t k, double Ef, double ox, double oy, double oz) {
            oE[k] = Ef;
            o2[3 * k] = ox; o2[3 * k + 1] = oy; o2[3 * k + 2] = oz;
          },
          [&](int64_t k, double& ix, double& iy, double& iz) {
            ix = dirs[3 * k]; iy = dirs[3 * k + 1]; iz = dirs[3 * k + 2];
          });
    }
    for (int j = 255 - tid; j < high; j += 256) {  // from the waves that had the least above
      const int64_t k = k0 + list[sl][kList - 1 - j];
      Rng rng;
      rng.init(seed, stream, (uint64_t)k);
      if (skip) rng.gen();
      double Ef, mu;
      const int rc = sab_sample_iso(s, rng, ekin[(total == n) ? k : (k % n)], Ef, mu);
      comp_store<Dirs>(k, rc, Ef, mu, rng, dirs, oE, o2, nerr);
    }
  }
}

__global__ void __launch_bounds__(256) k_sab_ab(SABView s, const double* __restrict__ ekin, int64_t n,
                                                uint64_t seed, uint32_t stream, double* __restrict__ oa,
                                                double* __restrict__ ob,
                                                unsigned long long* __restrict__ nerr) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gstride) {
    Rng rng;
    rng.init(seed, stream, (uint64_t)k);
    double a, b;
    const int rc = sab_sample_ab(s, ekin[k], rng, a, b);
    if (rc) { a = -1.0; b = 0.0; atomicAdd(nerr, 1ull); }
    oa[k] = a;
    ob[k] = b;
  }
}

// S(alpha,beta)-only materials: the free-gas extender (E >= Emax) is rare and
// register-hungry, so the main kernel leaves those neutrons in a queue that a
// second kernel drains.  Both draw from the neutron's own Philox stream from
// its first draw, so the split does not change any result.
template <bool Lds>
__global__ void __launch_bounds__(256, 4) k_sab_sample_iso_main(SABView s, const double* __restrict__ ekin,
                                                                int64_t n, int64_t total, uint64_t seed,
                                                                uint32_t stream, double* __restrict__ oE,
                                                                double* __restrict__ oMu,
                                                                unsigned long long* __restrict__ nerr,
                                                                int64_t* __restrict__ queue,
                                                                unsigned long long* __restrict__ qcount,
                                                                int domain_check) {
  __shared__ double lds[Lds ? kSabLds : 1];
  // places in the share of neutrons for the high-energy queue, kept until there are
  // four waves of them: appends to it run one after the other, 13 ns each, and
  // would pace a batch that has many (5e6 of 1e7, in order: 1.85 ms with one
  // append per wave of them)
  constexpr int kKeep = 256;
  __shared__ uint32_t bufs[4][kKeep + 64];
  __shared__ int counts[4];
  const int lane = (int)(threadIdx.x & 63);
  uint32_t* buf = bufs[threadIdx.x >> 6];
  int* have = counts + (threadIdx.x >> 6);
  if (lane == 0) *have = 0;
  __syncthreads();
  const SabSmall<Lds> small(s, lds);
  const SabShare share(total, blockIdx.x * 4 + (threadIdx.x >> 6), gridDim.x * 4);
  const double emax = s.egrid[s.ne - 1];
  sab_stream<false>(
      s, small, seed, stream, 0, share,
      [&](int64_t i, int64_t& k, double& E) {
        k = share.at(i);
        E = ekin[(total == n) ? k : (k % n)];
        if (domain_check && !(E >= 0.0 && E <= __builtin_huge_val())) {
          // a composition outside its energy domain does not scatter
          oE[k] = E;
          oMu[k] = 1.0;
          return false;
        }
        if (E < emax) return true;
        // the free-gas kernel, and the sampler's own handling of non-finite E
        buf[atomicAdd(have, 1)] = (uint32_t)i;
        return false;
      },
      [&](bool last) {  // at most kKeep - 1 kept and 64 new ones
        wave_lds_fence();
        const int c = *have;
        if (c < (last ? 1 : kKeep)) return;
        unsigned long long at = 0ull;
        if (lane == 0) at = atomicAdd(qcount, (unsigned long long)c);
        at = __shfl(at, 0, 64);
        for (int j = lane; j < c; j += 64) queue[at + j] = share.at(buf[j]);
        wave_lds_fence();
        if (lane == 0) *have = 0;
        wave_lds_fence();
      },
      [&](int64_t k, int rc, double Ef, double mu) {
        if (rc) atomicAdd(nerr, 1ull);
        oE[k] = rc ? -1.0 : Ef;
        oMu[k] = rc ? -999.0 : mu;
      },
      [](int64_t, double, double, double, double) {}, [](int64_t, double&, double&, double&) {});
}

__global__ void __launch_bounds__(256) k_sab_sample_iso_highe(SABView s, const double* __restrict__ ekin,
                                                              int64_t n, int64_t total, uint64_t seed,
                                                              uint32_t stream, double* __restrict__ oE,
                                                              double* __restrict__ oMu,
                                                              unsigned long long* __restrict__ nerr,
                                                              const int64_t* __restrict__ queue,
                                                              const unsigned long long* __restrict__ qcount) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  const int64_t nq = (int64_t)*qcount;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nq; q += gstride) {
    const int64_t k = queue[q];
    const int64_t i = (total == n) ? k : (k % n);
    Rng rng;
    rng.init(seed, stream, (uint64_t)k);
    double Ef, mu;
    const int rc = sab_sample_iso(s, rng, ekin[i], Ef, mu);
    if (rc) { Ef = -1.0; mu = -999.0; atomicAdd(nerr, 1ull); }
    oE[k] = Ef;
    oMu[k] = mu;
  }
}

// search-acceleration tables of an S(alpha,beta) process (built once)
__global__ void k_sab_cdf_guides(SABView s, unsigned short* __restrict__ guide) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per = kCdfGuide + 1;
  if (t >= (int64_t)s.ne * per) return;
  const int ie = (int)(t / per), g = (int)(t % per);
  const int4 hdr = s.shdr[ie];
  unsigned short r = 0;
  if (hdr.x == 1) {
    const double* cdf = s.scdf + (size_t)ie * (s.nb + 1);
    r = (unsigned short)lower_bound_d(cdf, 0, hdr.z, (double)g / (double)kCdfGuide);
  }
  guide[t] = r;
}
__global__ void k_sab_row_guides(SABView s, unsigned short* __restrict__ guide, double* __restrict__ scale) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per = kRowGuide + 1;
  if (t >= (int64_t)s.nb * per) return;
  const int ib = (int)(t / per), g = (int)(t % per);
  const double* row = s.cumul + (size_t)ib * s.na;
  const double rmax = row[s.na - 1];
  const double rs = rmax > 0.0 ? (double)kRowGuide / rmax : 0.0;
  if (g == 0) scale[ib] = rs;
  int lo = g == kRowGuide ? s.na : 0, n = s.na - lo;  // the last entry is na
  while (n > 0) {
    const int h = n >> 1, m = lo + h;
    if (row_bucket(row[m], rs) < g) { lo = m + 1; n -= h + 1; } else n = h;
  }
  guide[t] = rs > 0.0 ? (unsigned short)lo : (unsigned short)0;
}
// the sampler's layout of the tables (built once, after the guides)
__global__ void k_sab_pack(SABView s, SabPt* __restrict__ pt, SabHead* __restrict__ head, SabBin* __restrict__ bin,
                           double* __restrict__ small) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < (int64_t)s.nb * s.na) {
    const double2 q = s.sl[t];
    pt[t] = SabPt{q.x, q.y, s.cumul[t]};
  }
  if (t < (int64_t)s.ne * s.nb) {
    const int ie = (int)(t / s.nb), row = s.shdr[ie].y + (int)(t % s.nb);
    const AInfo i = s.sinfo[t];
    SabHead h{i.prob_front, i.prob_notback, 0.0, 0.0};
    if (row < s.nb) {  // (the records past the last row are not used)
      h.cl = s.cumul[(size_t)row * s.na + i.f_idx];
      h.cu = s.cumul[(size_t)row * s.na + i.b_idx];
    }
    head[t] = h;
  }
  if (t < (int64_t)s.ne * (s.nb + 1)) {
    const double2 q = s.sxy[t];
    bin[t] = SabBin{s.scdf[t], q.x, q.y};
  }
  if (t < s.na) small[t] = s.alpha[t];
  if (t < s.nb) {
    small[s.na + t] = s.beta[t];
    small[s.na + s.nb + t] = s.row_scale[t];
  }
  if (t < s.ne) {
    double* e = small + s.na + 2 * s.nb;
    e[t] = s.egrid[t];
    const int4 h = s.shdr[t];
    const int nv = h.x == 1 ? h.z : (h.x == 0 ? -1 : -2);
    e[s.ne + 2 * t] = s.sfirst[t];
    e[s.ne + 2 * t + 1] = __longlong_as_double((long long)(((unsigned long long)(unsigned)nv << 32) | (unsigned)h.y));
  }
}

static inline unsigned grid_for(int64_t n, int bs) {
  int64_t g = (n + bs - 1) / bs;
  // enough waves for the 256 CUs, bounded so a grid-stride loop covers the rest
  const int64_t gmax = 256 * 64;
  if (g > gmax) g = gmax;
  if (g < 1) g = 1;
  return (unsigned)g;
}

// persistent kernels: four workgroups (of four waves) per CU
static inline unsigned stream_grid(int64_t n) {
  const int64_t g = (n + 255) / 256;
  return (unsigned)(g < 1 ? 1 : (g > 1024 ? 1024 : g));
}

__global__ void k_zero_u64(unsigned long long* p) { *p = 0ull; }

__global__ void k_zero_u64_n(unsigned long long* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0ull;
}

// the stage launches of a composition with an S(alpha,beta) part, after the
// pick kernel filled one queue per staged component from both ends (queues +
// s * total, counters at qcount + s)
template <bool Dirs>
void launch_stages(const CompView& c, const double* ekin, const double* dirs, int64_t n, int64_t total,
                   uint64_t seed, uint32_t stream, double* oE, double* o2, unsigned long long* nerr,
                   int64_t* queues, unsigned long long* qcount, hipStream_t st) {
  const int skip = c.n > 1 ? 1 : 0;
  const dim3 b(256);
  const unsigned gs = stream_grid(total), nhigh = gs < 512 ? gs : 512;
  for (int sl = 0; sl < c.nstaged; ++sl) {
    const int comp = c.stage_comp[sl];
    int64_t* q = queues + (int64_t)sl * total;
    if (c.kind[comp] == kKindSAB) {
      if (sab_small_fits(c.sab[sl]))
        hipLaunchKernelGGL((k_comp_sab<Dirs, true>), dim3(gs + nhigh), b, 0, st, c.sab[sl], ekin, dirs, n, total, seed,
                           stream, skip, oE, o2, nerr, q, qcount + sl, nhigh);
      else
        hipLaunchKernelGGL((k_comp_sab<Dirs, false>), dim3(gs + nhigh), b, 0, st, c.sab[sl], ekin, dirs, n, total,
                           seed, stream, skip, oE, o2, nerr, q, qcount + sl, nhigh);
    } else {
      hipLaunchKernelGGL(k_comp_fg<Dirs>, dim3(grid_for(total, 256)), b, 0, st, c.fg[comp], ekin, dirs, n, total, seed,
                         stream, skip, oE, o2, nerr, q, qcount + sl);
    }
  }
}


// Batches of at most 1024 workgroups of 256 neutrons, what the chip holds at once
// (four to a CU), are staged within workgroups; beyond, the second round's
// workgroups cost more than the queues.  Within workgroups against through queues
// [us], isotropic calls, powder (one S(alpha,beta)) and rock salt (two):
//   neutrons      1000     100000     200000     260000     300000     1000000
//   powder      27   43   48   58    63   65    66   70    95   81   208  151
//   rock salt   39   76   67  101    78  106    81  110   119  126   261  194
constexpr int64_t kLocalMax = 1024 * 256;
bool staged_locally(int64_t total) { return total <= kLocalMax; }
template <bool Dirs>
void launch_staged(const CompView& c, const double* ekin, const double* dirs, int64_t n, int64_t total, uint64_t seed,
                   uint32_t stream, double* oE, double* o2, unsigned long long* nerr, int64_t* queues,
                   unsigned long long* qcount, hipStream_t st, const double* ext, int64_t* cq,
                   unsigned long long* cqc) {
  const bool gas = comp_has_gas(c);
  if (staged_locally(total)) {
    bool fits = true;
    for (int sl = 0; sl < c.nstaged; ++sl)
      if (c.kind[c.stage_comp[sl]] == kKindSAB) fits = fits && sab_small_fits(c.sab[sl]);
    const int64_t spread = (total + 767) / 768;  // three workgroups per CU
    const int per = (int)(spread < 16 ? 16 : (spread > 256 ? 256 : spread));
    const dim3 g((unsigned)((total + per - 1) / per)), b(256);
    const auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, g, b, 0, st, c, ekin, dirs, n, total, seed, stream, oE, o2, nerr, ext, cq, cqc, per);
    };
    if (gas) fits ? go(k_comp_local<Dirs, true, true>) : go(k_comp_local<Dirs, true, false>);
    else fits ? go(k_comp_local<Dirs, false, true>) : go(k_comp_local<Dirs, false, false>);
    return;
  }
  hipLaunchKernelGGL(k_zero_u64_n, dim3(1), dim3(64), 0, st, qcount, 2 * kMaxStaged);
  const dim3 g(grid_for(total, kPickThreads)), b(kPickThreads);
  hipLaunchKernelGGL((gas ? k_comp_pick<Dirs, true> : k_comp_pick<Dirs, false>), g, b, 0, st, c, ekin, dirs, n, total,
                     seed, stream, oE, o2, nerr, queues, qcount, ext, cq, cqc);
  launch_stages<Dirs>(c, ekin, dirs, n, total, seed, stream, oE, o2, nerr, queues, qcount, st);
}


// synthetic neutron energies, log-uniform, from a dedicated Philox stream
__global__ void __launch_bounds__(256) k_fill_loguniform(double* __restrict__ out, int64_t n, double lemin,
                                                         double lemax, uint64_t seed) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gstride) {
    Rng rng;
    rng.init(seed, 0xFFFFFFFFu, (uint64_t)k);
    const double u = rng.gen();
    out[k] = exp(lemin + u * (lemax - lemin));
  }
}


void launch_simple_xs(int kind, const FGView& g, double abs_c, const double* ekin, int64_t n, int64_t repeat,
                      double* out, hipStream_t st) {
  const int64_t total = n * repeat;
  if (total <= 0) return;
  hipLaunchKernelGGL(k_simple_xs, dim3(grid_for(total, 256)), dim3(256), 0, st, kind, g, abs_c, ekin, n, total, out);
}
void launch_fg_sample(const FGView& g, const double* ekin, const double* dirs, int64_t n, int64_t repeat,
                      uint64_t seed, uint32_t stream, double* oE, double* oX, unsigned long long* nerr,
                      hipStream_t st) {
  const int64_t total = n * repeat;
  if (total <= 0) return;
  if (dirs)
    hipLaunchKernelGGL(k_fg_sample<true>, dim3(grid_for(total, 256)), dim3(256), 0, st, g, ekin, dirs, n, total, seed,
                       stream, oE, oX, nerr);
  else
    hipLaunchKernelGGL(k_fg_sample<false>, dim3(grid_for(total, 256)), dim3(256), 0, st, g, ekin, dirs, n, total,
                       seed, stream, oE, oX, nerr);
}


void launch_xs_iso(const CompView& c, const double* ekin, int64_t n, int64_t repeat, double* out,
                   bool fp32, hipStream_t st) {
  if (n <= 0 || repeat <= 0) return;
  const dim3 g(grid_for(n, 256)), b(256);
  const bool past = past_caches(8 * n * (1 + repeat));
  const int v = comp_variant(c);
  const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, b, 0, st, c, ekin, n, repeat, out); };
  const auto variant = [&](auto kind) {
    constexpr int V = decltype(kind)::value;
    if (fp32) past ? go(k_xs_iso<true, V, true>) : go(k_xs_iso<true, V, false>);
    else past ? go(k_xs_iso<false, V, true>) : go(k_xs_iso<false, V, false>);
  };
  if (v == kCompPBOnly) variant(std::integral_constant<int, kCompPBOnly>{});
  else if (v == kCompFG || comp_has_gas(c)) variant(std::integral_constant<int, kCompFG>{});
  else variant(std::integral_constant<int, kCompNoSAB>{});
}
void launch_sample_iso(const CompView& c, const double* ekin, int64_t n, int64_t repeat, uint64_t seed,
                       uint32_t stream, double* oE, double* oMu, unsigned long long* nerr, int64_t* queues,
                       unsigned long long* qcount, hipStream_t st) {
  const int64_t total = n * repeat;
  if (total <= 0) return;
  const bool past = past_caches(8 * n + 16 * total);
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid_for(total, 256)), dim3(256), 0, st, c, ekin, n, total, seed, stream, oE, oMu,
                       nerr);
  };
  switch (comp_variant(c)) {
    case kCompPBOnly:
      past ? go(k_sample_iso<kCompPBOnly, true>) : go(k_sample_iso<kCompPBOnly, false>);
      break;
    case kCompNoSAB:
      past ? go(k_sample_iso<kCompNoSAB, true>) : go(k_sample_iso<kCompNoSAB, false>);
      break;
    case kCompFG:
      past ? go(k_sample_iso<kCompFG, true>) : go(k_sample_iso<kCompFG, false>);
      break;
    default:
      launch_staged<false>(c, ekin, nullptr, n, total, seed, stream, oE, oMu, nerr, queues, qcount, st, nullptr,
                           nullptr, nullptr);
  }
}
__global__ void __launch_bounds__(256) k_xs_ext(CompView c, const double* __restrict__ ekin,
                                                const double* __restrict__ ext, int64_t n, double* __restrict__ out) {
  const int64_t gstride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gstride)
    out[k] = comp_xs<false, true>(c, ekin[k], nullptr, ext[k]);  // FreeGas components may sit beside SCBragg
}
void launch_xs_ext(const CompView& c, const double* ekin, const double* ext, int64_t n, double* out,
                   hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_xs_ext, dim3(grid_for(n, 256)), dim3(256), 0, st, c, ekin, ext, n, out);
}

void launch_sample_dirs(const CompView& c, const double* ekin, const double* dirs, int64_t n, uint64_t seed,
                        uint32_t stream, double* oE, double* oD, unsigned long long* nerr, int64_t* queues,
                        unsigned long long* qcount, hipStream_t st, const double* ext, int64_t* cq,
                        unsigned long long* cqc) {
  if (cqc) hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, st, cqc);
  if (n <= 0) return;
  switch (comp_variant(c)) {
    case kCompPBOnly:
      hipLaunchKernelGGL(k_sample_dirs<kCompPBOnly>, dim3(grid_for(n, 256)), dim3(256), 0, st, c, ekin, dirs, n,
                         seed, stream, oE, oD, nerr);
      break;
    case kCompNoSAB:
      hipLaunchKernelGGL(k_sample_dirs<kCompNoSAB>, dim3(grid_for(n, 256)), dim3(256), 0, st, c, ekin, dirs, n,
                         seed, stream, oE, oD, nerr);
      break;
    case kCompFG:
      hipLaunchKernelGGL(k_sample_dirs<kCompFG>, dim3(grid_for(n, 256)), dim3(256), 0, st, c, ekin, dirs, n,
                         seed, stream, oE, oD, nerr);
      break;
    default:
      launch_staged<true>(c, ekin, dirs, n, n, seed, stream, oE, oD, nerr, queues, qcount, st, ext, cq, cqc);
  }
}
void launch_sab_ab(const SABView& s, const double* ekin, int64_t n, uint64_t seed, uint32_t stream, double* oa,
                   double* ob, unsigned long long* nerr, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_sab_ab, dim3(grid_for(n, 256)), dim3(256), 0, st, s, ekin, n, seed, stream, oa, ob, nerr);
}

void launch_sab_sample_iso(const SABView& s, const double* ekin, int64_t n, int64_t repeat, uint64_t seed,
                           uint32_t stream, double* oE, double* oMu, unsigned long long* nerr, int64_t* queue,
                           unsigned long long* qcount, int domain_check, hipStream_t st) {
  const int64_t total = n * repeat;
  if (total <= 0) return;
  // kernel instead of a memset node, so that callers may capture this in a graph
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, st, qcount);
  if (sab_small_fits(s))
    hipLaunchKernelGGL(k_sab_sample_iso_main<true>, dim3(stream_grid(total)), dim3(256), 0, st, s, ekin, n, total,
                       seed, stream, oE, oMu, nerr, queue, qcount, domain_check);
  else
    hipLaunchKernelGGL(k_sab_sample_iso_main<false>, dim3(stream_grid(total)), dim3(256), 0, st, s, ekin, n, total,
                       seed, stream, oE, oMu, nerr, queue, qcount, domain_check);
  hipLaunchKernelGGL(k_sab_sample_iso_highe, dim3(grid_for(total, 256)), dim3(256), 0, st, s, ekin, n, total, seed,
                     stream, oE, oMu, nerr, queue, qcount);
}
__global__ void k_copy_u64(const unsigned long long* __restrict__ from, unsigned long long* __restrict__ to) {
  *to = *from;
}
void launch_copy_u64(const unsigned long long* from, unsigned long long* to, hipStream_t st) {
  hipLaunchKernelGGL(k_copy_u64, dim3(1), dim3(1), 0, st, from, to);
}
void launch_zero_u64(unsigned long long* p, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, st, p);
}
void launch_sab_queue(const SABView& s, const double* ekin, int64_t n, int64_t total, uint64_t seed, uint32_t stream,
                      double* oE, double* oMu, unsigned long long* nerr, const int64_t* queue,
                      const unsigned long long* qcount, hipStream_t st) {
  hipLaunchKernelGGL(k_sab_sample_iso_highe, dim3(grid_for(total, 256)), dim3(256), 0, st, s, ekin, n, total, seed,
                     stream, oE, oMu, nerr, queue, qcount);
}
void launch_sab_guides(const SABView& s, unsigned short* cdf_guide, unsigned short* row_guide, double* row_scale,
                       hipStream_t st) {
  const int64_t n1 = (int64_t)s.ne * (kCdfGuide + 1);
  hipLaunchKernelGGL(k_sab_cdf_guides, dim3((unsigned)((n1 + 255) / 256)), dim3(256), 0, st, s, cdf_guide);
  const int64_t n2 = (int64_t)s.nb * (kRowGuide + 1);
  hipLaunchKernelGGL(k_sab_row_guides, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, st, s, row_guide,
                     row_scale);
}
void launch_sab_pack(const SABView& s, SabPt* pt, SabHead* head, SabBin* bin, double* small, hipStream_t st) {
  const int64_t n = std::max((int64_t)s.nb * s.na, (int64_t)s.ne * (s.nb + 1));
  hipLaunchKernelGGL(k_sab_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, s, pt, head, bin, small);
}
void launch_fill_loguniform(double* out, int64_t n, double lemin, double lemax, uint64_t seed, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_loguniform, dim3(grid_for(n, 256)), dim3(256), 0, st, out, n, lemin, lemax, seed);
}

}  // namespace ncamd

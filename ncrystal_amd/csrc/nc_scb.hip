// Per-neutron kernels of the mosaic single-crystal Bragg process: oriented
// cross sections and scatter sampling, one lane per neutron.
//
// Scheduling: the cost of a neutron is the number of demi-normals of the
// families with 2d > lambda, which varies as lambda^-3 across a batch.  A
// counting sort by that number (k_scb_keys / k_scb_offsets / k_scb_scatter)
// gives every wavefront neutrons of nearly equal cost; the kernels then take
// neutron perm[k] in lane k.  Results are written at the neutron's own index
// and every neutron draws from its own Philox stream, so the order changes
// no result.
//
// Each kernel pair is a main kernel without the Romberg circle integral and
// a queue kernel that redoes, with it, the neutrons whose scan met a
// contribution outside the spline's validity (backscattering within the
// mosaic spread), one wave per neutron or, for long queues of a narrow beam,
// several or one lane (scb_wave_group).  Cross sections involve no random numbers
// and sampling draws from the neutron's own Philox stream from its first draw, so
// the split does not change any result either.
//
// Reference: ncrystal_core/src/scbragg/NCSCBragg.cc:233-323 (crossSection,
// sampleScatter), ncrystal_core/src/cinterface/ncrystal.cc:1248-1282 (batched
// layout).
#include "nc_kernels.hh"

namespace ncamd {

namespace {

NCD void scb_xs_one(const SCBView& v, bool valid, int64_t i, const double* __restrict__ ekin,
                    const double* __restrict__ dirs, double* __restrict__ out, int64_t* __restrict__ queue,
                    unsigned long long* __restrict__ qcount, uint16_t* __restrict__ list) {
  ScbLane L;
  L.wl = 1.0;
  L.u = V3{0.0, 0.0, 1.0};
  L.jlim = 0;
  bool can = false;
  if (valid) can = scb_lane_setup(v, ekin[i], dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2], L);
  scb_walk<false>(v, L, 0, 0.0, list);
  if (!valid) return;
  if (L.slow) {
    const unsigned long long slot = atomicAdd(qcount, 1ull);
    queue[slot] = i;
    return;
  }
  out[i] = (can && L.count) ? L.total : 0.0;
}

// Contributions of one neutron evaluated by a whole wave, with the Romberg
// circle integral: lane t tests demi-normal jb + t; the candidates collect in
// order in the wave's list and are evaluated 64 at a time, one per lane, but for
// their Romberg integrals: a few take the whole wave one after the other, a point
// per lane (on its own lane each would hold the wave for its 17 points and more);
// the contributions are then added up in order (the sums and
// the selection of scb_eval_list) from the lanes' registers.  The queue usually
// holds few neutrons (0.2 % of a beam on a 30 arcmin crystal), each with a long
// scan and some integrals: one lane per neutron left 60 waves to run 0.8 ms
// (cross sections of 2e6 neutrons) and 1.8 ms (two passes, sampling).
// The scan keeps four loads in flight (a scan of 15000 demi-normals, 1 Aa, is
// otherwise one load's latency per 64 of them), and the selection reads the
// candidates from the list where it held them all.
constexpr int kScbWaveList = 1024;
constexpr int kScbWaveLoads = 4;
static_assert(2 * kScbWaveList * sizeof(int) >= kScbListWave * sizeof(uint16_t), "a wave's lists, of either kind");
// integrals of a batch that the wave does together; more are done a lane each
// (5 degree crystal, dozens in a batch, 30000 isotropic neutrons: 15 ms together,
// 4.8 a lane each)
constexpr int kScbWaveSlow = 2;
// A narrow beam near backscattering puts most of a batch in the queue.  Then a
// wave takes several neutrons in a row and, where their directions are as close
// as for the wave-level filter (scb_walk), scans the demi-normals once for all of
// them: the ones left are the list that each neutron tests.
constexpr int kScbWaveGroup = 32;
constexpr int kScbWaveShare = 3;  // from this many neutrons on
// lists of a wave in LDS: the neutron's candidates, the group's demi-normals (n
// of them, or -1: scan all)
struct ScbWaveLists {
  int* cand;
  int* near;
  int n;
};
// neutrons of a wave at a time, of a queue of nq: several if 64 of them, from all
// over the queue, are close (every wave finds the same), and 64 of these, one per
// lane, if there are enough to fill the chip that way: lanes with the same
// candidates cost one evaluation for 64 neutrons, and add up side by side.
// Otherwise one, and the next a launch's waves on: the queue is sorted by scan
// length, and neighbours would all be the long ones.
// Cross sections / sampling, all neutrons queued, narrow beam: 20000 at
// backscattering off a 0.2 degree crystal 0.33 / 0.59 ms with one per wave, 0.26 /
// 0.44 several, 0.26 / 0.38 in lanes; off a 5 degree crystal 2.28 / 4.51, 2.07 / 3.54
// and 3.23 / 5.90; 100000 of 1.5 Aa, 5 degrees: 9.8 / 21.2, 7.7 / 15.2 and 3.1 / 5.5.
constexpr int64_t kScbLaneQueue = 65536;
NCD int scb_wave_group(const SCBView& v, const double* __restrict__ ekin, const double* __restrict__ dirs,
                       const int64_t* __restrict__ queue, int64_t nq, int64_t nwaves) {
  const int64_t g = (nq + nwaves - 1) / nwaves;
  if (g < kScbWaveShare) return 1;
  const int64_t i = queue[(int64_t)((double)__lane_id() * ((double)nq * 0x1.0p-6))];
  ScbLane L;
  L.wl = 1.0;
  L.u = V3{0.0, 0.0, 1.0};
  scb_lane_setup(v, ekin[i], dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2], L);
  if (!scb_bounds(L.u, (float)gm_round(L.wl), true).ok) return 1;
  if (nq >= kScbLaneQueue) return 64;
  return (int)(g < kScbWaveGroup ? g : kScbWaveGroup);
}
NCD void scb_wave_near(const SCBView& v, const double* __restrict__ ekin, const double* __restrict__ dirs,
                       const int64_t* __restrict__ queue, int ng, ScbWaveLists& W) {
  W.n = -1;
  if (ng < kScbWaveShare) return;
  const int lane = (int)__lane_id();
  const uint64_t below = lane ? ~0ull >> (64 - lane) : 0ull;
  ScbLane L;
  L.wl = 1.0;
  L.u = V3{0.0, 0.0, 1.0};
  L.jlim = 0;
  if (lane < ng) {
    const int64_t i = queue[lane];
    scb_lane_setup(v, ekin[i], dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2], L);
  }
  const ScbBounds B = scb_bounds(L.u, (float)gm_round(L.wl), L.jlim > 0);
  const int jmax = wave_max_i(L.jlim);
  if (!B.ok) return;
  int n = 0;
  for (int jb = 0; jb < jmax; jb += 64) {
    const int j = jb + lane;
    const bool pass = j < jmax && scb_bounds_pass(v, B, v.nrec32[j < jmax ? j : jmax - 1]);
    const uint64_t M = __ballot(pass);
    if (n + __popcll(M) > kScbWaveList) return;
    if (pass) W.near[n + __popcll(M & below)] = j;
    n += __popcll(M);
  }
  wave_lds_fence();
  W.n = n;
}
template <bool Select>
NCD bool scb_wave_eval(const SCBView& v, ScbLane& L, ScbAcc& a, int n_select, double target, double w, double wl3,
                       const int* __restrict__ list, int n) {
  const int lane = (int)__lane_id();
  for (int b = 0; b < n; b += 64) {
    double4 r = make_double4(0.0, 0.0, 0.0, 0.0);
    double xs0 = 0.0, xs1 = 0.0;
    ScbSlow slow{0u, 0.0, 0.0, 0.0, 0.0};
    int f = 0;
    if (b + lane < n) {
      const int j = list[b + lane];
      r = v.nrec[j];
      const double2 nf = v.nfx[j];
      f = (int)nf.y;
      scb_candidate<true>(v, r, nf.x, w, wl3, L.u.x, L.u.y, L.u.z, xs0, xs1, &slow);
    }
    const uint64_t S0 = __ballot(slow.sides & 1u), S1 = __ballot(slow.sides & 2u);
    if (__popcll(S0) + __popcll(S1) > kScbWaveSlow) {
      scb_slow_sides(v, slow, xs0, xs1);
    } else {
#pragma nounroll
      for (int side = 0; side < 2; ++side) {
        uint64_t S = side ? S1 : S0;
#pragma nounroll
        while (S) {
          const int t = __builtin_ctzll(S);
          S &= S - 1ull;
          const double dot = readlane_d(slow.dot, t);
          const double cc = dclamp(side == 0 ? dot : -dot, -1.0, 1.0);
          const double ci = gos_circle_slow<true>(v, cc, sqrt(1.0 - cc * cc), readlane_d(slow.sinpt, t),
                                                  readlane_d(slow.cospt, t));
          if (lane == t) (side == 0 ? xs0 : xs1) = slow.Q * ci;
        }
      }
    }
    const uint64_t B0 = __ballot(xs0 != 0.0), B1 = __ballot(xs1 != 0.0);
    uint64_t C = B0 | B1;
    while (C) {
      const int t = __builtin_ctzll(C);
      C &= C - 1ull;
      const int ft = __builtin_amdgcn_readlane(f, t);
      if (ft != a.cur_f) {
        a.cur_f = ft;
        a.xsoffset = a.commul_last;
        a.xssum = 0.0;
      }
      for (int side = 0; side < 2; ++side) {
        if (!(((side ? B1 : B0) >> t) & 1ull)) continue;
        const double xs = readlane_d(side ? xs1 : xs0, t);
        const double cm = a.xsoffset + (a.xssum += xs);
        a.commul_last = cm;
        if constexpr (Select) {
          const bool hit = n_select < 5 ? (cm > target) : !(cm < target);
          if (hit || L.count == n_select - 1) {
            const double nx = readlane_d(r.x, t), ny = readlane_d(r.y, t), nz = readlane_d(r.z, t);
            L.found = true;
            L.sel_inv2d_r = readlane_d(r.w, t);
            L.sel_normal = side == 0 ? V3{-nx, -ny, -nz} : V3{nx, ny, nz};
            return true;
          }
        }
        L.count++;
      }
    }
  }
  return false;
}
// complete: the list holds all candidates (set by the first pass and taken by
// the second); nlist: their number
template <bool Select>
NCD void scb_wave_walk(const SCBView& v, ScbLane& L, int n_select, double target, const ScbWaveLists& W, int& nlist,
                       bool& complete) {
  const int lane = (int)__lane_id();
  const uint64_t below = lane ? ~0ull >> (64 - lane) : 0ull;
  int* list = W.cand;
  L.count = 0;
  L.total = 0.0;
  L.slow = false;
  L.found = false;
  const double w = gm_round(L.wl);
  const double wl3 = w * w * w;
  ScbAcc a{-1, 0.0, 0.0, 0.0};
  if (Select && complete) {
    scb_wave_eval<Select>(v, L, a, n_select, target, w, wl3, list, nlist);
    return;
  }
  const float fx = (float)L.u.x, fy = (float)L.u.y, fz = (float)L.u.z, fw = (float)w;
  int n = 0;
  complete = true;
  const int end = L.jlim > 0 && W.n >= 0 ? W.n : L.jlim;
  for (int jb = 0; jb < end; jb += 64 * kScbWaveLoads) {
    if (n > kScbWaveList - 64 * kScbWaveLoads) {
      wave_lds_fence();
      if (scb_wave_eval<Select>(v, L, a, n_select, target, w, wl3, list, n)) return;
      wave_lds_fence();
      n = 0;
      complete = false;
    }
    int js[kScbWaveLoads];
    float4 r[kScbWaveLoads];
#pragma unroll
    for (int q = 0; q < kScbWaveLoads; ++q) {
      const int at = jb + 64 * q + lane;
      js[q] = at < end ? (W.n >= 0 ? W.near[at] : at) : L.jlim;
      r[q] = v.nrec32[js[q] < L.jlim ? js[q] : L.jlim - 1];
    }
#pragma unroll
    for (int q = 0; q < kScbWaveLoads; ++q) {
      const bool cand = js[q] < L.jlim && scb_prefilter(v, r[q].x, r[q].y, r[q].z, r[q].w, fx, fy, fz, fw);
      const uint64_t M = __ballot(cand);
      if (cand) list[n + __popcll(M & below)] = js[q];
      n += __popcll(M);
    }
  }
  wave_lds_fence();
  nlist = n;
  if (scb_wave_eval<Select>(v, L, a, n_select, target, w, wl3, list, n)) return;
  L.total = a.commul_last;
}

}  // namespace

// ---- counting sort of the batch by scan length
__global__ void __launch_bounds__(256) k_scb_keys(SCBView v, const double* __restrict__ ekin,
                                                  const double* __restrict__ dirs, int64_t n,
                                                  unsigned* __restrict__ keys, unsigned* __restrict__ hist) {
  __shared__ unsigned lh[kScbBuckets];
  for (int b = threadIdx.x; b < kScbBuckets; b += blockDim.x) lh[b] = 0u;
  __syncthreads();
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    ScbLane L;
    L.jlim = 0;
    scb_lane_setup(v, ekin[i], dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2], L);
    // the scan length grows as the cube of the wave number: buckets of equal
    // wave-number width, which a batch of any spectrum fills evenly enough
    // that the counters below are not all taken at one place
    const unsigned c = (unsigned)(cbrtf((float)L.jlim / (float)(v.nnormals + 1)) * (float)kScbBuckets);
    const unsigned b = c < (unsigned)kScbBuckets ? c : (unsigned)kScbBuckets - 1u;
    keys[i] = b;
    atomicAdd(&lh[b], 1u);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < kScbBuckets; b += blockDim.x)
    if (lh[b]) atomicAdd(&hist[b], lh[b]);
}

// exclusive prefix sum of the bucket counts (one block); cursors start at
// the bucket offsets, the histogram is cleared for the next call
__global__ void __launch_bounds__(kScbBuckets) k_scb_offsets(unsigned* __restrict__ hist,
                                                              unsigned long long* __restrict__ cursor) {
  __shared__ unsigned long long s[kScbBuckets];
  const int t = threadIdx.x;
  s[t] = hist[t];
  __syncthreads();
  for (int o = 1; o < kScbBuckets; o <<= 1) {
    const unsigned long long x = t >= o ? s[t - o] : 0ull;
    __syncthreads();
    s[t] += x;
    __syncthreads();
  }
  cursor[t] = s[t] - hist[t];
  hist[t] = 0u;
}

// each block takes kScbScatterItems x 256 consecutive neutrons, ranks them
// inside the block with LDS atomics and reserves one range per bucket with
// a single global atomic, so that global atomics do not pile up on the few
// buckets a batch usually fills
constexpr int kScbScatterItems = 16;
__global__ void __launch_bounds__(256) k_scb_scatter(const unsigned* __restrict__ keys, int64_t n,
                                                     unsigned long long* __restrict__ cursor,
                                                     int64_t* __restrict__ perm) {
  __shared__ unsigned cnt[kScbBuckets];
  __shared__ unsigned long long base[kScbBuckets];
  const int64_t chunk = (int64_t)blockDim.x * kScbScatterItems;
  for (int64_t c0 = (int64_t)blockIdx.x * chunk; c0 < n; c0 += (int64_t)gridDim.x * chunk) {
    for (int b = threadIdx.x; b < kScbBuckets; b += blockDim.x) cnt[b] = 0u;
    __syncthreads();
    unsigned key[kScbScatterItems], rank[kScbScatterItems];
#pragma unroll
    for (int j = 0; j < kScbScatterItems; ++j) {
      const int64_t i = c0 + (int64_t)j * blockDim.x + threadIdx.x;
      key[j] = i < n ? keys[i] : 0u;
      rank[j] = i < n ? atomicAdd(&cnt[key[j]], 1u) : 0u;
    }
    __syncthreads();
    for (int b = threadIdx.x; b < kScbBuckets; b += blockDim.x)
      base[b] = cnt[b] ? atomicAdd(&cursor[b], (unsigned long long)cnt[b]) : 0ull;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kScbScatterItems; ++j) {
      const int64_t i = c0 + (int64_t)j * blockDim.x + threadIdx.x;
      if (i < n) perm[base[key[j]] + rank[j]] = i;
    }
    __syncthreads();
  }
}

__global__ void k_scb_clear(unsigned* __restrict__ hist, unsigned long long* __restrict__ qcount) {
  for (int b = threadIdx.x; b < kScbBuckets; b += blockDim.x) hist[b] = 0u;
  if (threadIdx.x == 0) *qcount = 0ull;
}

// ---- main and queue kernels.  Grid-stride loops step over whole blocks so
// that every lane of a wavefront reaches the wave-uniform scan together.
__global__ void __launch_bounds__(256) k_scb_xs_main(SCBView v, const double* __restrict__ ekin,
                                                     const double* __restrict__ dirs, int64_t n,
                                                     const int64_t* __restrict__ perm, double* __restrict__ out,
                                                     int64_t* __restrict__ queue,
                                                     unsigned long long* __restrict__ qcount) {
  __shared__ uint16_t lists[4 * kScbListWave];
  uint16_t* list = lists + (threadIdx.x >> 6) * kScbListWave;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n; base += stride) {
    const int64_t k = base + threadIdx.x;
    const bool valid = k < n;
    scb_xs_one(v, valid, valid ? perm[k] : 0, ekin, dirs, out, queue, qcount, list);
  }
}
__global__ void __launch_bounds__(256) k_scb_xs_slow(SCBView v, const double* __restrict__ ekin,
                                                     const double* __restrict__ dirs, double* __restrict__ out,
                                                     const int64_t* __restrict__ queue,
                                                     const unsigned long long* __restrict__ qcount) {
  __shared__ __align__(16) int lists[4][2][kScbWaveList];
  ScbWaveLists W{lists[threadIdx.x >> 6][0], lists[threadIdx.x >> 6][1], -1};
  const int64_t nq = (int64_t)*qcount;
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  const int group = scb_wave_group(v, ekin, dirs, queue, nq, nwaves);
  const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * group;
  if (group == 64) {
    for (int64_t q0 = first; q0 < nq; q0 += nwaves * 64) {
      const int64_t q = q0 + (threadIdx.x & 63);
      const int64_t i = queue[q < nq ? q : nq - 1];
      ScbLane L;
      L.wl = 1.0;
      L.u = V3{0.0, 0.0, 1.0};
      L.jlim = 0;
      const bool can = q < nq && scb_lane_setup(v, ekin[i], dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2], L);
      scb_walk<false, true>(v, L, 0, 0.0, reinterpret_cast<uint16_t*>(W.cand));
      if (q < nq) out[i] = (can && L.count) ? L.total : 0.0;
    }
    return;
  }
  // (every lane of a wave has the same q; from the end, where the longest scans are)
  for (int64_t q1 = nq - first; q1 > 0; q1 -= nwaves * group)
  for (int64_t q0 = q1 > group ? q1 - group : 0, q = q0; q < q1; ++q) {
    if (q == q0) scb_wave_near(v, ekin, dirs, queue + q0, (int)(q1 - q0), W);
    const int64_t i = queue[q];
    ScbLane L;
    const bool can = scb_lane_setup(v, ekin[i], dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2], L);
    int nlist = 0;
    bool complete = false;
    scb_wave_walk<false>(v, L, 0, 0.0, W, nlist, complete);
    if ((threadIdx.x & 63) == 0) out[i] = (can && L.count) ? L.total : 0.0;
  }
}
// Sampling in three kernels over the sorted batch (fewer registers each
// than one kernel doing it all): the first counts the contributions and
// their total for sorted position k (cnt[k], tot[k]; 0 for a neutron that
// does not scatter, whose output it writes, or that goes to the Romberg
// queue); the second draws the target and repeats the scan until the
// selected contribution (sel[k]: normal of the reflecting side, rounded
// 1/(2d); 0 if none); the third generates the scattered direction, with the
// neutron's Philox stream continued after the target draw.
__global__ void __launch_bounds__(256) k_scb_sample_count(SCBView v, const double* __restrict__ ekin,
                                                          const double* __restrict__ dirs, int64_t n,
                                                          const int64_t* __restrict__ perm, double* __restrict__ oE,
                                                          double* __restrict__ oD, int* __restrict__ cnt,
                                                          double* __restrict__ tot, int64_t* __restrict__ queue,
                                                          unsigned long long* __restrict__ qcount,
                                                          const int64_t* __restrict__ idmap) {
  __shared__ uint16_t lists[4 * kScbListWave];
  uint16_t* list = lists + (threadIdx.x >> 6) * kScbListWave;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n; base += stride) {
    const int64_t k = base + threadIdx.x;
    const bool valid = k < n;
    const int64_t i = valid ? perm[k] : 0;
    double E = 0.0;
    V3 din{0.0, 0.0, 1.0};
    ScbLane L;
    L.wl = 1.0;
    L.u = din;
    L.jlim = 0;
    bool can = false;
    if (valid) {
      E = ekin[i];
      din = V3{dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]};
      can = scb_lane_setup(v, E, din.x, din.y, din.z, L);
    }
    scb_walk<false>(v, L, 0, 0.0, list);
    if (!valid) continue;
    if (L.slow) {
      const unsigned long long slot = atomicAdd(qcount, 1ull);
      queue[slot] = i;
      cnt[k] = 0;
      continue;
    }
    const bool scatter = can && L.count > 0 && L.total > 0.0;
    cnt[k] = scatter ? L.count : 0;
    tot[k] = L.total;
    if (!scatter) {
      const int64_t o = idmap ? idmap[i] : i;
      oE[o] = E;
      oD[3 * o] = din.x;
      oD[3 * o + 1] = din.y;
      oD[3 * o + 2] = din.z;
    }
  }
}
__global__ void __launch_bounds__(256) k_scb_sample_pick(SCBView v, const double* __restrict__ ekin,
                                                         const double* __restrict__ dirs, int64_t n,
                                                         const int64_t* __restrict__ perm, uint64_t seed,
                                                         uint32_t stream, const int* __restrict__ cnt,
                                                         const double* __restrict__ tot, double4* __restrict__ sel,
                                                         const int64_t* __restrict__ idmap, int skip) {
  __shared__ uint16_t lists[4 * kScbListWave];
  uint16_t* list = lists + (threadIdx.x >> 6) * kScbListWave;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n; base += stride) {
    const int64_t k = base + threadIdx.x;
    const int c = k < n ? cnt[k] : 0;
    const int64_t i = c > 0 ? perm[k] : 0;
    double E = 0.0;
    V3 din{0.0, 0.0, 1.0};
    ScbLane L;
    L.wl = 1.0;
    L.u = din;
    L.jlim = 0;
    if (c > 0) {
      E = ekin[i];
      din = V3{dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]};
      scb_lane_setup(v, E, din.x, din.y, din.z, L);
    }
    Rng rng;
    rng.init(seed, stream, (uint64_t)(idmap && c > 0 ? idmap[i] : i));
    for (int q = 0; q < skip; ++q) (void)rng.gen();
    double target = 0.0;
    if (c > 1) target = tot[k] * rng.gen();
    scb_walk<true>(v, L, c, target, list);
    if (c <= 0) continue;
    sel[k] = L.found ? make_double4(L.sel_normal.x, L.sel_normal.y, L.sel_normal.z, L.sel_inv2d_r)
                     : make_double4(0.0, 0.0, 0.0, 0.0);
  }
}
__global__ void __launch_bounds__(256) k_scb_sample_scatter(SCBView v, const double* __restrict__ ekin,
                                                            const double* __restrict__ dirs, int64_t n,
                                                            const int64_t* __restrict__ perm, uint64_t seed,
                                                            uint32_t stream, double* __restrict__ oE,
                                                            double* __restrict__ oD, const int* __restrict__ cnt,
                                                            const double4* __restrict__ sel,
                                                            const int64_t* __restrict__ idmap, int skip) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
    const int c = cnt[k];
    if (c <= 0) continue;
    const int64_t i = perm[k];
    const double E = ekin[i];
    const V3 din{dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]};
    ScbLane L;
    scb_lane_setup(v, E, din.x, din.y, din.z, L);
    const int64_t oi = idmap ? idmap[i] : i;
    Rng rng;
    rng.init(seed, stream, (uint64_t)oi);
    for (int q = 0; q < skip; ++q) (void)rng.gen();
    if (c > 1) (void)rng.gen();  // the target draw of the selection
    const double4 s4 = sel[k];
    V3 o = din;
    if (s4.w != 0.0) o = gm_genscat(v, rng, V3{s4.x, s4.y, s4.z}, s4.w, L.wl, L.u);
    oE[oi] = E;
    oD[3 * oi] = o.x;
    oD[3 * oi + 1] = o.y;
    oD[3 * oi + 2] = o.z;
  }
}
__global__ void __launch_bounds__(256) k_scb_sample_slow(SCBView v, const double* __restrict__ ekin,
                                                         const double* __restrict__ dirs, uint64_t seed,
                                                         uint32_t stream, double* __restrict__ oE,
                                                         double* __restrict__ oD, const int64_t* __restrict__ queue,
                                                         const unsigned long long* __restrict__ qcount,
                                                         const int64_t* __restrict__ idmap, int skip) {
  __shared__ __align__(16) int lists[4][2][kScbWaveList];
  ScbWaveLists W{lists[threadIdx.x >> 6][0], lists[threadIdx.x >> 6][1], -1};
  const int64_t nq = (int64_t)*qcount;
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  const int group = scb_wave_group(v, ekin, dirs, queue, nq, nwaves);
  const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * group;
  if (group == 64) {
    uint16_t* list = reinterpret_cast<uint16_t*>(W.cand);
    for (int64_t q0 = first; q0 < nq; q0 += nwaves * 64) {
      const int64_t q = q0 + (threadIdx.x & 63);
      const int64_t i = queue[q < nq ? q : nq - 1];
      const double E = ekin[i];
      const V3 din{dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]};
      ScbLane L;
      L.wl = 1.0;
      L.u = V3{0.0, 0.0, 1.0};
      L.jlim = 0;
      const bool can = q < nq && scb_lane_setup(v, E, din.x, din.y, din.z, L);
      scb_walk<false, true>(v, L, 0, 0.0, list);
      const bool scatter = can && L.count > 0 && L.total > 0.0;
      const int64_t o = idmap ? idmap[i] : i;
      Rng rng;
      rng.init(seed, stream, (uint64_t)o);
      for (int s = 0; s < skip; ++s) (void)rng.gen();
      const int n = L.count;
      const double target = scatter && n > 1 ? L.total * rng.gen() : 0.0;
      if (!scatter) L.jlim = 0;
      scb_walk<true, true>(v, L, n, target, list);
      V3 d = din;
      if (scatter && L.found) d = gm_genscat(v, rng, L.sel_normal, L.sel_inv2d_r, L.wl, L.u);
      if (q < nq) {
        oE[o] = E;
        oD[3 * o] = d.x;
        oD[3 * o + 1] = d.y;
        oD[3 * o + 2] = d.z;
      }
    }
    return;
  }
  // (every lane of a wave has the same q; from the end, where the longest scans are)
  for (int64_t q1 = nq - first; q1 > 0; q1 -= nwaves * group)
  for (int64_t q0 = q1 > group ? q1 - group : 0, q = q0; q < q1; ++q) {
    if (q == q0) scb_wave_near(v, ekin, dirs, queue + q0, (int)(q1 - q0), W);
    const int64_t i = queue[q];
    const double E = ekin[i];
    const V3 din{dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]};
    ScbLane L;
    const bool can = scb_lane_setup(v, E, din.x, din.y, din.z, L);
    int nlist = 0;
    bool complete = false;
    scb_wave_walk<false>(v, L, 0, 0.0, W, nlist, complete);
    const int64_t o = idmap ? idmap[i] : i;  // output slot and Philox index
    V3 d = din;
    if (can && L.count > 0 && L.total > 0.0) {  // the same for every lane
      Rng rng;
      rng.init(seed, stream, (uint64_t)o);
      for (int s = 0; s < skip; ++s) (void)rng.gen();
      const int n = L.count;
      const double target = n > 1 ? L.total * rng.gen() : 0.0;
      scb_wave_walk<true>(v, L, n, target, W, nlist, complete);
      if (L.found) d = gm_genscat(v, rng, L.sel_normal, L.sel_inv2d_r, L.wl, L.u);
    }
    if ((threadIdx.x & 63) == 0) {
      oE[o] = E;
      oD[3 * o] = d.x;
      oD[3 * o + 1] = d.y;
      oD[3 * o + 2] = d.z;
    }
  }
}

static inline unsigned scb_grid(int64_t n) {
  int64_t g = (n + 255) / 256;
  const int64_t gmax = 256 * 64;
  if (g > gmax) g = gmax;
  if (g < 1) g = 1;
  return (unsigned)g;
}

// queue kernels: a wave per queued neutron, at most as many workgroups as the
// chip holds at once
static inline unsigned scb_slow_grid(int64_t n) { return (unsigned)(n < 4096 ? (n + 3) / 4 : 1024); }

// every workgroup of k_scb_keys adds its LDS counters to the global ones:
// eight neutrons per lane at least, and at most four workgroups per CU
static inline unsigned scb_keys_grid(int64_t n) {
  const int64_t g = (n + 2047) / 2048;
  return (unsigned)(g < 1 ? 1 : (g > 1024 ? 1024 : g));
}

// sorts the batch by scan length into w.perm and clears the queue counter
static void scb_order(const SCBView& v, const double* ekin, const double* dirs, int64_t n, const ScbWork& w,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_scb_clear, dim3(1), dim3(256), 0, st, w.hist, w.qcount);
  hipLaunchKernelGGL(k_scb_keys, dim3(scb_keys_grid(n)), dim3(256), 0, st, v, ekin, dirs, n, w.keys, w.hist);
  hipLaunchKernelGGL(k_scb_offsets, dim3(1), dim3(kScbBuckets), 0, st, w.hist, w.cursor);
  hipLaunchKernelGGL(k_scb_scatter, dim3(scb_grid((n + kScbScatterItems - 1) / kScbScatterItems)), dim3(256), 0, st,
                     w.keys, n, w.cursor, w.perm);
}

void launch_scb_xs(const SCBView& v, const double* ekin, const double* dirs, int64_t n, double* out,
                   const ScbWork& w, hipStream_t st) {
  if (n <= 0) return;
  scb_order(v, ekin, dirs, n, w, st);
  hipLaunchKernelGGL(k_scb_xs_main, dim3(scb_grid(n)), dim3(256), 0, st, v, ekin, dirs, n, w.perm, out, w.queue,
                     w.qcount);
  hipLaunchKernelGGL(k_scb_xs_slow, dim3(scb_slow_grid(n)), dim3(256), 0, st, v, ekin, dirs, out, w.queue, w.qcount);
}

// gathers the neutrons listed in q (count *qc, at most nmax) into compact
// arrays, with their original indices in idmap
__global__ void __launch_bounds__(256) k_scb_gather(const int64_t* __restrict__ q,
                                                    const unsigned long long* __restrict__ qc,
                                                    const double* __restrict__ ekin, const double* __restrict__ dirs,
                                                    double* __restrict__ cE, double* __restrict__ cD,
                                                    int64_t* __restrict__ idmap) {
  const int64_t m = (int64_t)*qc;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < m; t += stride) {
    const int64_t k = q[t];
    cE[t] = ekin[k];
    cD[3 * t] = dirs[3 * k];
    cD[3 * t + 1] = dirs[3 * k + 1];
    cD[3 * t + 2] = dirs[3 * k + 2];
    idmap[t] = k;
  }
}
void launch_scb_gather(const int64_t* q, const unsigned long long* qc, int64_t nmax, const double* ekin,
                       const double* dirs, double* cE, double* cD, int64_t* idmap, hipStream_t st) {
  if (nmax <= 0) return;
  hipLaunchKernelGGL(k_scb_gather, dim3(scb_grid(nmax)), dim3(256), 0, st, q, qc, ekin, dirs, cE, cD, idmap);
}

void launch_scb_sample(const SCBView& v, const double* ekin, const double* dirs, int64_t n, uint64_t seed,
                       uint32_t stream, double* oE, double* oD, const ScbWork& w, hipStream_t st,
                       const int64_t* idmap, int skip) {
  if (n <= 0) return;
  scb_order(v, ekin, dirs, n, w, st);
  hipLaunchKernelGGL(k_scb_sample_count, dim3(scb_grid(n)), dim3(256), 0, st, v, ekin, dirs, n, w.perm, oE, oD,
                     w.cnt, w.tot, w.queue, w.qcount, idmap);
  hipLaunchKernelGGL(k_scb_sample_pick, dim3(scb_grid(n)), dim3(256), 0, st, v, ekin, dirs, n, w.perm, seed, stream,
                     w.cnt, w.tot, w.sel, idmap, skip);
  hipLaunchKernelGGL(k_scb_sample_scatter, dim3(scb_grid(n)), dim3(256), 0, st, v, ekin, dirs, n, w.perm, seed,
                     stream, oE, oD, w.cnt, w.sel, idmap, skip);
  hipLaunchKernelGGL(k_scb_sample_slow, dim3(scb_slow_grid(n)), dim3(256), 0, st, v, ekin, dirs, seed, stream, oE, oD, w.queue,
                     w.qcount, idmap, skip);
}

}  // namespace ncamd

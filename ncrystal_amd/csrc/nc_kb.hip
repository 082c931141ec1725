// Box-envelope sampler of S(alpha,beta): the sampling kernels (device code in
// nc_kb.hh; the boxes' bounds in nc_kb_build.hip).
#include "nc_kernels.hh"

namespace ncamd {

// Sampling: one lane per neutron at a time, one proposal per lane per loop
// step, so that lanes whose neutron needs more proposals do not hold up the
// others.  A wave owns chunks of kKBChunk consecutive neutrons (chunk c of
// the wave w: c = w, w + nwaves, ...); lanes that finish a neutron take the
// next ones of the chunk in lane order, so that a step's loads and stores
// fall on neighbouring entries.  Neutrons outside the sampler's energy range
// or without an accepted proposal after maxtries go to the queue of the
// plain-sampler kernel, which restarts their Philox stream from draw 0.
// Mode 0: outputs (E', mu); mode 1: raw (alpha, beta).
constexpr int64_t kKBChunk = 1024;
template <int Mode>
__global__ void __launch_bounds__(256) k_kb_sample(SABView s, KBView k, const double* __restrict__ ekin, int64_t n,
                                                   int64_t total, uint64_t seed, uint32_t stream,
                                                   double* __restrict__ o1, double* __restrict__ o2,
                                                   unsigned long long* __restrict__ nerr,
                                                   int64_t* __restrict__ queue,
                                                   unsigned long long* __restrict__ qcount, int maxtries) {
  const int lane = (int)(threadIdx.x & 63);
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  // wave-uniform chunk state
  int64_t chunk = wave;
  int64_t next = chunk * kKBChunk;
  int64_t cend = next + kKBChunk < total ? next + kKBChunk : total;
  // lane state: the neutron, its energy (and E/kT), interval and the draw
  // counter of its Philox stream (key and stream are the kernel's)
  bool active = false;
  int64_t kk = 0;
  int tries = 0, iv = 0;
  uint32_t draw = 0;
  double E = 0.0, ediv = 0.0;
  while (true) {
    // idle lanes take the next neutrons of the chunk, moving on to the
    // wave's next chunk when this one is used up
    uint64_t idle = __ballot(!active);
    while (idle && next < total) {
      const int64_t take = (int64_t)__popcll(idle) < cend - next ? (int64_t)__popcll(idle) : cend - next;
      if (!active) {
        const int64_t rank = (int64_t)__popcll(idle & below);
        if (rank < take) {
          kk = next + rank;
          E = ekin[(total == n) ? kk : (kk % n)];
          iv = kb_interval(k, E);
          if (iv < 0) {
            queue[atomicAdd(qcount, 1ull)] = kk;
          } else {
            ediv = E * k.inv_kT;
            draw = 0;
            tries = 0;
            active = true;
          }
        }
      }
      next += take;
      if (next >= cend) {
        chunk += nwaves;
        next = chunk * kKBChunk;
        if (next > total) next = total;
        cend = next + kKBChunk < total ? next + kKBChunk : total;
      }
      idle = __ballot(!active);
    }
    if (!__ballot(active)) break;
    if (active) {
      Rng rng;
      rng.init(seed, stream, (uint64_t)kk);
      rng.c0 = draw;
      uint32_t r0, r1, r2, r3;
      rng.gen4(r0, r1, r2, r3);
      ++draw;
      double a, b;
      if (kb_propose(s, k, iv, ediv, r0, r1, r2, r3, a, b)) {
        if constexpr (Mode == 0) {
          double Ef, mu;
          if (sab_ab_to_emu(s, rng, E, a, b, Ef, mu)) { Ef = -1.0; mu = -999.0; atomicAdd(nerr, 1ull); }
          o1[kk] = Ef;
          o2[kk] = mu;
        } else {
          o1[kk] = a;
          o2[kk] = b;
        }
        active = false;
      } else if (++tries >= maxtries) {
        queue[atomicAdd(qcount, 1ull)] = kk;
        active = false;
      }
    }
  }
}

// raw (alpha, beta) of the plain sampler for the neutrons the envelope
// sampler handed back (from the first draw of their stream)
__global__ void k_kb_queue_ab(SABView s, const double* __restrict__ ekin, uint64_t seed, uint32_t stream,
                              double* __restrict__ oa, double* __restrict__ ob, const int64_t* __restrict__ queue,
                              const unsigned long long* __restrict__ qcount) {
  const int64_t nq = (int64_t)*qcount;
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < nq; j += (int64_t)gridDim.x * blockDim.x) {
    const int64_t kk = queue[j];
    Rng rng;
    rng.init(seed, stream, (uint64_t)kk);
    double a = -1.0, b = 0.0;
    if (sab_sample_ab(s, ekin[kk], rng, a, b)) { a = -1.0; b = 0.0; }
    oa[kk] = a;
    ob[kk] = b;
  }
}

static inline unsigned kb_grid(int64_t n) {
  int64_t g = (n + 255) / 256;
  const int64_t gmax = 256 * 64;
  if (g > gmax) g = gmax;
  if (g < 1) g = 1;
  return (unsigned)g;
}

// persistent grid: as many blocks as fit on the device at once (the chunks
// are handed out statically), fewer for small batches
template <int Mode>
static unsigned kb_sample_grid(int64_t total) {
  static int per_cu = 0, cus = 0;
  if (!per_cu) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
      cus = 256;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_kb_sample<Mode>, 256, 0) != hipSuccess || nb < 1) nb = 2;
    per_cu = nb;
  }
  const int64_t chunks = (total + kKBChunk - 1) / kKBChunk;
  int64_t g = (chunks + 3) / 4;  // 4 waves per block, one chunk per wave at least
  const int64_t gmax = (int64_t)per_cu * cus;
  if (g > gmax) g = gmax;
  if (g < 1) g = 1;
  return (unsigned)g;
}

void launch_kb_sample_iso(const SABView& s, const KBView& k, const double* ekin, int64_t n, int64_t repeat,
                          uint64_t seed, uint32_t stream, double* oE, double* oMu, unsigned long long* nerr,
                          int64_t* queue, unsigned long long* qcount, int maxtries, hipStream_t st) {
  const int64_t total = n * repeat;
  if (total <= 0) return;
  launch_zero_u64(qcount, st);
  hipLaunchKernelGGL(k_kb_sample<0>, dim3(kb_sample_grid<0>(total)), dim3(256), 0, st, s, k, ekin, n, total, seed,
                     stream, oE, oMu, nerr, queue, qcount, maxtries);
  launch_sab_queue(s, ekin, n, total, seed, stream, oE, oMu, nerr, queue, qcount, st);
}

void launch_kb_sample_ab(const SABView& s, const KBView& k, const double* ekin, int64_t n, uint64_t seed,
                         uint32_t stream, double* oa, double* ob, int64_t* queue, unsigned long long* qcount,
                         int maxtries, hipStream_t st) {
  if (n <= 0) return;
  launch_zero_u64(qcount, st);
  hipLaunchKernelGGL(k_kb_sample<1>, dim3(kb_sample_grid<1>(n)), dim3(256), 0, st, s, k, ekin, n, n, seed, stream, oa,
                     ob, (unsigned long long*)nullptr, queue, qcount, maxtries);
  hipLaunchKernelGGL(k_kb_queue_ab, dim3(kb_grid(n)), dim3(256), 0, st, s, ekin, seed, stream, oa, ob, queue,
                     qcount);
}

}  // namespace ncamd

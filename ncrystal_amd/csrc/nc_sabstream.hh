// S(alpha,beta) sampling (Alg1) of a list of neutrons by one wave, a try per
// lane and step.
//
// A neutron takes a random number of tries, and inside a try one of several
// ways to its alpha values.  One lane per neutron with the tries in a loop
// (sab_sample_iso) runs a wave at the pace of its unluckiest lane and pays for
// every way that any lane takes.  Here a lane that finishes takes the next
// neutron of the wave's range, and a step is the same for every lane: two
// numbers of the neutron's stream (one Philox block), a beta, the alpha of one
// or two table rows by one evaluation each whatever part of the row they fall
// in, the kinematic limits.  The first-bin rule's inner tries, the tries of the
// outgoing direction and the ultra-cold retries are states of the lane and take
// steps like the others.  The numbers a neutron draws, and the arithmetic on
// them, are those of sab_sample_iso (and rand_dir_given_mu), so the results are
// the same.
#pragma once
#include "nc_dev.hh"

namespace ncamd {

//
// What bounds it is the cache: a wave's lanes sit at unrelated places of the
// tables, so a load costs one access per lane whatever its width (up to 16
// bytes), and the accesses per neutron set the pace (the address unit is busy
// three quarters of the time).  So what is used together lies together (SabPt,
// SabHead, SabBin), a guide's two ends are one load, guides are fine enough that few
// searches need a probe, and the tables of one value per grid point are kept in
// LDS.  3e7 neutrons, 200 x 800 table: 4.68 ms with one lane per neutron, 3.88 ms
// streamed (44 accesses per neutron), 2.50 ms with this layout (26).

// The small tables (SABView::small), in LDS where they fit.  The constructor
// fills lds; the whole workgroup calls it.
NCHD bool sab_small_fits(const SABView& s) {
  return (int64_t)s.na + 2 * (int64_t)s.nb + 3 * (int64_t)s.ne <= kSabLds;
}
template <bool Lds>
struct SabSmall {
  const double *alpha, *beta, *scale, *egrid, *start;
  NCD SabSmall(const SABView& s, double* lds) {
    const double* p = s.small;
    if constexpr (Lds) {
      const int n = s.na + 2 * s.nb + 3 * s.ne;
      __syncthreads();  // the last user of lds
      for (int i = (int)threadIdx.x; i < n; i += (int)blockDim.x) lds[i] = p[i];
      __syncthreads();
      p = lds;
    }
    alpha = p;
    beta = p + s.na;
    scale = beta + s.nb;
    egrid = scale + s.nb;
    start = egrid + s.ne;
  }
};
// two neighbouring points (48 bytes) as three loads (the vector type keeps the
// compiler from splitting them)
typedef double sab_double2 __attribute__((ext_vector_type(2), aligned(8)));
NCD void load_points(const SabPt* __restrict__ p, SabPt& p0, SabPt& p1) {
  const sab_double2* q = reinterpret_cast<const sab_double2*>(p);
  const sab_double2 a = q[0], b = q[1], c = q[2];
  p0 = SabPt{a.x, a.y, b.x};
  p1 = SabPt{b.y, c.x, c.y};
}
NCD void load_bins(const SabBin* __restrict__ p, SabBin& p0, SabBin& p1) {
  const sab_double2* q = reinterpret_cast<const sab_double2*>(p);
  const sab_double2 a = q[0], b = q[1], c = q[2];
  p0 = SabBin{a.x, a.y, b.x};
  p1 = SabBin{b.y, c.x, c.y};
}

// one row's alpha at percentile rp, as the arguments of sample_loglin_fast
// (fb = fa selects its linear form)
struct Alg1Alpha {
  double a, fa, lfa, b, fb, lfb, r;
};
template <class Small>
NCD Alg1Alpha alg1_alpha_args(const SABView& s, const Small& small, int ie, int ibl, int ibeta, double rp) {
  const size_t at = (size_t)ie * s.nb + (ibeta - ibl);
  const double2* hp = reinterpret_cast<const double2*>(s.head + at);
  const double2 prob = hp[0], area = hp[1];
  const SabPt* __restrict__ pt = s.pt + (size_t)s.na * ibeta;
  const AInfo* __restrict__ info = s.sinfo + at;
  Alg1Alpha o;
  o.r = rp;
  if (rp > prob.x && rp <= prob.y) {
    // between the first and the last table point inside the limits, the usual
    // case; cumul there is area.x <= sel <= area.y
    const double p2 = dclamp((rp - prob.x) / (prob.y - prob.x), 0.0, 1.0);
    const double sel = area.x + p2 * (area.y - area.x);
    if (sel < area.y) {
      int lo, hi;
      guide_pair(s.row_guide + (size_t)ibeta * (kRowGuide + 1) + row_bucket(sel, small.scale[ibeta]), lo, hi);
      while (lo < hi) {  // upper_bound
        const int m = (lo + hi) >> 1;
        if (!(sel < pt[m].cumul)) lo = m + 1; else hi = m;
      }
      SabPt p0, p1;
      load_points(pt + lo - 1, p0, p1);
      o.a = small.alpha[lo - 1]; o.fa = p0.s; o.lfa = p0.logs;
      o.b = small.alpha[lo]; o.fb = p1.s; o.lfb = p1.logs;
      o.r = dclamp((sel - p0.cumul) / (p1.cumul - p0.cumul), kDblMin, 1.0);
    } else {
      o.a = o.b = small.alpha[info->b_idx];
      o.fa = o.fb = o.lfa = o.lfb = 0.0;
      o.r = 0.0;
    }
  } else if (rp <= prob.x) {
    o.a = info->f_alpha; o.fa = info->f_sval; o.lfa = info->f_logsval;
    if (prob.x == 2.0 || prob.x == 1.0) {
      o.b = info->b_alpha; o.fb = info->b_sval; o.lfb = info->b_logsval;
      if (prob.x == 2.0) o.fb = o.fa;
    } else {
      o.r = dclamp(rp / prob.x, kDblMin, 1.0);
      const SabPt q = pt[info->f_idx];
      o.b = small.alpha[info->f_idx]; o.fb = q.s; o.lfb = q.logs;
    }
  } else {
    o.r = dclamp((rp - prob.y) / (1.0 - prob.y), kDblMin, 1.0);
    const SabPt q = pt[info->b_idx];
    o.a = small.alpha[info->b_idx]; o.fa = q.s; o.lfa = q.logs;
    o.b = info->b_alpha; o.fb = info->b_sval; o.lfb = info->b_logsval;
  }
  return o;
}
NCD double alg1_alpha_eval(const Alg1Alpha& o) { return sample_loglin_fast(o.a, o.fa, o.b, o.fb, o.r, o.lfa, o.lfb); }

// PointwiseDist::percentileWithIndex (pw_percentile) on the packed points
NCD double bin_percentile(const SabBin* __restrict__ bin, const unsigned short* __restrict__ guide, int n, double p,
                          int& idx) {
  int i;
  if (p == 1.) {
    i = n - 1;
  } else {
    int lo, hi;
    guide_pair(guide + (int)(p * kCdfGuide), lo, hi);
    while (lo < hi) {  // lower_bound
      const int m = (lo + hi) >> 1;
      if (bin[m].cdf < p) lo = m + 1; else hi = m;
    }
    i = lo < n - 1 ? lo : n - 1;
    if (i < 1) i = 1;
  }
  SabBin p0, p1;
  load_bins(bin + i - 1, p0, p1);
  idx = i - 1;
  if (p == 1.) return p1.x;
  const double dx = p1.x - p0.x;
  const double c = (p - p0.cdf);
  const double a = p0.y;
  const double d = p1.y - a;
  double zdx;
  if (!a) {
    zdx = d > 0.0 ? sqrt((2.0 * c * dx) / d) : 0.5 * dx;
  } else {
    const double e = d * c / (dx * a * a);
    if (fabs(e) > 1e-7) zdx = (sqrt(1.0 + 2.0 * e) - 1.0) * dx * a / d;
    else zdx = (1 + 0.5 * e * (e - 1.0)) * c / a;
  }
  return dclamp(p0.x + zdx, p0.x, p1.x);
}
// the sampler of energy E >= egrid[0]: the first energy-grid point at or above
// E x margin, or the last one (sab_sample_ab steps there from E's own interval)
NCD int egrid_sampler(const SABView& s, const double* egrid, double E) {
  const double x = E * s.egrid_margin;
  if (!(x < egrid[s.ne - 1])) return s.ne - 1;
  const long long b = (long long)((unsigned long long)__double_as_longlong(x) >> s.eg_shift) - s.eg_base;
  unsigned long long v;
  __builtin_memcpy(&v, s.eg_bucket + b, 8);
  int lo = (int)(unsigned)v - 1, hi = (int)(v >> 32);  // (a point at the bucket's edge may equal x)
  lo = lo < 0 ? 0 : lo;
  while (lo < hi) {  // lower_bound
    const int m = (lo + hi) >> 1;
    if (egrid[m] < x) lo = m + 1; else hi = m;
  }
  return lo;
}

// A wave's share of a list of n among nw waves: every nw-th piece of 1 << shift
// places.  Pieces, because a list in the order of its energies has the tries of cold
// neutrons, or nothing but neutrons above Emax, side by side (1e7 neutrons of 1 meV
// to 1 eV, ordered: 660 us with one run of the list per wave, 590 in pieces).
// share_shift: 64 places fill a wave before the next one is begun; of long lists
// larger ones cost less (3e7 neutrons: 2.56 ms with 64, 2.52 with 256; one run each:
// 2.55).
NCD int share_shift(int64_t n) { return n > (1 << 24) ? 8 : 6; }
// Places are numbered from begin to end, at(i) is the one in the list.
struct SabShare {
  uint32_t nw;
  int shift;
  int64_t w, end;
  static constexpr int64_t begin = 0;
  NCD SabShare(int64_t n, unsigned wave, unsigned nwaves)
      : nw(nwaves), shift(share_shift(n)), w(__builtin_amdgcn_readfirstlane(wave)), end(0) {
    const int64_t pieces = (n + (1 << shift) - 1) >> shift;
    if (w >= pieces) return;
    end = ((pieces - w + nw - 1) / nw) << shift;
    if ((pieces - 1 - w) % nw == 0) end -= (pieces << shift) - n;  // the list's last piece
  }
  // (a wave's pieces are fewer than 2^32)
  NCD int64_t at(int64_t i) const {
    const uint64_t piece = (uint64_t)(uint32_t)(i >> shift) * nw + (uint64_t)w;
    return (int64_t)(piece << shift) | (i & ((1 << shift) - 1));
  }
};
// The same of a workgroup's own short list: one run, at least `fill` places
struct SabRun {
  int64_t begin, end;
  NCD SabRun(int n, int w, int nwaves, int fill) {
    const int wave = __builtin_amdgcn_readfirstlane(w);
    int per = (n + nwaves - 1) / nwaves;
    per = per < fill ? fill : per;
    begin = wave * per < n ? wave * per : n;
    end = begin + per < n ? begin + per : n;
  }
  NCD int64_t at(int64_t i) const { return i; }
};

// Samples the neutrons of a wave's share of a list, all lanes of the wave
// together.  take(i, k, E): the neutron at place i of the share (index k, which is
// also its Philox index; E below the table's Emax), or false if there is nothing to
// sample; put(k, rc, Ef, mu) for an isotropic outcome or an error, and with Dirs
// put_dir(k, Ef, ox, oy, oz) for the outcome about the incoming direction that
// dir(k, ix, iy, iz) gives.  after(last) runs, the whole wave together, when lanes have taken
// neutrons and once at the end.  skip: numbers of the stream already used.
template <bool Dirs, class Small, class Share, class Take, class After, class Put, class PutDir, class Dir>
NCD void sab_stream(const SABView& s, const Small& small, uint64_t seed, uint32_t stream, int skip,
                    const Share& share, const Take& take, const After& after, const Put& put,
                    const PutDir& put_dir, const Dir& dir) {
  // kTry: the next try (nv >= 0: from the sampler; -1: alpha = beta = 0; -2: no
  // sampler); kFirst: an inner try of the first-bin rule; kDir: a try of the
  // outgoing direction
  enum : int { kIdle, kTry, kFirst, kDir };
  const int lane = (int)(threadIdx.x & 63);
  const uint64_t below = lane ? ~0ull >> (64 - lane) : 0ull;
  const double beta0 = small.beta[0];
  int mode = kIdle;
  int64_t k = 0;
  double E = 0.0, sdiv = 0.0, firstbin = 0.0, aux = 0.0;  // aux: mu of kDir
  int isamp = 0, ibl = 0, nv = 0, it = 0, iii = 0, loop = 0;
  bool ultra = false;
  // the neutron's stream: index of its next number; the last block made (its
  // number and halves), whose second half is kept while the index is odd
  int64_t next = share.begin;
  uint32_t drawn = 0, blk = 0;
  uint64_t h0 = 0, h1 = 0;
  const auto block = [&](uint32_t b) {
    Rng g;
    g.init(seed, stream, (uint64_t)k);
    g.c0 = b;
    uint32_t w0, w1, w2, w3;
    g.gen4(w0, w1, w2, w3);
    h0 = ((uint64_t)w1 << 32) | w0;
    h1 = ((uint64_t)w3 << 32) | w2;
    blk = b;
  };
  // one number outside the pairs of a step (rare)
  const auto single = [&]() {
    uint64_t x = h1;
    if (!(drawn & 1)) {
      if (blk != drawn >> 1) block(drawn >> 1);
      x = h0;
    }
    ++drawn;
    return Rng::to01(x);
  };
  while (true) {
    uint64_t idle = __ballot(mode == kIdle);
    while (idle && next < share.end) {
      const int64_t room = share.end - next;
      const int cnt = room < (int64_t)__popcll(idle) ? (int)room : __popcll(idle);
      if (mode == kIdle) {
        const int rank = __popcll(idle & below);
        if (rank < cnt && take(next + rank, k, E)) {
          ultra = E < small.egrid[0];
          isamp = ultra ? 0 : egrid_sampler(s, small.egrid, E);
          sdiv = (ultra ? small.egrid[0] : E) / s.kT;
          firstbin = small.start[2 * isamp];
          const long long hdr = __double_as_longlong(small.start[2 * isamp + 1]);
          ibl = (int)(unsigned)hdr;
          nv = (int)(hdr >> 32);
          it = loop = 0;
          drawn = (uint32_t)skip;
          blk = ~0u;
          if (skip & 1) block((uint32_t)skip >> 1);
          mode = kTry;
        }
      }
      next += cnt;
      after(false);
      idle = __ballot(mode == kIdle);
    }
    if (!__ballot(mode != kIdle)) break;
    if (mode == kIdle) continue;
    double u0 = 0.0, u1 = 0.0;
    if (nv >= 0 || mode != kTry) {
      const uint64_t kept = h1;
      const uint32_t nb = (drawn + 1u) >> 1;
      if (blk != nb) block(nb);
      const bool odd = drawn & 1u;
      u0 = Rng::to01(odd ? kept : h0);
      u1 = Rng::to01(odd ? h0 : h1);
    }
    if constexpr (Dirs) {
      if (mode == kDir) {  // rand_dir_given_mu, one try
        drawn += 2;
        double ix, iy, iz;
        dir(k, ix, iy, iz);
        const double x0 = 2.0 * u0 - 1.0;
        const double x1 = 2.0 * u1 - 1.0;
        const double sq = x0 * x0 + x1 * x1;
        if (sq < 1.0) {
          const double m2 = ix * ix + iy * iy + iz * iz;
          const double invm = (fabs(m2 - 1.0) < 1e-14 ? 1.0 : 1.0 / sqrt(m2));
          double v0 = ix * invm, v1 = iy * invm, v2 = iz * invm;
          const double t = 2.0 * sqrt(1.0 - sq);
          const double a0 = x0 * t, a1 = x1 * t, a2 = 1.0 - 2.0 * sq;
          double t0 = a1 * v2 - a2 * v1, t1 = a2 * v0 - a0 * v2, t2 = a0 * v1 - a1 * v0;
          const double tm2 = t0 * t0 + t1 * t1 + t2 * t2;
          if (!(tm2 < 0.001)) {
            v0 *= aux; v1 *= aux; v2 *= aux;
            const double f = sqrt((1 - aux * aux) / tm2);
            t0 *= f; t1 *= f; t2 *= f;
            put_dir(k, E, v0 + t0, v1 + t1, v2 + t2);  // E: the outgoing energy by now
            mode = kIdle;
          }
        }
        continue;
      }
    }
    int rc = kOK;
    bool ok = false;
    double alpha = 0.0, beta = 0.0;
    if (nv < 0) {
      if (nv == -2) rc = kErrBadSampler;
      else ok = true;
    } else {
      const SabBin* __restrict__ bin = s.bin + (size_t)isamp * (s.nb + 1);
      bool rows = false;
      int row = ibl;
      if (mode == kTry) {
        int ibs;
        beta = bin_percentile(bin, s.cdf_guide + (size_t)isamp * (kCdfGuide + 1), nv, u0, ibs);
        ++drawn;
        if (ibs == 0 && firstbin <= 0.0) {
          if (bin[1].x < -sdiv) {
            ++it;
          } else {
            mode = kFirst;
            iii = 0;
          }
        } else if (beta <= dmax(-sdiv, beta0)) {
          ++it;
        } else {
          ++drawn;
          if (ibs < 1) {
            ++it;
          } else {
            rows = true;
            row = ibl + ibs - 1;
          }
        }
      } else {
        const double b1 = bin[1].x;
        const double db = b1 - firstbin;
        beta = dmax(firstbin, firstbin + db * u0);
        ++drawn;
        if (beta < -sdiv) {
          ++it;
          mode = kTry;
        } else {
          ++drawn;
          rows = true;
        }
      }
      if (rows) {
        const Alg1Alpha lo = alg1_alpha_args(s, small, isamp, ibl, row, u1);
        // (the first-bin rule takes one row; the other evaluation is then unused)
        const Alg1Alpha hi = mode == kTry ? alg1_alpha_args(s, small, isamp, ibl, row + 1, u1) : lo;
        const double al = alg1_alpha_eval(lo), ah = alg1_alpha_eval(hi);
        alpha = al;
        if (mode == kTry) {
          const double bl = small.beta[row], bh = small.beta[row + 1];
          alpha = al + (ah - al) * (beta - bl) / (bh - bl);
        }
        Lims l = alpha_limits(mode == kTry ? sdiv : -firstbin, beta);
        ok = in_interval(l.lo, l.hi, alpha);
        if (mode == kTry) {
          if (!ok) ++it;
        } else if (ok || iii == 29) {
          if (!ok) alpha = 0.5 * (l.lo + l.hi);
          l = alpha_limits(sdiv, beta);
          ok = in_interval(l.lo, l.hi, alpha);
          if (!ok) ++it;
          mode = kTry;
        } else {
          ++iii;
        }
      }
      if (it >= 100) rc = kErrAlg1Loop;
    }
    if (ok && ultra) {  // sampled at egrid[0] for a colder neutron
      const double ediv = E / s.kT;
      if (beta < -ediv) {
        ok = false;
        it = 0;
        if (++loop >= 100) rc = kErrSamplerLoop;
      } else {
        const Lims l = alpha_limits(ediv, beta);
        if (!in_interval(l.lo, l.hi, alpha)) alpha = l.lo + single() * (l.hi - l.lo);
      }
    }
    double Ef = 0.0, mu = 0.0;
    if (ok) {  // sab_ab_to_emu
      const double dE = beta * s.kT;
      if (mu_iso_at_beta(beta, E / s.kT)) {
        mu = single() * 2.0 - 1.0;
      } else {
        const double ef = E + dE;
        const double denom = 2.0 * sqrt(E * ef);
        if (!denom) {
          rc = kErrKinematics;
        } else {
          StableSum sm;
          sm.add(E); sm.add(ef); sm.add(-alpha * s.kT);
          mu = dclamp(sm.sum() / denom, -1.0, 1.0);
        }
      }
      Ef = dmax(0.0, E + dE);
    }
    if (ok || rc) {
      if (Dirs && !rc) {
        E = Ef;
        aux = mu;
        mode = kDir;
      } else {
        put(k, rc, Ef, mu);
        mode = kIdle;
      }
    }
  }
  after(true);
}

}  // namespace ncamd

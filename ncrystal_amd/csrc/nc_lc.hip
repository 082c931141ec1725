// Layered-crystal Bragg scattering by the reference models of
// ncrystal_core/src/extd_utils/NCLCRefModels.cc: a mosaic single crystal
// (the SCBragg kernels) averaged over rotations of the crystal around the
// layer axis.  A rotation of the crystal by phi is a rotation of the neutron
// by -phi in the crystal's frame, so each neutron is expanded into N
// rotated directions (one lane per neutron and rotation), the SCBragg
// kernels evaluate all of them in one launch, and small per-neutron kernels
// average (cross sections) or pick one rotation by its cross section and
// rotate the scattered direction back (sampling).
#include "nc_kernels.hh"
#include "nc_dev.hh"
#include "nc_scb.hh"

namespace ncamd {
namespace {

// Rodrigues' rotation of the unit vector v by (c, s) = (cos phi, sin phi)
// around the unit axis a, in the operation order of
// ncrystal_core/include/NCrystal/internal/utils/NCRotMatrix.hh:172-184:
// v c + (a x v) s + a ((a . v)(1 - c))
NCD void lc_rotate(const LCView& L, double vx, double vy, double vz, double c, double s, double& ox, double& oy,
                   double& oz) {
  const double cx = L.ay * vz - L.az * vy, cy = L.az * vx - L.ax * vz, cz = L.ax * vy - L.ay * vx;
  const double f = (L.ax * vx + L.ay * vy + L.az * vz) * (1.0 - c);
  ox = vx * c + cx * s + L.ax * f;
  oy = vy * c + cy * s + L.ay * f;
  oz = vz * c + cz * s + L.az * f;
}

// lane t = i * N + j: neutron i rotated by rotation j, from the fixed table
// cs (equally spaced angles) or, with cs null, by a uniform random angle
// (Philox draw t of (seed, stream)), whose (cos, sin) goes to ocs
__global__ void __launch_bounds__(256) k_lc_expand(const double* __restrict__ ekin, const double* __restrict__ dirs,
                                                   int64_t n, int N, LCView L, const double2* __restrict__ cs,
                                                   uint64_t seed, uint32_t stream, double* __restrict__ oE,
                                                   double* __restrict__ oD, double2* __restrict__ ocs) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * (int64_t)N) return;
  const int64_t i = t / N;
  const int j = (int)(t - i * N);
  double c, s;
  if (cs) {
    const double2 v = cs[j];
    c = v.x;
    s = v.y;
  } else {
    Rng r;
    r.init(seed, stream, (uint64_t)t);
    sincos(k2Pi * r.gen() - kPi, &s, &c);
    ocs[t] = make_double2(c, s);
  }
  double ux = dirs[3 * i], uy = dirs[3 * i + 1], uz = dirs[3 * i + 2];
  const double inv = 1.0 / sqrt(ux * ux + uy * uy + uz * uz);
  ux *= inv; uy *= inv; uz *= inv;
  double rx, ry, rz;
  lc_rotate(L, ux, uy, uz, c, s, rx, ry, rz);
  oE[t] = ekin[i];
  oD[3 * t] = rx;
  oD[3 * t + 1] = ry;
  oD[3 * t + 2] = rz;
}

// mean of each neutron's N cross sections, compensated (Neumaier) sum as the
// reference's StableSum
__global__ void __launch_bounds__(256) k_lc_mean(const double* __restrict__ xs, int64_t n, int N,
                                                 double* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double sum = 0.0, comp = 0.0;
  for (int j = 0; j < N; ++j) {
    const double x = xs[i * N + j];
    const double t = sum + x;
    comp += fabs(sum) >= fabs(x) ? (sum - t) + x : (x - t) + sum;
    sum = t;
  }
  out[i] = (sum + comp) / (double)N;
}

// one rotation per neutron with probability proportional to its cross
// section (running sums and the first one above u x total, as
// pickRandIdxByWeight); neutrons whose rotations all have zero cross section
// get sel = -1.  The chosen rotated direction goes to sD, the energy to sE.
__global__ void __launch_bounds__(256) k_lc_pick(const double* __restrict__ xs, const double* __restrict__ rE,
                                                 const double* __restrict__ rD, int64_t n, int N, uint64_t seed,
                                                 uint32_t stream, double* __restrict__ sE, double* __restrict__ sD,
                                                 int* __restrict__ sel) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double tot = 0.0;
  for (int j = 0; j < N; ++j) tot += xs[i * N + j];
  int pick = -1;
  if (tot > 0.0) {
    Rng r;
    r.init(seed, stream, (uint64_t)i);
    const double u = r.gen() * tot;
    double run = 0.0;
    pick = N - 1;
    for (int j = 0; j < N; ++j) {
      run += xs[i * N + j];
      if (u < run && xs[i * N + j] > 0.0) { pick = j; break; }
    }
    while (pick > 0 && !(xs[i * N + pick] > 0.0)) --pick;  // u == tot: the last rotation that contributes
  }
  const int64_t t = i * N + (pick < 0 ? 0 : pick);
  sel[i] = pick;
  sE[i] = rE[t];
  sD[3 * i] = rD[3 * t];
  sD[3 * i + 1] = rD[3 * t + 1];
  sD[3 * i + 2] = rD[3 * t + 2];
}

// scattered directions rotated back by the chosen rotation (reverse sense);
// neutrons without a rotation leave unchanged
__global__ void __launch_bounds__(256) k_lc_unrotate(const double* __restrict__ scD, const int* __restrict__ sel,
                                                     const double2* __restrict__ cs, const double* __restrict__ ekin,
                                                     const double* __restrict__ dirs, int64_t n, int N, LCView L,
                                                     double* __restrict__ oE, double* __restrict__ oD) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int j = sel[i];
  oE[i] = ekin[i];
  if (j < 0) {
    oD[3 * i] = dirs[3 * i];
    oD[3 * i + 1] = dirs[3 * i + 1];
    oD[3 * i + 2] = dirs[3 * i + 2];
    return;
  }
  const double2 v = cs[i * N + j];
  double rx, ry, rz;
  lc_rotate(L, scD[3 * i], scD[3 * i + 1], scD[3 * i + 2], v.x, -v.y, rx, ry, rz);
  oD[3 * i] = rx;
  oD[3 * i + 1] = ry;
  oD[3 * i + 2] = rz;
}

unsigned lc_blocks(int64_t n) { return (unsigned)((n + 255) / 256); }

// ---- lcmode=0: ncrystal_core/src/extd_utils/NCLCUtils.cc

// values on the 2^-40 grid of the model's cache keys (:45-52)
NCD double lc_discr(double x) {
  return (double)(uint64_t)(x * 1099511627776.0 + 0.5) * (1.0 / 1099511627776.0);
}

// GaussMos::calcRawCrossSectionValue after InteractionPars::set
// (NCGaussMos.hh:204-214, NCGaussMos.cc:252-280): Q times the
// Gaussian-on-sphere circle integral, Q = wl^3 / (sin cos theta_Bragg) x
// fsq / 2.  The part that depends on the plane set and the wavelength alone;
// Q < 0 marks the value kept in `fixed` for every angle.
struct LC0Raw {
  double sinpt, cospt, Q, fixed;
};
NCD LC0Raw lc0_raw_setup(double wl, double inv2d, double fsq) {
  LC0Raw r;
  const double w = gm_round(wl), i2 = gm_round(inv2d);
  r.sinpt = w * i2;
  r.cospt = sqrt(1 - r.sinpt * r.sinpt);
  const double tmp2 = r.cospt * r.sinpt;
  const double Qprime = tmp2 > 0 ? (w * w * w) / tmp2 : ((r.sinpt > 0.5 && fsq != 0.0) ? -2.0 : 0.0);
  r.fixed = Qprime != 0.0 ? __builtin_huge_val() : 0.0;
  r.Q = Qprime > 0.0 ? Qprime * (fsq * 0.5) : -1.0;
  return r;
}
// cos(phi) for phi in [0, pi]: phi = j pi/2 + r + rl with |r| <= pi/4 and the
// Taylor series of sine and cosine at r, the cosine's 1 - r^2/2 + .. with the
// rounding of its first two terms added back (the usual compensated tail) and rl's
// share.  Half the instructions of the general cosine, whose argument may be of any
// size.
NCD double lc0_cos(double phi) {
  const double j = rint(phi * 0.63661977236758134308);
  const double t = fma(-j, kPiHalf, phi);  // exact
  const double lo = j * 6.123233995736766036e-17;
  const double r = t - lo;
  const double rl = (t - r) - lo;
  const double z = r * r;
  double c = -1.5619206968586226e-16, s = 2.8114572543455206e-15;  // -1/18!, 1/17!
  c = fma(z, c, 4.7794773323873853e-14); s = fma(z, s, -7.6471637318198164e-13);
  c = fma(z, c, -1.1470745597729725e-11); s = fma(z, s, 1.6059043836821615e-10);
  c = fma(z, c, 2.0876756987868099e-09); s = fma(z, s, -2.5052108385441719e-08);
  c = fma(z, c, -2.7557319223985891e-07); s = fma(z, s, 2.7557319223985893e-06);
  c = fma(z, c, 2.4801587301587302e-05); s = fma(z, s, -1.9841269841269841e-04);
  c = fma(z, c, -1.3888888888888889e-03); s = fma(z, s, 8.3333333333333333e-03);
  c = fma(z, c, 4.1666666666666664e-02); s = fma(z, s, -1.6666666666666666e-01);
  const double h = 0.5 * z, w = 1.0 - h;
  const double vc = w + (((1.0 - w) - h) + fma(z * z, c, -r * rl));
  const double vs = r + fma(z * r, s, rl * w);
  return j == 1.0 ? -vs : (j == 0.0 ? vc : -vc);
}
// value at cos(gamma) = cosg; Slow false: sets `slow` (and returns 0) where
// the circle integral is outside the spline's validity
template <bool Slow>
NCD double lc0_raw(const SCBView& v, const LC0Raw& r, double cosg, bool& slow) {
  if (!(r.Q >= 0.0)) return r.fixed;
  const double cc = dclamp(cosg, -1.0, 1.0);
  const double sc = sqrt(1.0 - cc * cc);
  double val;
  if (!gos_circle_fast_ok(v, cc, sc, r.sinpt, r.cospt, val)) {
    if constexpr (Slow) {
      val = gos_circle_slow(v, cc, sc, r.sinpt, r.cospt);
    } else {
      if (!(r.sinpt * cc + r.cospt * sc <= v.cta)) slow = true;  // gos_circle_slow is 0 outside the cone
      val = 0.0;
    }
  }
  return r.Q * val;
}

// a rotation range (ROI) of a plane set: kind 0 normal along the axis, 1
// neutron along the axis, 2 the range [r0, r1] of phi, over which
// cos(gamma) = k1 cos(phi) + k0 (kinds 0 and 1: cos(gamma) = k0)
struct LC0Roi {
  int kind;
  double k1, k0, r0, r1;
};

// the ROI of one side (sg = +-1) of plane set ps for a neutron (wavelength
// wl, |cos| and sin of its angle to the axis c3, s3), false if there is none
// (LCROIFinder::findROIs, NCLCUtils.cc:184-303); the set is known to reach it
NCD bool lc0_side(const LC0View& L, const LC0Set& ps, double c2, double s2, double c3, double s3, double sg,
                  double& p1, double& p2) {
  const double c2low = c2 * L.cta - s2 * L.sta;
  const double c2high = s2 < L.sta ? 1.0 : c2 * L.cta + s2 * L.sta;
  const double b = 1.0 / (ps.s1 * s3);
  const double mab = -(ps.c1 * c3) * b;
  p1 = dclamp(mab + sg * (c2low * b), -1.0, 1.0);
  p2 = dclamp(mab + sg * (c2high * b), -1.0, 1.0);
  return fabs(p1 - p2) > 1e-10;
}
// ROIs of a plane set: bit 0 the normal side, bit 1 the anti-normal side
NCD unsigned lc0_sides(const LC0View& L, const LC0Set& ps, double wl, double c3, double s3) {
  const double c2 = ps.inv2d * wl;
  const double c23 = c3 * c2;
  const double s2 = sqrt(1.0 - c2 * c2);
  const double s23 = s3 * s2;
  const double lo = c23 - s23, hi = c23 + s23;
  if (dmax(lo, ps.c1plus) > dmin(hi, ps.c1minus)) return 0u;
  const bool anti = dmax(lo, -ps.c1minus) <= dmin(hi, -ps.c1plus);
  if (ps.s1 == 0.0 || fabs(s3) < 1e-10) return anti ? 3u : 1u;
  double p1, p2;
  unsigned m = lc0_side(L, ps, c2, s2, c3, s3, 1.0, p1, p2) ? 1u : 0u;
  if (anti && lc0_side(L, ps, c2, s2, c3, s3, -1.0, p1, p2)) m |= 2u;
  return m;
}
NCD LC0Roi lc0_roi(const LC0View& L, const LC0Set& ps, double wl, double c3, double s3, double sg) {
  LC0Roi roi{2, 0.0, 0.0, 0.0, 0.0};
  if (ps.s1 == 0.0) {
    roi.kind = 0;
    roi.k0 = sg * c3;
  } else if (fabs(s3) < 1e-10) {
    roi.kind = 1;
    roi.k0 = (ps.c1 * c3) * sg;
  } else {
    const double c2 = ps.inv2d * wl;
    const double s2 = sqrt(1.0 - c2 * c2);
    double p1, p2;
    lc0_side(L, ps, c2, s2, c3, s3, sg, p1, p2);
    roi.k1 = ps.s1 * s3 * sg;
    roi.k0 = ps.c1 * sg * c3;
    roi.r0 = acos(dmax(p1, p2));
    roi.r1 = acos(dmin(p1, p2));
  }
  return roi;
}

// Romberg integration of NCRomberg.cc:58-140 (17 points, halvings up to
// level 15, accept |R_k - R_(k-1)| <= acc |R_k|) of the cross section over
// crystallite rotations phi.  The 17 points are summed into the groups of the
// first five levels (ends, midpoint, quarters, eighths, sixteenths).
struct LC0Sums {
  double s_end = 0.0, s_mid = 0.0, s_q = 0.0, s_e = 0.0, s_s = 0.0;
  NCD void add(int i, double f) {
    if (i == 0 || i == 16) s_end += f;
    else if (i == 8) s_mid += f;
    else if (i == 4 || i == 12) s_q += f;
    else if ((i & 1) == 0) s_e += f;
    else s_s += f;
  }
};
// rows 0-4 of the tableau from the point sums (r: row 4); true if accepted
NCD bool lc0_rows4(const LC0Sums& p, double len, double acc, double* r) {
  double h = len;
  h *= 0.5;
  const double r00 = p.s_end * h;
  const double r10 = h * p.s_mid + 0.5 * r00;
  const double r11 = (4.0 * r10 - r00) / 3.0;
  h *= 0.5;
  const double r20 = h * p.s_q + 0.5 * r10;
  const double r21 = (4.0 * r20 - r10) / 3.0;
  const double r22 = (16.0 * r21 - r11) / 15.0;
  h *= 0.5;
  const double r30 = h * p.s_e + 0.5 * r20;
  const double r31 = (4.0 * r30 - r20) / 3.0;
  const double r32 = (16.0 * r31 - r21) / 15.0;
  const double r33 = (64.0 * r32 - r22) / 63.0;
  h *= 0.5;
  r[0] = h * p.s_s + 0.5 * r30;
  r[1] = (4.0 * r[0] - r30) / 3.0;
  r[2] = (16.0 * r[1] - r31) / 15.0;
  r[3] = (64.0 * r[2] - r32) / 63.0;
  r[4] = (256.0 * r[3] - r33) / 255.0;
  return fabs(r[4] - r33) <= acc * fabs(r[4]);
}
// row 5 from row 4 (in place) and the sum c of its 16 new points
NCD bool lc0_row5(double c, double len, double acc, double* r) {
  const double h = len * 0.03125;
  const double p0 = r[0], p1 = r[1], p2 = r[2], p3 = r[3], p4 = r[4];
  r[0] = h * c + 0.5 * p0;
  r[1] = (4.0 * r[0] - p0) / 3.0;
  r[2] = (16.0 * r[1] - p1) / 15.0;
  r[3] = (64.0 * r[2] - p2) / 63.0;
  r[4] = (256.0 * r[3] - p3) / 255.0;
  r[5] = (1024.0 * r[4] - p4) / 1023.0;
  return fabs(r[5] - p4) <= acc * fabs(r[5]);
}
// row 6 from row 5; x: its last entry
NCD bool lc0_row6(double c, double len, double acc, const double* p, double& x) {
  const double h = len * 0.015625;
  const double q0 = h * c + 0.5 * p[0];
  const double q1 = (4.0 * q0 - p[0]) / 3.0;
  const double q2 = (16.0 * q1 - p[1]) / 15.0;
  const double q3 = (64.0 * q2 - p[2]) / 63.0;
  const double q4 = (256.0 * q3 - p[3]) / 255.0;
  const double q5 = (1024.0 * q4 - p[4]) / 1023.0;
  x = (4096.0 * q5 - p[5]) / 4095.0;
  return fabs(x - p[5]) <= acc * fabs(x);
}
// row i >= 6 in place
NCD bool lc0_row(int i, double c, double h, double acc, double* r) {
  double old = r[0];
  r[0] = h * c + 0.5 * old;
  double nk = 1.0;
#pragma nounroll
  for (int j = 0; j < i; ++j) {
    nk *= 4.0;
    const double nx = (nk * r[j] - old) / (nk - 1.0);
    if (j + 1 < i) old = r[j + 1];
    else return (r[j + 1] = nx, fabs(nx - old) <= acc * fabs(nx));
    r[j + 1] = nx;
  }
  return false;
}

// discretised wavelength and |cos| to the layer axis (:332-344)
NCD void lc0_neutron(const LC0View& L, double E, double& ux, double& uy, double& uz, double& wl, double& c3raw,
                     double& c3, double& s3) {
  const double inv = 1.0 / sqrt(ux * ux + uy * uy + uz * uz);
  ux *= inv; uy *= inv; uz *= inv;
  wl = lc_discr(sqrt(kWl2Ekin / E));
  c3raw = L.ax * ux + L.ay * uy + L.az * uz;
  c3 = dmin(lc_discr(fabs(c3raw)), 1.0);
  s3 = sqrt(fabs(1.0 - c3 * c3));
}

// Layered-crystal kernel: a workgroup takes 4 to 256 neutrons and works on all
// their rotation ranges together.
//
// A neutron has between none and twice the number of plane sets of ranges
// (pyrolytic graphite, 0.5-7 Aa: none for 45 % of the neutrons, 127 for some,
// 14 on average), and each costs an integral of 17 to 65 points.  One lane per
// neutron ran at the pace of the longest lane of its wave, with the nested
// circle integral in line (256 registers, one wave per SIMD, 480 B of scratch
// per lane): 22 ms for the cross sections of 131072 neutrons and 30 ms for
// scattering, against 1.05 and 1.15 ms now, bound by the FP64 arithmetic of the
// points (about 210 vector instructions each).  Here
//  - every lane first looks at one neutron and its first plane sets; neutrons
//    without a range are done (k_lc0), and where the first sets were all the
//    sets in reach, the ranges are listed;
//  - else the ranges are found with one lane per (neutron, 32 plane sets) and
//    listed in the neutrons' order (bit masks and a prefix sum);
//  - one lane per range integrates up to row 5 of the Romberg tableau (33
//    points), where 90 to 97 % are accepted; row 6 of the others takes half a
//    wave each, a point per lane;
//  - the few left, and the ranges with a point outside the spline's validity
//    (backscattering within the mosaic spread: 3 % of the ranges, nearly all
//    their points, each an integral of its own), are listed again and spread
//    over the workgroup, four points per lane, up to the last row;
//  - the values are added per neutron in the order of the list, so that
//    every sum is the one a single lane would form.
// Neutrons with more ranges than the lists hold together, and more plane sets
// than a round's masks, are worked on in rounds; only with more than kLc0Sets
// plane sets does sampling run them again to find its range.
//
// The first step is what batches with few or no ranges need, beyond the
// wavelengths of all sets but one or two: without it 1e6 neutrons of 8 to 20 Aa
// took 142 us (cross sections) and 349 us (scattering), with it 18 and 19 (one
// lane per neutron: 51 and 52), of 4.3 to 6 Aa 175 and 589 us, now 63 and 156
// (70 and 198).  Where such a batch is small (1e3 to 1e5 neutrons, 4.3 Aa and
// beyond), the steps' latencies leave the cross sections at 7 to 43 us, 1.2 to
// 1.8 times those of one lane per neutron.
constexpr int kLc0Threads = 256;
constexpr int kLc0Neutrons = 128;                 // neutrons worked on together at most
constexpr int kLc0Words = 8;                      // mask words (32 plane sets each) per neutron and round
constexpr int kLc0Sets = 32 * kLc0Words;
constexpr int kLc0Units = 512;                    // mask words of those neutrons at most
constexpr int kLc0List = 1536;
constexpr int kLc0Redo = 28;                      // listed ranges redone together: 28 x 9 groups of 4 points
constexpr int kLc0RedoPts = 33;

struct Lc0Lds {
  uint64_t mask[kLc0Units];
  double wl[kLc0Neutrons], c3[kLc0Neutrons], s3[kLc0Neutrons];
  double val[kLc0List];
  double sv[kLc0Redo * (kLc0RedoPts + 16)];  // points of the ranges redone, then their rows (the rotation step takes all)
  int off[kLc0Units + 1];
  uint16_t item[kLc0List];   // neutron << 9 | set of the round << 1 | side
  uint16_t redo[kLc0List];   // ranges not done by their one lane: not accepted at row 6 from the front, slow from the back
  int nredo, nslow, nact, nwork, nlisted, more;
  uint8_t act[kLc0Redo];
  uint8_t work[kLc0Threads];   // neutrons of the workgroup that may have ranges
  uint8_t turn[kLc0Neutrons];  // neutrons of the rotation step
};
static_assert(kLc0Redo * (kLc0RedoPts + 16) >= 10 * kLc0Neutrons && kLc0List >= 8 * kLc0Neutrons, "rotation step");
static_assert(kLc0Neutrons <= 128 && 2 * kLc0Sets <= 512 && kLc0Words <= kLc0Units, "bits of item");

// integrates the ranges listed in S.item[0..n) (plane sets k0 + .. of this
// round) into S.val; the whole workgroup calls it
NCD void lc0_values(const LC0View& L, const SCBView& v, Lc0Lds& S, int k0, int n) {
  const int tid = (int)threadIdx.x;
  if (tid == 0) { S.nredo = 0; S.nslow = 0; }
  __syncthreads();
  const int lane = tid & 63;
  for (int p0 = 0; p0 < n; p0 += kLc0Threads) {
    const int p = p0 + tid;
    bool slow = false, need6 = false;
    double x = 0.0, len = 0.0, r[6];
    LC0Roi roi{0, 0.0, 0.0, 0.0, 0.0};
    LC0Raw raw{0.0, 0.0, -1.0, 0.0};
    if (p < n) {
      const unsigned it = S.item[p];
      const int nu = (int)(it >> 9);
      const LC0Set ps = L.sets[k0 + (int)((it >> 1) & 255u)];
      const double wl = S.wl[nu];
      roi = lc0_roi(L, ps, wl, S.c3[nu], S.s3[nu], (it & 1u) ? -1.0 : 1.0);
      raw = lc0_raw_setup(wl, ps.inv2d, ps.fsq);
      if (roi.kind != 2) {
        x = lc0_raw<false>(v, raw, roi.k0, slow);
      } else {
        LC0Sums sm;
        len = roi.r1 - roi.r0;
        const double delta = len * 0.0625;
#pragma nounroll
        for (int i = 0; i < 17 && !slow; ++i)
          sm.add(i, lc0_raw<false>(v, raw, roi.k1 * lc0_cos(roi.r0 + delta * (double)i) + roi.k0, slow));
        bool done = lc0_rows4(sm, len, L.acc, r);
        x = r[4];
        if (!done && !slow) {
          const double hh = len * 0.0625, h = len * 0.03125;
          double c = 0.0;
#pragma nounroll
          for (int j = 0; j < 16 && !slow; ++j)
            c += lc0_raw<false>(v, raw, roi.k1 * lc0_cos(roi.r0 + h + hh * (double)j) + roi.k0, slow);
          done = lc0_row5(c, len, L.acc, r);
          x = r[5];
        }
        need6 = !done && !slow;
      }
    }
    // row 6 of the ranges of this wave that need it: two at a time, a point of
    // each per lane of a half
    uint64_t M = __ballot(need6);
    bool more = false;
    while (M) {
      const int l0 = __builtin_ctzll(M);
      M &= M - 1ull;
      const int l1 = M ? __builtin_ctzll(M) : l0;
      M &= M - 1ull;
      const int src = lane < 32 ? l0 : l1;
      const double k1 = __shfl(roi.k1, src, 64), kk0 = __shfl(roi.k0, src, 64), r0 = __shfl(roi.r0, src, 64),
                   ln = __shfl(len, src, 64);
      const LC0Raw rw{__shfl(raw.sinpt, src, 64), __shfl(raw.cospt, src, 64), __shfl(raw.Q, src, 64),
                      __shfl(raw.fixed, src, 64)};
      bool sl = false;
      const double hh = ln * 0.03125;
      double f = lc0_raw<false>(v, rw, k1 * lc0_cos(r0 + hh * 0.5 + hh * (double)(lane & 31)) + kk0, sl);
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) f += __shfl_xor(f, o, 64);
      const double c0 = __shfl(f, 0, 64), c1 = __shfl(f, 32, 64);
      const uint64_t B = __ballot(sl);
      if (lane == l0 || lane == l1) {
        slow = (lane == l0 ? (uint32_t)B : (uint32_t)(B >> 32)) != 0u;
        more = !lc0_row6(lane == l0 ? c0 : c1, len, L.acc, r, x);
      }
    }
    if (p < n) {
      if (roi.kind == 2) x *= 1.0 / kPi;
      if (slow) S.redo[kLc0List - 1 - atomicAdd(&S.nslow, 1)] = (uint16_t)p;
      else if (more) S.redo[atomicAdd(&S.nredo, 1)] = (uint16_t)p;
      else S.val[p] = x;
    }
  }
  __syncthreads();
  // the listed ranges from the start again, a few points per lane, the tableau
  // of range t kept by lane t
  // (the two kinds apart, so that lanes of a wave have alike work)
  const int nredo = S.nredo, nslow = S.nslow;
  for (int b0 = nredo > 0 ? 0 : kLc0List - nslow; b0 < kLc0List;) {
    const int end = b0 < nredo ? nredo : kLc0List;
    const int nr = end - b0 < kLc0Redo ? end - b0 : kLc0Redo;
    if (tid < nr) S.act[tid] = 1;
    bool first = true;
#pragma nounroll
    for (int i = 5; i < 16; ++i, first = false) {
      // rows 4 and 5 together (17 + 16 points), then the 2^(i-1) new points
      // of row i
      const int np = first ? kLc0RedoPts : 1 << (i - 1);
      double c = 0.0;
      LC0Sums sm;
      for (int j0 = 0; j0 < np; j0 += kLc0RedoPts) {
        const int m = np - j0 < kLc0RedoPts ? np - j0 : kLc0RedoPts;
        const int groups = (m + 3) >> 2;
        __syncthreads();
        for (int q = tid; q < nr * groups; q += kLc0Threads) {
          const int t = q / groups, ja = 4 * (q - t * groups), jb = ja + 4 < m ? ja + 4 : m;
          if (!S.act[t]) continue;
          const unsigned it = S.item[S.redo[b0 + t]];
          const int nu = (int)(it >> 9);
          const LC0Set ps = L.sets[k0 + (int)((it >> 1) & 255u)];
          const double wl = S.wl[nu];
          const LC0Roi roi = lc0_roi(L, ps, wl, S.c3[nu], S.s3[nu], (it & 1u) ? -1.0 : 1.0);
          const LC0Raw raw = lc0_raw_setup(wl, ps.inv2d, ps.fsq);
          const double len = roi.r1 - roi.r0;
          bool dummy = false;
#pragma nounroll
          for (int j = ja; j < jb; ++j) {
            double f = 0.0;
            if (roi.kind == 2 || j0 + j == 0) {
              double cg = roi.k0;
              if (roi.kind == 2) {
                const bool r4 = first && j < 17;
                const double hh = r4 ? len * 0.0625 : ldexp(len, 1 - i);
                const double at = r4 ? roi.r0 : roi.r0 + hh * 0.5;
                const double step = (double)(first && !r4 ? j - 17 : j0 + j);
                cg = roi.k1 * lc0_cos(at + hh * step) + roi.k0;
              }
              f = lc0_raw<true>(v, raw, cg, dummy);
            }
            S.sv[t * kLc0RedoPts + j] = f;
          }
        }
        __syncthreads();
        if (tid < nr && S.act[tid])
          for (int j = 0; j < m; ++j) {
            const double f = S.sv[tid * kLc0RedoPts + j];
            if (first && j < 17) sm.add(j, f);
            else c += f;
          }
      }
      if (tid == 0) S.nact = 0;
      __syncthreads();
      if (tid < nr && S.act[tid]) {
        const int p = S.redo[b0 + tid];
        const unsigned it = S.item[p];
        const int nu = (int)(it >> 9);
        const LC0Roi roi = lc0_roi(L, L.sets[k0 + (int)((it >> 1) & 255u)], S.wl[nu], S.c3[nu], S.s3[nu],
                                   (it & 1u) ? -1.0 : 1.0);
        const double len = roi.r1 - roi.r0;
        double* row = S.sv + kLc0Redo * kLc0RedoPts + 16 * tid;
        bool done = true;
        double x;
        if (roi.kind != 2) {
          x = sm.s_end;  // its one value
        } else if (first) {
          double r[6];
          done = lc0_rows4(sm, len, L.acc, r);
          x = r[4];
          if (!done) {
            done = lc0_row5(c, len, L.acc, r);
            x = r[5];
            for (int j = 0; j < 6; ++j) row[j] = r[j];
          }
          x *= 1.0 / kPi;
        } else {
          done = lc0_row(i, c, ldexp(len, -i), L.acc, row);
          x = row[i] * (1.0 / kPi);
        }
        if (done || i == 15) {
          S.val[p] = x;
          S.act[tid] = 0;
        } else {
          S.nact = 1;
        }
      }
      __syncthreads();
      if (!S.nact) break;  // the same for the whole workgroup
    }
    b0 += nr;
    if (b0 == nredo) b0 = kLc0List - nslow;
  }
  __syncthreads();
}

// One pass over the ranges of the workgroup's neutrons in order, in rounds of
// whole neutrons; lane nu < nb holds neutron nu's running sum tot (valid: it
// has one).  Mode kLc0Sum adds up the values.  kLc0Find also keeps in pick
// (plane set << 1 | side) the first range at which the sum exceeds target, or
// the last range.  kLc0SumPick, for plane sets that fit one round's masks, does
// both at once: the sum of a round's neutrons is complete and their values are
// still in S, so the target is drawn (the first number of neutron i's stream) and
// the values walked again.  listed >= 0: that many ranges are in S.item already, all
// there are, with S.mask and S.off per neutron.
enum : int { kLc0Sum, kLc0SumPick, kLc0Find };
template <int Mode>
NCD void lc0_pass(const LC0View& L, const SCBView& v, Lc0Lds& S, int nb, int listed, bool valid, uint64_t seed,
                  uint32_t stream, int64_t i, double target, double& tot, int64_t& pick) {
  const int tid = (int)threadIdx.x;
  bool found = false;
  for (int k0 = 0; k0 < L.nsets; k0 += kLc0Sets) {
    const int nk = L.nsets - k0 < kLc0Sets ? L.nsets - k0 : kLc0Sets;
    const int nw = listed < 0 ? (nk + 31) >> 5 : 1;
    const int units = nb * nw;  // unit u: mask word u % nw of neutron u / nw
    if (listed < 0) {
      for (int u = tid; u < units; u += kLc0Threads) {
        const int nu = u / nw;
        const int ka = k0 + 32 * (u - nu * nw), kb = ka + 32 < k0 + nk ? ka + 32 : k0 + nk;
        const double wl = S.wl[nu], c3 = S.c3[nu], s3 = S.s3[nu];
        uint64_t m = 0;
        for (int k = ka; k < kb; ++k) {
          const LC0Set ps = L.sets[k];
          if (wl > ps.twodsp) break;
          m |= (uint64_t)lc0_sides(L, ps, wl, c3, s3) << (2 * (k - ka));
        }
        S.mask[u] = m;
      }
      __syncthreads();
      if (tid < 64) {  // prefix sum of the units' counts
        const int per = (units + 63) >> 6;
        int s = 0;
        for (int u = tid * per; u < (tid + 1) * per && u < units; ++u) s += __popcll(S.mask[u]);
        int run = s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int y = __shfl_up(run, o, 64);
          if (tid >= o) run += y;
        }
        int at = run - s;
        for (int u = tid * per; u < (tid + 1) * per && u < units; ++u) {
          S.off[u] = at;
          at += __popcll(S.mask[u]);
        }
        if (tid == 63) S.off[units] = run;
      }
      __syncthreads();
    }
    for (int n0 = 0; n0 < nb;) {
      // neutrons n0 .. n1 - 1: as many as the lists hold (one always fits)
      int base = 0, n1 = nb, n = listed;
      if (listed < 0) {
        base = S.off[n0 * nw];
        if (S.off[units] - base > kLc0List) {
          n1 = n0 + 1;
          while (S.off[(n1 + 1) * nw] - base <= kLc0List) ++n1;
        }
        n = S.off[n1 * nw] - base;
        if (n == 0) break;  // none in reach: n1 is nb
        for (int u = n0 * nw + tid; u < n1 * nw; u += kLc0Threads) {
          const int nu = u / nw;
          uint64_t m = S.mask[u];
          for (int p = S.off[u] - base; m; ++p) {
            const int b = __builtin_ctzll(m);
            m &= m - 1ull;
            S.item[p] = (uint16_t)((nu << 9) | (64 * (u - nu * nw) + b));
          }
        }
        __syncthreads();
      }
      lc0_values(L, v, S, k0, n);
      if (valid && tid >= n0 && tid < n1) {
        const int p0 = S.off[tid * nw] - base;
        const int e = listed < 0 ? S.off[(tid + 1) * nw] - base : p0 + __popcll(S.mask[tid]);
        for (int p = p0; p < e; ++p) {
          tot += S.val[p];
          if (Mode == kLc0Find && !found) {
            pick = 2 * (int64_t)k0 + (S.item[p] & 511u);
            found = tot > target;
          }
        }
        if (Mode == kLc0SumPick && tot > 0.0) {
          Rng r;
          r.init(seed, stream, (uint64_t)i);
          target = r.gen() * tot;
          double run = 0.0;
          for (int p = p0; p < e && !found; ++p) {
            run += S.val[p];
            pick = S.item[p] & 511u;
            found = run > target;
          }
        }
      }
      n0 = n1;
      if (n0 < nb) __syncthreads();  // the lists are rewritten
    }
    if (listed >= 0) break;  // all
    if (k0 + kLc0Sets < L.nsets) __syncthreads();
  }
}
static_assert(2 * kLc0Sets <= kLc0List, "a neutron's ranges of one round fit the lists");

// Cross sections, or scattering (LCHelper::genScatter, NCLCUtils.cc:518-690):
// a ROI by its cross section; in it a rotation phi by rejection under the
// reference's envelope (8 bins over the range, each the larger end value
// times 1.7 plus 2% of the largest, at most 1000 tries), uniform for a neutron
// along the axis; a random sign of sin(phi); the Gaussian-mosaic scattering of
// the reversed neutron (-s3, 0, -c3) off that normal in the frame of the axis
// (LCStdFrame::genScat, :755-772), taken to the lab frame by the neutron and
// the axis (rotateToFrame) and reversed.  For the workgroup's neutrons base +
// S.work[r0 .. r0 + nb); listed: see lc0_pass.
template <bool Sample>
NCD void lc0_round(const LC0View& L, const SCBView& v, Lc0Lds& S, const double* __restrict__ ekin,
                   const double* __restrict__ dirs, int64_t base, int r0, int nb, int listed,
                   uint64_t seed, uint32_t stream, double* __restrict__ o1, double* __restrict__ oD) {
  const int tid = (int)threadIdx.x;
  const bool valid = tid < nb;
  const int64_t i = base + (valid ? S.work[r0 + tid] : 0);
  // (nothing of a neutron but its place stays in registers through the
  // integrals: it is read again)
  if (listed < 0) {
    if (valid) {
      double ux = dirs[3 * i], uy = dirs[3 * i + 1], uz = dirs[3 * i + 2], c3raw;
      lc0_neutron(L, ekin[i], ux, uy, uz, S.wl[tid], c3raw, S.c3[tid], S.s3[tid]);
    }
    __syncthreads();
  }
  double tot = 0.0;
  int64_t pick = 0;
  if constexpr (!Sample) {
    lc0_pass<kLc0Sum>(L, v, S, nb, listed, valid, seed, stream, i, -1.0, tot, pick);
    if (valid) o1[i] = L.xsfact * tot;
  } else {
    if (L.nsets <= kLc0Sets) {
      lc0_pass<kLc0SumPick>(L, v, S, nb, listed, valid, seed, stream, i, -1.0, tot, pick);
    } else {
      lc0_pass<kLc0Sum>(L, v, S, nb, listed, valid, seed, stream, i, -1.0, tot, pick);
      double target = 0.0, run = 0.0;
      if (valid && tot > 0.0) {
        Rng r;
        r.init(seed, stream, (uint64_t)i);
        target = r.gen() * tot;
      }
      __syncthreads();
      lc0_pass<kLc0Find>(L, v, S, nb, listed, valid && tot > 0.0, seed, stream, i, target, run, pick);
    }
    const bool scat = valid && tot > 0.0;
    // The rotation in the picked range, with the workgroup's lanes shared out
    // among the neutrons that need one: the envelope's 9 points, then `per`
    // tries at a time (each try takes the next three numbers of the neutron's
    // stream, so a lane can draw try t without the ones before; the first
    // accepted one counts).  One lane per neutron made a wave wait for its
    // longest rejection, 0.8 ms more for 131072 neutrons than the ranges' own
    // 1.05 ms; shared out it is 0.2 ms.
    if (tid == 0) S.nact = 0;
    __syncthreads();  // S.val and S.sv change their use
    LC0Set ps{};
    double sg = 1.0;
    int kind = 0, mine = 0;                // mine: place among those neutrons
    double* par = S.val;                   // [nact][8] k1, k0, r0, length, sinpt, cospt, Q, fixed
    double* env = S.sv;                    // [nact][9]
    double* got = S.sv + 9 * kLc0Neutrons; // [nact] cos(phi), with the number of tries in S.off
    if (scat) {
      ps = L.sets[pick >> 1];
      sg = (pick & 1) ? -1.0 : 1.0;
      const LC0Roi roi = lc0_roi(L, ps, S.wl[tid], S.c3[tid], S.s3[tid], sg);
      kind = roi.kind;
      if (kind == 2) {
        mine = atomicAdd(&S.nact, 1);
        S.turn[mine] = (uint8_t)tid;
        const LC0Raw raw = lc0_raw_setup(S.wl[tid], ps.inv2d, ps.fsq);
        double* q = par + 8 * mine;
        q[0] = roi.k1; q[1] = roi.k0; q[2] = roi.r0; q[3] = roi.r1 - roi.r0;
        q[4] = raw.sinpt; q[5] = raw.cospt; q[6] = raw.Q; q[7] = raw.fixed;
      }
    }
    __syncthreads();
    const int ns = S.nact;
    bool dummy = false;
    for (int q = tid; q < 9 * ns; q += kLc0Threads) {
      const int nu = q / 9, j = q - 9 * nu;
      const double* z = par + 8 * nu;
      const LC0Raw raw{z[4], z[5], z[6], z[7]};
      env[q] = lc0_raw<true>(v, raw, z[0] * lc0_cos(z[2] + j * (z[3] * 0.125)) + z[1], dummy);
    }
    __syncthreads();
    if (ns > 0) {
      int per = 64;  // lanes of a neutron (a power of two)
      while (per * ns > kLc0Threads) per >>= 1;
      const int nu = tid / per, q = tid - nu * per;
      const bool on = nu < ns;
      const int64_t inu = base + S.work[r0 + S.turn[on ? nu : 0]];
      const double* z = par + 8 * (on ? nu : 0);
      float data[8];
      if (on) {
        double mx = 0.0;
#pragma unroll
        for (int j = 0; j < 9; ++j) mx = dmax(mx, env[9 * nu + j]);
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          data[j] = (sum += (float)(dmax(env[9 * nu + j], env[9 * nu + j + 1]) * 1.7 + 0.02 * mx));
      }
      const LC0Raw raw{z[4], z[5], z[6], z[7]};
      const uint64_t group = (per == 64 ? ~0ull : ((1ull << per) - 1ull)) << ((tid & 63) / per * per);
      bool open = on;
      for (int t0 = 0; t0 < 1000; t0 += per) {
        const int t = t0 + q;
        bool ok = false;
        double cosphi = 0.0;
        if (open && t < 1000) {
          Rng g;  // draws 1 + 3 t .. of the neutron's stream
          g.init(seed, stream, (uint64_t)inu);
          g.c0 = (uint32_t)(1 + 3 * t) >> 1;
          if ((1 + 3 * t) & 1) (void)g.gen();
          const float y = data[7] * (float)g.gen();
          int b = 0;
          float below = 0.0f, at = data[0];
#pragma unroll
          for (int k = 1; k < 8; ++k)
            if (b == k - 1 && at < y) { b = k; below = at; at = data[k]; }
          const double ov = b ? (double)at - (double)below : (double)at;
          cosphi = lc0_cos(z[2] + ((b + g.gen()) * 0.125) * z[3]);
          const double xs = lc0_raw<true>(v, raw, z[0] * cosphi + z[1], dummy);
          ok = xs > ov * g.gen() || t == 999;  // the last try stands
        }
        const uint64_t m = __ballot(ok) & group;
        if (open && m) {
          if ((tid & 63) == __builtin_ctzll(m)) {
            got[nu] = cosphi;
            S.off[nu] = t + 2;
          }
          open = false;
        }
        if (!__any(open)) break;
      }
    }
    __syncthreads();
    if (valid) {
      const double E = ekin[i];
      double ox = dirs[3 * i], oy = dirs[3 * i + 1], oz = dirs[3 * i + 2];
      if (scat) {
        double ux = ox, uy = oy, uz = oz, wl, c3raw, c3, s3;
        lc0_neutron(L, E, ux, uy, uz, wl, c3raw, c3, s3);
        const V3 indir_std{-s3, 0.0, -c3};
        V3 normal{0.0, 0.0, sg};
        const int d = kind == 2 ? 1 + 3 * (S.off[mine] - 1) : 1;  // numbers drawn so far
        Rng r;
        r.init(seed, stream, (uint64_t)i);
        r.c0 = (uint32_t)d >> 1;
        if (d & 1) (void)r.gen();
        if (kind != 0) {
          const double cosphi = kind == 1 ? cos(r.gen() * kPi) : got[mine];
          const double sgn = r.gen() < 0.5 ? 1.0 : -1.0;
          const double sinphi = sgn * sqrt(dmax(0.0, 1.0 - cosphi * cosphi));
          const double ns1 = sg * ps.s1;
          normal = V3{ns1 * cosphi, ns1 * sinphi, sg * ps.c1};
        }
        const V3 w = gm_genscat(v, r, normal, gm_round(ps.inv2d), wl, indir_std);
        const double isg = c3raw >= 0.0 ? 1.0 : -1.0;
        const V3 a{ux, uy, uz}, b{L.ax * isg, L.ay * isg, L.az * isg};
        const V3 o = rotate_to_frame(s3, c3, a, b, w, r);
        ox = -o.x;
        oy = -o.y;
        oz = -o.z;
      }
      o1[i] = E;
      oD[3 * i] = ox;
      oD[3 * i + 1] = oy;
      oD[3 * i + 2] = oz;
    }
  }
}

// the ranges of the first plane sets (two bits each, lc0_sides); all: there are
// no others in reach
constexpr int kLc0Look = 4;
NCD unsigned lc0_look(const LC0View& L, double wl, double c3, double s3, bool& all) {
  unsigned m = 0;
  all = true;
  for (int k = 0; k < kLc0Look && k < L.nsets; ++k) {
    const LC0Set ps = L.sets[k];
    if (wl > ps.twodsp) return m;
    m |= lc0_sides(L, ps, wl, c3, s3) << (2 * k);
  }
  all = L.nsets <= kLc0Look;
  return m;
}
static_assert(2 * kLc0Look * kLc0Neutrons <= kLc0List, "listed ranges");

// A workgroup's `per` neutrons, one per lane first: those that have no range
// (all beyond the first plane sets' wavelengths, and there most others: 0.5-7
// Aa about half of a batch) are done at once, the others in rounds.
template <bool Sample>
__global__ void __launch_bounds__(kLc0Threads, 4) k_lc0(LC0View L, SCBView v, const double* __restrict__ ekin,
                                                     const double* __restrict__ dirs, int64_t i0, int64_t n, int per,
                                                     uint64_t seed, uint32_t stream, double* __restrict__ o1,
                                                     double* __restrict__ oD) {
  __shared__ Lc0Lds S;
  const int tid = (int)threadIdx.x;
  const int64_t base = i0 + (int64_t)blockIdx.x * per;
  if (tid == 0) { S.nwork = 0; S.nlisted = 0; S.more = 0; }
  __syncthreads();
  {
    const int64_t i = base + tid;
    const bool mine = tid < per && i < n;
    bool work = false, all = true;
    unsigned m = 0;
    double wl = 0.0, c3 = 0.0, s3 = 0.0;
    double E = 0.0, dx = 0.0, dy = 0.0, dz = 0.0;
    if (mine) {
      E = ekin[i];
      dx = dirs[3 * i]; dy = dirs[3 * i + 1]; dz = dirs[3 * i + 2];
      if (E > 0.0) {
        double ux = dx, uy = dy, uz = dz, c3raw;
        lc0_neutron(L, E, ux, uy, uz, wl, c3raw, c3, s3);
        m = lc0_look(L, wl, c3, s3, all);
        work = m || !all;
      }
    }
    const uint64_t B = __ballot(work);
    int at = 0;
    if ((tid & 63) == 0 && B) at = atomicAdd(&S.nwork, __popcll(B));
    at = __builtin_amdgcn_readfirstlane(at) + __popcll(B & ((1ull << (tid & 63)) - 1ull));
    if (work) S.work[at] = (uint8_t)tid;
    if (__any(!all)) {
      S.more = 1;
    } else if (work && at < kLc0Neutrons) {
      // listed here already, which counts if it holds for the whole workgroup
      S.wl[at] = wl;
      S.c3[at] = c3;
      S.s3[at] = s3;
      S.mask[at] = m;
      int p = atomicAdd(&S.nlisted, __popc(m));
      S.off[at] = p;
      for (unsigned q = m; q; q &= q - 1u) S.item[p++] = (uint16_t)((at << 9) | __builtin_ctz(q));
    }
    if (mine && !work) {
      if constexpr (Sample) {
        o1[i] = E;
        oD[3 * i] = dx;
        oD[3 * i + 1] = dy;
        oD[3 * i + 2] = dz;
      } else {
        o1[i] = 0.0;
      }
    }
  }
  __syncthreads();
  const int nwork = S.nwork;
  if (nwork == 0) return;
  const bool ready = !S.more && nwork <= kLc0Neutrons;
  const int nw = ready ? 1 : (L.nsets < kLc0Sets ? (L.nsets + 31) >> 5 : kLc0Words);
  const int most = kLc0Units / nw < kLc0Neutrons ? kLc0Units / nw : kLc0Neutrons;
  const int rounds = (nwork + most - 1) / most, nb = (nwork + rounds - 1) / rounds;
  for (int r0 = 0; r0 < nwork; r0 += nb) {
    if (r0) __syncthreads();
    lc0_round<Sample>(L, v, S, ekin, dirs, base, r0, nwork - r0 < nb ? nwork - r0 : nb, ready ? S.nlisted : -1, seed, stream,
                      o1, oD);
  }
}

// neutrons of a workgroup: 64 where that gives every CU two workgroups, fewer
// for small batches, so that a batch still spreads over the chip; 128 and 256
// where that leaves the chip filled 2 and 8 times.  Many share the steps' latencies
// where few have ranges (4.3-6 Aa, cross sections: 3e5 neutrons 25 us with 128, 21
// with 256; 2^21 126 and 73), but even out worse where most have (0.5-7 Aa, both
// calls of 131072 neutrons 2.20 ms with 64, 2.30 with 128; cross sections of 2^20
// 6.06 ms with 128, 6.35 with 256; of 2^21 11.6 and 12.0).
int lc0_group(int64_t n) {
  int nb = kLc0Threads;
  while (nb > 4 && n < (int64_t)(nb > 128 ? 8192 : (nb > 64 ? 2048 : 512)) * nb) nb >>= 1;
  return nb;
}

}  // namespace

// at most kLc0Launch neutrons a launch: a grid holds fewer than 2^32 work-items
constexpr int64_t kLc0Launch = (int64_t)1 << 28;
static_assert((kLc0Launch / kLc0Threads + 1) * kLc0Threads < ((int64_t)1 << 32), "work-items of a launch");
template <bool Sample>
static void launch_lc0(const LC0View& L, const SCBView& v, const double* ekin, const double* dirs, int64_t n,
                       uint64_t seed, uint32_t stream, double* o1, double* oD, hipStream_t st) {
  const int nb = lc0_group(n);
  for (int64_t i0 = 0; i0 < n; i0 += kLc0Launch) {
    const int64_t end = n - i0 < kLc0Launch ? n : i0 + kLc0Launch;
    hipLaunchKernelGGL(k_lc0<Sample>, dim3((unsigned)((end - i0 + nb - 1) / nb)), dim3(kLc0Threads), 0, st, L, v, ekin,
                       dirs, i0, end, nb, seed, stream, o1, oD);
  }
}
void launch_lc0_xs(const LC0View& L, const SCBView& v, const double* ekin, const double* dirs, int64_t n, double* out,
                   hipStream_t st) {
  launch_lc0<false>(L, v, ekin, dirs, n, 0, 0, out, nullptr, st);
}
void launch_lc0_sample(const LC0View& L, const SCBView& v, const double* ekin, const double* dirs, int64_t n,
                       uint64_t seed, uint32_t stream, double* oE, double* oD, hipStream_t st) {
  launch_lc0<true>(L, v, ekin, dirs, n, seed, stream, oE, oD, st);
}

void launch_lc_expand(const double* ekin, const double* dirs, int64_t n, int N, const LCView& L, const double2* cs,
                      uint64_t seed, uint32_t stream, double* oE, double* oD, double2* ocs, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_lc_expand, dim3(lc_blocks(n * N)), dim3(256), 0, st, ekin, dirs, n, N, L, cs, seed, stream, oE,
                     oD, ocs);
}
void launch_lc_mean(const double* xs, int64_t n, int N, double* out, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_lc_mean, dim3(lc_blocks(n)), dim3(256), 0, st, xs, n, N, out);
}
void launch_lc_pick(const double* xs, const double* rE, const double* rD, int64_t n, int N, uint64_t seed,
                    uint32_t stream, double* sE, double* sD, int* sel, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_lc_pick, dim3(lc_blocks(n)), dim3(256), 0, st, xs, rE, rD, n, N, seed, stream, sE, sD, sel);
}
void launch_lc_unrotate(const double* scD, const int* sel, const double2* cs, const double* ekin, const double* dirs,
                        int64_t n, int N, const LCView& L, double* oE, double* oD, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_lc_unrotate, dim3(lc_blocks(n)), dim3(256), 0, st, scD, sel, cs, ekin, dirs, n, N, L, oE, oD);
}

}  // namespace ncamd

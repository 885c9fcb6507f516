// Non-spherical particles on the device: support functions, the GJK distance
// with Johnson's sub-distance algorithm, the general ClosestPoint path with
// crust-shrunk transforms and its ContactError handling, and the rigid-body
// kinematics of ParticleKinematics3D.
//
//   RigidBodyWithCrust::ClosestPoint ........ RigidBodyWithCrust.cpp:205-354
//   ClosestPoint_ErreurHandling ............. RigidBodyWithCrust.cpp:534-590, 770-798
//   closest_points (Johnson, no Nesterov) ... Convex.cpp:219-435, 536-627
//   Sphere / Box / Polyhedron::support ...... Sphere.cpp:99-110, Box.cpp:307-316,
//                                              Polyhedron.cpp:265-293, 431-439
//   computeAngularAccelerationBodyFixed ..... ParticleKinematics3D.cpp:56-77
//   Transform::composeLeftByRotation ........ Transform.cpp:140-159
//
// The polyhedron support scans all vertices and keeps the first maximum
// (Polyhedron::support20); the reference hill-climbs from a per-particle warm
// start.  Both return the maximising vertex; they can differ only among tied
// maxima, i.e. for a face exactly parallel to the search direction.
#pragma once
#include <type_traits>

#include "dem_math.hpp"
#include "dem_types.hpp"

namespace dem {

constexpr double kEps2 = 1.e-15;  // Basic.hh EPSILON2
constexpr double kEps3 = 1.e-20;  // Basic.hh EPSILON3

// Work area of one distance search: the simplex of up to four points of the
// Minkowski difference by slot -- y (entries 0-11), the support points p and q
// in the local frames (12-23, 24-35) and the weight of each kept slot (36-39)
// -- with entry e at a[e * st].  On the device it lies in LDS, one column per
// lane, so that slots are addressed at run time without scratch memory or a
// copy of the code per slot.
constexpr int kGjkWork = 40;
struct GjkWork {
  double* a;
  int st;
};

// A rigid body with crust as ClosestPoint sees it
struct ConvexGeo {
  int type, nv;
  const double* verts;
  double r;       // sphere radius
  d3 e;           // box half extents
  double B[9];    // basis rows of the Transform (no crust)
  d3 o;           // origin
  d3 scaling;     // crust shrink factors
  d3 bext;        // bbox half extents at the identity transform
  double crust, circR;
  d3 obb;         // OBB half extents at the identity (bounding-volume pre-test)
  GjkOpts opt;    // the system's narrow-phase options
  GjkWork work{nullptr, 1};  // body A's: the search's work area (device)
};

struct Tf {
  double B[9];
  d3 o;
};

// Transform::operator() (Transform.cpp:312-317)
DEM_HD d3 tf_apply(const Tf& t, d3 p) {
  return d3{dot(d3{t.B[0], t.B[1], t.B[2]}, p) + t.o.x, dot(d3{t.B[3], t.B[4], t.B[5]}, p) + t.o.y,
            dot(d3{t.B[6], t.B[7], t.B[8]}, p) + t.o.z};
}
// Vector3 * Matrix (Matrix.cpp:238-241, 527-530)
DEM_HD d3 tf_vec_basis(d3 v, const Tf& t) {
  return d3{t.B[0] * v.x + t.B[3] * v.y + t.B[6] * v.z, t.B[1] * v.x + t.B[4] * v.y + t.B[7] * v.z,
            t.B[2] * v.x + t.B[5] * v.y + t.B[8] * v.z};
}
// Transform::composeWithScaling (Matrix.cpp:347-358)
DEM_HD Tf tf_scaled(const ConvexGeo& g, d3 sc) {
  Tf t;
  for (int i = 0; i < 3; ++i) {
    t.B[3 * i] = g.B[3 * i] * sc.x;
    t.B[3 * i + 1] = g.B[3 * i + 1] * sc.y;
    t.B[3 * i + 2] = g.B[3 * i + 2] * sc.z;
  }
  t.o = g.o;
  return t;
}

// norm(v) < 1e-10 and norm(v) > 1e-10 without the square root: the squares
// at which the correctly rounded root crosses the bound.
DEM_HD bool norm_below_eps(d3 v) { return v.x * v.x + v.y * v.y + v.z * v.z < 0x1.79ca10c924223p-67; }
DEM_HD bool norm_above_eps(d3 v) { return v.x * v.x + v.y * v.y + v.z * v.z > 0x1.79ca10c924224p-67; }

// Vertices of a polyhedron are scanned in groups of this many; the vertex
// table holds each shape's vertices filled up to whole groups with copies of
// the last one (never the first maximum).
constexpr int kVertGroup = 4;

DEM_HD d3 support(const ConvexGeo& g, d3 v) {
  if (g.type == kShapeSphere) {
    double s = norm(v);
    if (s > kEps) {
      double f = g.r / s;
      return d3{v.x * f, v.y * f, v.z * f};
    }
    return d3{0., 0., 0.};
  }
  if (g.type == kShapeBox) {
    if (norm_below_eps(v)) return d3{0., 0., 0.};
    return d3{v.x < 0. ? -g.e.x : g.e.x, v.y < 0. ? -g.e.y : g.e.y, v.z < 0. ? -g.e.z : g.e.z};
  }
  if (!norm_above_eps(v)) return d3{0., 0., 0.};
  // the first maximum; a group's loads overlap
  const double* p = g.verts;
  int best = 0;
  double h = -INFINITY;
  for (int i = 0; i < g.nv; i += kVertGroup) {
    double d[kVertGroup];
#pragma unroll
    for (int u = 0; u < kVertGroup; ++u) {
      const double* c = p + 3 * (i + u);
      d[u] = dot(d3{c[0], c[1], c[2]}, v);
    }
#pragma unroll
    for (int u = 0; u < kVertGroup; ++u) {
      const bool more = d[u] > h;
      h = more ? d[u] : h;
      best = more ? i + u : best;
    }
  }
  return d3{p[3 * best], p[3 * best + 1], p[3 * best + 2]};
}

// --- Johnson sub-distance algorithm -----------------------------------------
DEM_HD d3 work_get(const GjkWork& W, int e) { return d3{W.a[e * W.st], W.a[(e + 1) * W.st], W.a[(e + 2) * W.st]}; }
DEM_HD void work_put(const GjkWork& W, int e, d3 v) {
  W.a[e * W.st] = v.x;
  W.a[(e + 1) * W.st] = v.y;
  W.a[(e + 2) * W.st] = v.z;
}
DEM_HD d3 work_y(const GjkWork& W, int slot) { return work_get(W, 3 * slot); }
DEM_HD double& work_w(const GjkWork& W, int slot) { return W.a[(36 + slot) * W.st]; }

// f(integral_constant<int, i>) for i = B, B+1, ..., E-1
template <int B, int E, class F>
DEM_HD void sfor(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    sfor<B + 1, E>(f);
  }
}

// The determinants of computeDet (Convex.cpp:219-268) for subsets picked at
// run time, from the points in the work area; f is the slot just added, and
// the triple without it is the one kept by the last step, whose determinants
// are the weights in the work area.  Only the backup procedure below needs
// subsets by number; it runs once per search at most.
DEM_HD double j_det3(const GjkWork& W, unsigned s, int i, int f) {
  if (!(s & (1u << f))) return work_w(W, i);
  // k < j the other two
  const unsigned o = s & ~(1u << f);
  const int k = __builtin_ctz(o), j = __builtin_ctz(o & (o - 1));
  const d3 yk = work_y(W, k), yj = work_y(W, j), yl = work_y(W, f);
  const double kk = dot(yk, yk), jj = dot(yj, yj), ll = dot(yl, yl), jk = dot(yk, yj), lk = dot(yk, yl), lj = dot(yj, yl);
  if (i == k) return (ll - lj) * (jj - jk) + (jj - lj) * (lj - lk);
  if (i == j) return (ll - lk) * (kk - jk) + (kk - lk) * (lk - lj);
  return (jj - jk) * (kk - lk) + (kk - jk) * (jk - lj);
}
DEM_HD double j_det_of(const GjkWork& W, unsigned s, int i, int f) {
  const int c = __builtin_popcount(s);
  if (c == 1) return 1.;
  const unsigned rest = s & ~(1u << i);
  if (c == 2) {
    const d3 yi = work_y(W, i), yo = work_y(W, __builtin_ctz(rest));
    return dot(yo, yo) - dot(yi, yo);
  }
  if (c == 3) return j_det3(W, s, i, f);
  const int r = __builtin_ctz(rest);
  double det = 0.;
  bool first = true;
  for (unsigned m = rest; m; m &= m - 1) {
    const int j = __builtin_ctz(m);
    const d3 yj = work_y(W, j);
    const double t = j_det3(W, rest, j, f) * (dot(yj, work_y(W, r)) - dot(yj, work_y(W, i)));
    det = first ? t : det + t;
    first = false;
  }
  return det;
}

// The backup procedure of closest (Convex.cpp:389-414): the subset of
// all_bits with positive determinants whose point is nearest to the origin.
DEM_HD void j_backup(const GjkWork& W, unsigned& bits, unsigned all_bits, int f, d3& v) {
  double min_dist2 = INFINITY, w[4] = {0., 0., 0., 0.};
  unsigned best = 0u;
#pragma nounroll
  for (unsigned s = 15u; s > 0u; --s) {
    if ((s & all_bits) != s) continue;
    bool proper = true;
    double sum = 0., det[4] = {0., 0., 0., 0.};
    d3 u{0., 0., 0.};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (s & (1u << i)) {
        det[i] = j_det_of(W, s, i, f);
        if (det[i] <= kEps3) proper = false;
        sum += det[i];
        u += det[i] * work_y(W, i);
      }
    if (!proper) continue;
    u *= 1. / sum;
    const double d2 = dot(u, u);
    if (d2 < min_dist2) {
      min_dist2 = d2;
      best = s;
      v = u;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = det[i];
    }
  }
  if (!best) return;
  bits = best;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (best & (1u << i)) work_w(W, i) = w[i];
}

// closest (Convex.cpp:342-414) for the point w just added in slot f, the
// first free one: the smallest valid subset containing it, else the backup
// procedure.  The kept points of the last step, up to three, are called A, B
// and C in slot order, the new point L; every determinant of a subset
// containing L is the slot-indexed one's arithmetic with these names (pairs
// and triples do not depend on where L stands; the sums over four points and
// of the result run in slot order, in which L stands after f of A, B, C).
// One copy of this code serves every slot; of a copy for each slot a wave runs
// all that its lanes need, one after the other (623 us per launch against 289,
// 200,000-body hopper).
DEM_HD bool j_closest(const GjkWork& W, unsigned& bits, unsigned all_bits, int f, const d3& w, d3& v) {
  const bool hA = bits != 0u;
  const unsigned r1 = bits & (bits - 1u), r2 = r1 & (r1 - 1u);
  const bool hB = r1 != 0u, hC = r2 != 0u;
  const int sA = hA ? __builtin_ctz(bits) : 0, sB = hB ? __builtin_ctz(r1) : 0, sC = hC ? __builtin_ctz(r2) : 0;
  auto pos = [](double d) { return !(d <= kEps3); };
  auto neg = [](double d) { return !(d > 0.); };
  // the subset found: which of A, B, C (1, 2, 4) it holds beside L
  unsigned sel = 8u;
  auto take = [&](bool ok, unsigned m) { sel = sel == 8u && ok ? m : sel; };
  double pA = 0., lA = 0., pB = 0., lB = 0., pC = 0., lC = 0., abA = 0., abB = 0., abL = 0., acA = 0., acC = 0.,
         acL = 0., bcB = 0., bcC = 0., bcL = 0., qA = 0., qB = 0., qC = 0., qL = 0.;
  const d3 zero{0., 0., 0.};
  d3 yA = zero, yB = zero, yC = zero;
  const double LL = dot(w, w);
  if (hA) {
    yA = work_y(W, sA);
    const double AA = dot(yA, yA), LA = dot(yA, w);
    pA = LL - LA;  // det of {A, L}: A's, L's
    lA = AA - LA;
    bool onlyA = pos(pA) && pos(lA), onlyL = neg(pA);
    if (hB) {
      yB = work_y(W, sB);
      const double BB = dot(yB, yB), LB = dot(yB, w), AB = dot(yA, yB);
      pB = LL - LB;
      lB = BB - LB;
      abA = pB * (BB - AB) + lB * (LB - LA);
      abB = pA * (AA - AB) + lA * (LA - LB);
      abL = (BB - AB) * (AA - LA) + (AA - AB) * (AB - LB);
      bool onlyB = pos(pB) && pos(lB) && neg(abA), onAB = pos(abA) && pos(abB) && pos(abL);
      onlyA = onlyA && neg(abB);
      onlyL = onlyL && neg(pB);
      if (hC) {
        yC = work_y(W, sC);
        const double CC = dot(yC, yC), LC = dot(yC, w), AC = dot(yA, yC), BC = dot(yB, yC);
        pC = LL - LC;
        lC = CC - LC;
        acA = pC * (CC - AC) + lC * (LC - LA);
        acC = pA * (AA - AC) + lA * (LA - LC);
        acL = (CC - AC) * (AA - LA) + (AA - AC) * (AC - LC);
        bcB = pC * (CC - BC) + lC * (LC - LB);
        bcC = pB * (BB - BC) + lB * (LB - LC);
        bcL = (CC - BC) * (BB - LB) + (BB - BC) * (BC - LC);
        // four points: sums over the other three in slot order, with the
        // first of them as the reference point
        // (l + a and a + l are the same sum, so only "before b" matters)
        auto sum3 = [](bool l_before_b, double l, double a, double b) {
          return (a + (l_before_b ? l : b)) + (l_before_b ? b : l);
        };
        qL = (work_w(W, sA) * (AA - LA) + work_w(W, sB) * (AB - LB)) + work_w(W, sC) * (AC - LC);
        const bool l0 = f == 0, l1 = f <= 1, l2 = f <= 2;
        // others of A: B, C and L (first when f <= 1)
        qA = sum3(l2, bcL * ((l1 ? LL : LB) - LA), bcB * ((l1 ? LB : BB) - AB), bcC * ((l1 ? LC : BC) - AC));
        // others of B: A, C and L (first when f == 0)
        qB = sum3(l2, acL * ((l0 ? LL : LA) - LB), acA * ((l0 ? LA : AA) - AB), acC * ((l0 ? LC : AC) - BC));
        // others of C: A, B and L (first when f == 0)
        qC = sum3(l1, abL * ((l0 ? LL : LA) - LC), abA * ((l0 ? LA : AA) - AC), abB * ((l0 ? LB : AB) - BC));
        take(pos(qA) && pos(qB) && pos(qC) && pos(qL), 7u);
        take(pos(bcB) && pos(bcC) && pos(bcL) && neg(qA), 6u);
        take(pos(acA) && pos(acC) && pos(acL) && neg(qB), 5u);
        take(pos(pC) && pos(lC) && neg(acA) && neg(bcB), 4u);
        onAB = onAB && neg(qC);
        onlyB = onlyB && neg(bcC);
        onlyA = onlyA && neg(acC);
        onlyL = onlyL && neg(pC);
      }
      take(onAB, 3u);
      take(onlyB, 2u);
    }
    take(onlyA, 1u);
    take(onlyL, 0u);
  } else {
    sel = 0u;
  }
  if (sel == 8u) {
    j_backup(W, bits, all_bits, f, v);
    return false;
  }
  const bool cA = (sel & 1u) != 0u, cB = (sel & 2u) != 0u, cC = (sel & 4u) != 0u;
  const double kL = cC ? (cB ? (cA ? qL : bcL) : (cA ? acL : lC)) : (cB ? (cA ? abL : lB) : (cA ? lA : 1.));
  const double kA = !cA ? 0. : (cC ? (cB ? qA : acA) : (cB ? abA : pA));
  const double kB = !cB ? 0. : (cC ? (cA ? qB : bcB) : (cA ? abB : pB));
  const double kC = !cC ? 0. : (cB ? (cA ? qC : bcC) : (cA ? acC : pC));
  // computeVector (Convex.cpp:294-306): sums in slot order
  const bool l1 = f <= 1, l2 = f == 2, l3 = f <= 2;
  auto ordered = [&](double a, double b, double c, double l) {
    return (((0. + a) + (l1 ? l : b)) + (l1 ? b : (l2 ? l : c))) + (l3 ? c : l);
  };
  if (sel == 0u) {
    v = w;
  } else {
    v.x = ordered(kA * yA.x, kB * yB.x, kC * yC.x, kL * w.x);
    v.y = ordered(kA * yA.y, kB * yB.y, kC * yC.y, kL * w.y);
    v.z = ordered(kA * yA.z, kB * yB.z, kC * yC.z, kL * w.z);
    v *= 1. / ordered(kA, kB, kC, kL);
  }
  bits = 1u << f;
  work_w(W, f) = kL;
  if (sel & 1u) {
    bits |= 1u << sA;
    work_w(W, sA) = kA;
  }
  if (sel & 2u) {
    bits |= 1u << sB;
    work_w(W, sB) = kB;
  }
  if (sel & 4u) {
    bits |= 1u << sC;
    work_w(W, sC) = kC;
  }
  return true;
}

// degenerate (Convex.cpp:418-435)
DEM_HD bool j_degenerate(const GjkWork& W, unsigned all_bits, const d3& w) {
  bool deg = false;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (all_bits & (1u << i)) {
      const d3 y = work_y(W, i);
      if (y.x == w.x && y.y == w.y && y.z == w.z) deg = true;
    }
  return deg;
}

// computePoints (Convex.cpp:310-327) for the kept subset and its weights
DEM_HD void j_points(const GjkWork& W, unsigned bits, d3& p1, d3& p2) {
  double sum = 0.;
  p1 = d3{0., 0., 0.};
  p2 = d3{0., 0., 0.};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (bits & (1u << i)) {
      const double l = work_w(W, i);
      sum += l;
      p1 += l * work_get(W, 12 + 3 * i);
      p2 += l * work_get(W, 24 + 3 * i);
    }
  const double s = 1. / sum;
  p1 *= s;
  p2 *= s;
}

// Nesterov direction of closest_points (Convex.cpp:575-585; GJK_SV.cpp:479-489)
DEM_HD d3 nesterov_dir(int it, d3 d, d3 v, d3 w) {
  const double momentum = it / (it + 2.), omm = 1. - momentum;
  return momentum * d + momentum * omm * v + omm * omm * w;
}

// The search direction, support points and optimality-gap test of one
// iteration, with the tolerance and acceleration of o: 1 to go on with the
// support points P, Q (local frames) and w, 0 when the loop ends, 2 (sep >= 0,
// acceleration off) as soon as the support point w proves the distance larger
// than sep (the lower bound v.w / |v| of the distance exceeds it, with a
// margin above the rounding of v.w), so that a pair that cannot be in
// contact stops at once; the distance itself is then not computed.
DEM_HD int gjk_search(const ConvexGeo& A, const Tf& a2w, const ConvexGeo& B, const Tf& b2w, const GjkOpts& o,
                      int it, d3 v, double dist, double sep, d3& d, d3& w, bool& accel, d3& P, d3& Q) {
  const double relError = o.tol, absError = 1.e-4 * relError;
  d = (accel && it % 8 != 0) ? nesterov_dir(it, d, v, w) : v;
  P = support(A, tf_vec_basis(-d, a2w));
  Q = support(B, tf_vec_basis(d, b2w));
  w = tf_apply(a2w, P) - tf_apply(b2w, Q);
  if (sep >= 0. && !o.accel && dot(v, w) > sep * dist + 1.e-12 * dist * (fabs(w.x) + fabs(w.y) + fabs(w.z)))
    return 2;
  const double mu = dist - dot(v, w) / dist;
  if (mu < dist * relError || mu < absError) {
    if (!accel) return 0;
    if (norm(d - v) < kEps) return 0;
    accel = false;
    P = support(A, tf_vec_basis(-v, a2w));
    Q = support(B, tf_vec_basis(v, b2w));
    w = tf_apply(a2w, P) - tf_apply(b2w, Q);
  }
  return 1;
}

// --- Signed-volume sub-distance (GJK_SV.cpp:1-420) --------------------------
// Montanari, Petrinic and Barbieri (2017): the closest point of the simplex
// from signed volumes of its sub-simplices in the projection of largest
// area, recursing into the faces (edges) whose volume disagrees in sign.
// The points are named by their slot bits as in Johnson's; every slot index
// is a template argument so that the simplex lives in registers.
// Barycentric weights of the four slots, as named scalars (an array of
// them, written through references, would sit in scratch memory).
struct L4 {
  double w0, w1, w2, w3;
};
template <int I>
DEM_HD double& lw(L4& l) {
  if constexpr (I == 0) return l.w0;
  else if constexpr (I == 1) return l.w1;
  else if constexpr (I == 2) return l.w2;
  else return l.w3;
}

struct SvSimplex {
  d3 y[4];
  L4 lam;
};

DEM_HD bool sv_same_sign(double a, double b) { return !((a > 0) ^ (b > 0)); }
// sum of lam_i y_i over the slots of bits, in slot order
DEM_HD d3 sv_point(const d3 (&y)[4], unsigned bits, const L4& l) {
  d3 v{0., 0., 0.};
  if (bits & 1u) v += l.w0 * y[0];
  if (bits & 2u) v += l.w1 * y[1];
  if (bits & 4u) v += l.w2 * y[2];
  if (bits & 8u) v += l.w3 * y[3];
  return v;
}

// component i of v (0, 1, 2) selected among the values
DEM_HD double sel3(int i, d3 v) { return i == 0 ? v.x : (i == 1 ? v.y : v.z); }
// c ? a : b component by component (a select of values: a select of the
// addresses of a and b would keep them in scratch memory)
DEM_HD d3 pick(bool c, d3 a, d3 b) { return d3{c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z}; }
// a and b equal bit for bit (signed zeros told apart)
DEM_HD bool same_bits(d3 a, d3 b) {
  return __builtin_bit_cast(unsigned long long, a.x) == __builtin_bit_cast(unsigned long long, b.x) &&
         __builtin_bit_cast(unsigned long long, a.y) == __builtin_bit_cast(unsigned long long, b.y) &&
         __builtin_bit_cast(unsigned long long, a.z) == __builtin_bit_cast(unsigned long long, b.z);
}

// The sub-distance works on the active points gathered in slot order into
// named values (a, b, c, ...): one copy of the edge, triangle and
// tetrahedron code each, the faces (edges) to recurse into picked by a loop
// that is not unrolled.  The arithmetic is the slot-indexed one's, in the
// same order.  Each returns the mask of the points it keeps (bit k = k-th
// point) and writes their weights; a dropped point's weight is undefined.

// the point of the edge a-b closest to the origin (GJK_SV.cpp:19-93)
DEM_HD unsigned sv_edge(const d3& a, const d3& b, double& la, double& lb) {
  const d3 t = b - a;
  int I = 0;
  double neg_tI = -t.x;
  if (fabs(t.y) > fabs(neg_tI)) {
    I = 1;
    neg_tI = -t.y;
  }
  if (fabs(t.z) > fabs(neg_tI)) {
    I = 2;
    neg_tI = -t.z;
  }
  const double y2I = sel3(I, b), y1I = sel3(I, a);
  const double pI = dot(b, t) / dot(t, t) * neg_tI + y2I;
  const double C0 = -y2I + pI, C1 = y1I - pI;
  const bool s0 = sv_same_sign(neg_tI, C0), s1 = sv_same_sign(neg_tI, C1);
  const bool both = s0 && s1;
  la = both ? C0 / neg_tI : 1.;
  lb = both ? C1 / neg_tI : 1.;
  return both ? 3u : (s0 ? 1u : 2u);
}

// the triangle a-b-c (GJK_SV.cpp:99-228); the edges without a point whose
// signed area disagrees in sign are tried in point order, the closest kept
// (GJK_SV.cpp:190-225)
DEM_HD unsigned sv_tri(const d3& a, const d3& b, const d3& c, double& la, double& lb, double& lc) {
  const d3 n = cross(b - a, c - a);
  const d3 p0 = (dot(a, n) / dot(n, n)) * n;
  int ix = 1, iy = 2;
  double mu_max = (b.y * c.z + a.y * b.z + c.y * a.z - b.y * a.z - c.y * b.z - a.y * c.z);
  double mu = (b.z * a.x + c.z * b.x + a.z * c.x - b.z * c.x - a.z * b.x - c.z * a.x);
  if (fabs(mu) > fabs(mu_max)) {
    mu_max = mu;
    ix = 0;
  }
  mu = (b.x * c.y + a.x * b.y + c.x * a.y - b.x * a.y - c.x * b.y - a.x * c.y);
  if (fabs(mu) > fabs(mu_max)) {
    mu_max = mu;
    ix = 0;
    iy = 1;
  }
  const double px = sel3(ix, p0), py = sel3(iy, p0);
  const double y0x = sel3(ix, a), y0y = sel3(iy, a), y1x = sel3(ix, b), y1y = sel3(iy, b), y2x = sel3(ix, c),
               y2y = sel3(iy, c);
  const double C0 = (px * y1y + py * y2x + y1x * y2y - px * y2y - py * y1x - y2x * y1y);
  const double C1 = (px * y2y + py * y0x + y2x * y0y - px * y0y - py * y2x - y0x * y2y);
  const double C2 = (px * y0y + py * y1x + y0x * y1y - px * y1y - py * y0x - y1x * y0y);
  const bool s0 = sv_same_sign(mu_max, C0), s1 = sv_same_sign(mu_max, C1), s2 = sv_same_sign(mu_max, C2);
  if (s0 && s1 && s2) {
    la = C0 / mu_max;
    lb = C1 / mu_max;
    lc = C2 / mu_max;
    return 7u;
  }
  la = lb = lc = 0.;
  double dbest = 1.e9;
  unsigned best = 0;
#pragma nounroll
  for (int j = 0; j < 3; ++j) {
    if (j == 0 ? s0 : (j == 1 ? s1 : s2)) continue;
    // the edge without point j, its points in order
    const d3 e0 = pick(j == 0, b, a), e1 = pick(j == 2, b, c);
    double w0, w1;
    const unsigned k = sv_edge(e0, e1, w0, w1);
    d3 np{0., 0., 0.};
    if (k & 1u) np += w0 * e0;
    if (k & 2u) np += w1 * e1;
    const double ds = dot(np, np);
    if (ds < dbest) {
      dbest = ds;
      const unsigned m0 = j == 0 ? 2u : 1u, m1 = j == 2 ? 2u : 4u;
      best = ((k & 1u) ? m0 : 0u) | ((k & 2u) ? m1 : 0u);
      la = j == 0 ? la : w0;
      lb = j == 0 ? w0 : (j == 2 ? w1 : lb);
      lc = j == 2 ? lc : w1;
    }
  }
  return best;
}

// the tetrahedron y0-y1-y2-y3 (GJK_SV.cpp:234-373), its faces tried in
// point order as the triangle's edges (GJK_SV.cpp:338-370)
DEM_HD unsigned sv_tet(const d3 (&y)[4], L4& lam) {
  const double C0 = y[3].x * y[2].y * y[1].z + y[2].x * y[1].y * y[3].z + y[1].x * y[3].y * y[2].z -
                    y[1].x * y[2].y * y[3].z - y[2].x * y[3].y * y[1].z - y[3].x * y[1].y * y[2].z;
  const double C1 = y[0].x * y[2].y * y[3].z + y[2].x * y[3].y * y[0].z + y[3].x * y[0].y * y[2].z -
                    y[3].x * y[2].y * y[0].z - y[2].x * y[0].y * y[3].z - y[0].x * y[3].y * y[2].z;
  const double C2 = y[3].x * y[1].y * y[0].z + y[1].x * y[0].y * y[3].z + y[0].x * y[3].y * y[1].z -
                    y[0].x * y[1].y * y[3].z - y[1].x * y[3].y * y[0].z - y[3].x * y[0].y * y[1].z;
  const double C3 = y[0].x * y[1].y * y[2].z + y[1].x * y[2].y * y[0].z + y[2].x * y[0].y * y[1].z -
                    y[2].x * y[1].y * y[0].z - y[1].x * y[0].y * y[2].z - y[0].x * y[2].y * y[1].z;
  const double dM = C0 + C1 + C2 + C3;
  const bool s0 = sv_same_sign(dM, C0), s1 = sv_same_sign(dM, C1), s2 = sv_same_sign(dM, C2),
             s3 = sv_same_sign(dM, C3);
  if (s0 && s1 && s2 && s3) {
    lam.w0 = C0 / dM;
    lam.w1 = C1 / dM;
    lam.w2 = C2 / dM;
    lam.w3 = C3 / dM;
    return 15u;
  }
  double dbest = 1.e9;
  unsigned best = 0;
#pragma nounroll
  for (int j = 0; j < 4; ++j) {
    if (j == 0 ? s0 : (j == 1 ? s1 : (j == 2 ? s2 : s3))) continue;
    // the face without point j: points q0 < q1 < q2
    const int q0 = j == 0 ? 1 : 0, q1 = j <= 1 ? 2 : 1, q2 = j <= 2 ? 3 : 2;
    const d3 f0 = pick(j == 0, y[1], y[0]), f1 = pick(j <= 1, y[2], y[1]), f2 = pick(j <= 2, y[3], y[2]);
    double w0, w1, w2;
    const unsigned k = sv_tri(f0, f1, f2, w0, w1, w2);
    d3 np{0., 0., 0.};
    if (k & 1u) np += w0 * f0;
    if (k & 2u) np += w1 * f1;
    if (k & 4u) np += w2 * f2;
    const double ds = dot(np, np);
    if (ds < dbest) {
      dbest = ds;
      best = ((k & 1u) ? 1u << q0 : 0u) | ((k & 2u) ? 1u << q1 : 0u) | ((k & 4u) ? 1u << q2 : 0u);
      lam.w0 = q0 == 0 ? w0 : lam.w0;
      lam.w1 = q0 == 1 ? w0 : (q1 == 1 ? w1 : lam.w1);
      lam.w2 = q1 == 2 ? w1 : (q2 == 2 ? w2 : lam.w2);
      lam.w3 = q2 == 3 ? w2 : lam.w3;
    }
  }
  return best;
}

// the point of slot k, selected among the values
DEM_HD d3 sv_slot(const d3 (&y)[4], int k) { return pick(k == 0, y[0], pick(k == 1, y[1], pick(k == 2, y[2], y[3]))); }
// weight w into slot k of lam
DEM_HD void sv_put(L4& lam, int k, double w) {
  lam.w0 = k == 0 ? w : lam.w0;
  lam.w1 = k == 1 ? w : lam.w1;
  lam.w2 = k == 2 ? w : lam.w2;
  lam.w3 = k == 3 ? w : lam.w3;
}

// sv_subalgorithm (GJK_SV.cpp:380-410) by the number of points of the
// simplex, its points taken in slot order
DEM_HD void sv_sub(const d3 (&y)[4], unsigned& bits, L4& lam) {
  const int n = __builtin_popcount(bits);
  if (n == 1) {
    sv_put(lam, __builtin_ctz(bits), 1.);
  } else if (n == 2) {
    const int k0 = __builtin_ctz(bits), k1 = 31 - __builtin_clz(bits);
    double w0, w1;
    const unsigned k = sv_edge(sv_slot(y, k0), sv_slot(y, k1), w0, w1);
    sv_put(lam, k0, w0);
    sv_put(lam, k1, w1);
    bits = ((k & 1u) ? 1u << k0 : 0u) | ((k & 2u) ? 1u << k1 : 0u);
  } else if (n == 3) {
    const int m = __builtin_ctz(~bits & 15u);
    const int q0 = m == 0 ? 1 : 0, q1 = m <= 1 ? 2 : 1, q2 = m <= 2 ? 3 : 2;
    double w0, w1, w2;
    const unsigned k = sv_tri(sv_slot(y, q0), sv_slot(y, q1), sv_slot(y, q2), w0, w1, w2);
    sv_put(lam, q0, w0);
    sv_put(lam, q1, w1);
    sv_put(lam, q2, w2);
    bits = ((k & 1u) ? 1u << q0 : 0u) | ((k & 2u) ? 1u << q1 : 0u) | ((k & 4u) ? 1u << q2 : 0u);
  } else {
    bits = sv_tet(y, lam);
  }
}

// The search of one iteration of closest_points_GJK_SV with the new point
// in slot LAST (a compile-time index, as in gjk_iter): 1 when the point
// joins the simplex (y[LAST] set, bits updated), 0 when the loop ends, 2
// when the pair is proven farther apart than sep.
// closest_points_GJK_SV (GJK_SV.cpp:428-525), tolerance and acceleration of
// A.opt; witness points in the local frames; returns the distance
DEM_HD double gjk_sv_closest(const ConvexGeo& A, const Tf& a2w, const ConvexGeo& B, const Tf& b2w, const GjkWork& W,
                             d3& pa, d3& pb, int& iters, double sep, bool* separated) {
  SvSimplex S;
  sfor<0, 4>([&](auto I) {
    constexpr int i = decltype(I)::value;
    S.y[i] = d3{0., 0., 0.};
  });
  S.lam = L4{0., 0., 0., 0.};
  unsigned bits = 0;
  const d3 zero{0., 0., 0.};
  d3 v = tf_apply(a2w, support(A, zero)) - tf_apply(b2w, support(B, zero));
  d3 w = v, d = v;
  bool accel = A.opt.accel != 0;
  double dist = norm(v);
  int it = 0;
  while (bits < 15 && dist > kEps2 && it < 1000) {
    ++it;
    const bool plain = !accel;
    const unsigned bits0 = bits;
    const d3 v0 = v;
    // the first free slot
    const int f = __builtin_ctz(~bits);
    d3 P, Q;
    const int go = gjk_search(A, a2w, B, b2w, A.opt, it, v, dist, sep, d, w, accel, P, Q);
    if (go == 2) {
      if (separated) *separated = true;
      iters = it;
      return dist;
    }
    if (!go) break;
    bool degen = false;
    sfor<0, 4>([&](auto I) {
      constexpr int i = decltype(I)::value;
      if ((bits & (1u << i)) && S.y[i].x == w.x && S.y[i].y == w.y && S.y[i].z == w.z) degen = true;
    });
    if (degen) break;
    sfor<0, 4>([&](auto I) {
      constexpr int i = decltype(I)::value;
      S.y[i] = pick(f == i, w, S.y[i]);
    });
    work_put(W, 12 + 3 * f, P);
    work_put(W, 24 + 3 * f, Q);
    bits |= 1u << f;
    // one copy of the sub-distance for every slot the point went to
    sv_sub(S.y, bits, S.lam);
    v = sv_point(S.y, bits, S.lam);
    dist = norm(v);
    // A step searched along v that drops its new point again and leaves v
    // bit for bit as it was is a fixed point: the next step sees the same
    // simplex and direction, so every step up to the cap repeats it, weights
    // included.  The loop ends here as it would at the cap (a body against
    // a long thin box meets this within ten steps).
    if (plain && bits == bits0 && same_bits(v, v0)) {
      it = 1000;
      break;
    }
  }
  pa = d3{0., 0., 0.};
  pb = d3{0., 0., 0.};
  sfor<0, 4>([&](auto I) {
    constexpr int i = decltype(I)::value;
    if (bits & (1u << i)) {
      pa += lw<i>(S.lam) * work_get(W, 12 + 3 * i);
      pb += lw<i>(S.lam) * work_get(W, 24 + 3 * i);
    }
  });
  iters = it;
  return dist;
}

// --- Bounding-volume pre-tests (OBB.cpp:144-198, OBC.cpp:226-363) -----------
// On the full transforms (RigidBodyWithCrust::isContactBVolume,
// RigidBodyWithCrust.cpp:1095-1100).

// separating-axis test of two OBBs (Gottschalk et al. 1996): the face
// normals of both and their nine cross products, with a 1e-6 margin on the
// absolute rotation
DEM_HD bool obb_overlap(const ConvexGeo& A, const ConvexGeo& B) {
  constexpr double kLowEps = 1.0e-6;
  const double a[3] = {A.obb.x, A.obb.y, A.obb.z}, b[3] = {B.obb.x, B.obb.y, B.obb.z};
  const d3 dc = B.o - A.o;
  double cen[3], ori[3][3], oa[3][3];
  for (int i = 0; i < 3; ++i) cen[i] = A.B[i] * dc.x + A.B[3 + i] * dc.y + A.B[6 + i] * dc.z;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      ori[i][j] = A.B[i] * B.B[j] + A.B[3 + i] * B.B[3 + j] + A.B[6 + i] * B.B[6 + j];
      oa[i][j] = fabs(ori[i][j]) + kLowEps;
    }
  for (int i = 0; i < 3; ++i)
    if (fabs(cen[i]) > (a[i] + b[0] * oa[i][0] + b[1] * oa[i][1] + b[2] * oa[i][2])) return false;
  for (int i = 0; i < 3; ++i)
    if (fabs(cen[0] * ori[0][i] + cen[1] * ori[1][i] + cen[2] * ori[2][i]) >
        (b[i] + a[0] * oa[0][i] + a[1] * oa[1][i] + a[2] * oa[2][i]))
      return false;
  for (int j = 0; j < 3; ++j)
    for (int i = 0; i < 3; ++i) {
      const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
      if (fabs(cen[i2] * ori[i1][j] - cen[i1] * ori[i2][j]) >
          (a[i1] * oa[i2][j] + a[i2] * oa[i1][j] + b[j1] * oa[i][j2] + b[j2] * oa[i][j1]))
        return false;
    }
  return true;
}

// OBC of a body from its OBB extents (Box/Polyhedron::computeBVolume): the
// axis along the extent closest to another one, height twice that extent,
// radius the norm of the two others; spheres: radius r, height 2r, axis x
DEM_HD void obc_of(const ConvexGeo& g, double& r, double& h, d3& e) {
  if (g.type == kShapeSphere) {
    r = g.r;
    h = 2. * g.r;
    e = d3{1., 0., 0.};
    return;
  }
  const double ex = g.obb.x, ey = g.obb.y, ez = g.obb.z;
  double xy = fabs(ex - ey);
  const double xz = fabs(ex - ez), yz = fabs(ey - ez);
  int z = xy < xz ? 2 : 1;
  xy = xy < xz ? xy : xz;
  z = xy < yz ? z : 0;
  const double ez2 = z == 0 ? ex : (z == 1 ? ey : ez);
  e = d3{z == 0 ? 1. : 0., z == 1 ? 1. : 0., z == 2 ? 1. : 0.};
  h = 2. * ez2;
  r = sqrt(ex * ex + ey * ey + ez * ez - ez2 * ez2);
}

// real roots of x^4 + b x^3 + c x^2 + d x + e: depressed quartic, the
// biquadratic case or Ferrari's resolvent cubic (OBC.cpp:143-222)
DEM_HD int quartic_roots(double b, double c, double d, double e, double (&sol)[4]) {
  int nb = 0;
  const double b2 = b * b;
  const double p = c - 3. * b2 / 8.;
  const double q = b2 * b / 8. - b * c / 2. + d;
  const double r = -3. * b2 * b2 / 256. + e - b * d / 4. + b2 * c / 16.;
  const double p2 = p * p;
  if (fabs(q) < kEps) {
    const double del = p2 / 4. - r;
    if (del < 0.) return 0;
    const double m1 = -p / 2. + sqrt(del), m2 = -p / 2. - sqrt(del);
    if (m1 > 0.) {
      sol[nb++] = sqrt(m1) - b / 4.;
      sol[nb++] = -sqrt(m1) - b / 4.;
    }
    if (m2 > 0.) {
      sol[nb++] = sqrt(m2) - b / 4.;
      sol[nb++] = -sqrt(m2) - b / 4.;
    }
    return nb;
  }
  const double u = -p2 / 36. - r / 3.;
  const double v = -p2 * p / 216. + r * p / 6. - q * q / 16.;
  const double del = u * u * u + v * v;
  double m;
  if (del < 0) {
    m = 2. * sqrt(-u) * cos(acos(v / sqrt(-u) / u) / 3.) - p / 3.;
  } else {
    m = cbrt(-v + sqrt(del));
    m = m - u / m - p / 3.;
  }
  if (m < 0.) return 0;
  const double sm = sqrt(m / 2.);
  const double f1 = -p / 2. - m / 2. - q / sm / 4.;
  const double f2 = f1 + q / sm / 2.;
  if (f1 > 0.) {
    sol[nb++] = sm + sqrt(f1) - b / 4.;
    sol[nb++] = sm - sqrt(f1) - b / 4.;
  }
  if (f2 > 0.) {
    sol[nb++] = -sm + sqrt(f2) - b / 4.;
    sol[nb++] = -sm - sqrt(f2) - b / 4.;
  }
  return nb;
}

// one ellipse step of the OBC test: the other cylinder's cap as an ellipse
// (semi-axis re) against this one's circle of radius rc; true when a point
// of the ellipse boundary lies outside the circle
DEM_HD bool obc_ellipse_apart(double x0, double yTop, double yBottom, double ez, double ey, double re, double rc) {
  if (__builtin_signbit(yTop) != __builtin_signbit(yBottom)) return false;
  const double y0 = fabs(yTop) > fabs(yBottom) ? yBottom : yTop;
  if (!(x0 * x0 + y0 * y0 / ez / ez > re * re)) return false;
  const double ey_sq = ey * ey;
  const double A = re * re * ey_sq * ey_sq;
  const double B = 2. * y0 * ez / re / ey_sq;
  const double C = x0 * x0 / A;
  const double D = y0 * y0 * ez * ez / A;
  double sint[4];
  const int nb = quartic_roots(-B, C + D - 1., B, -D, sint);
  const double sx = (0. < x0) - (x0 < 0.);
  for (int i = 0; i < 4; ++i)
    if (i < nb && __builtin_signbit(sint[i]) != __builtin_signbit(B)) {
      const double cost = -sx * sqrt(1. - sint[i] * sint[i]);
      const double ptX = x0 + re * cost;
      const double ptY = y0 + re * ez * sint[i];
      if (ptX * ptX + ptY * ptY > rc * rc) return true;
    }
  return false;
}

DEM_HD d3 basis_times(const double* B, d3 v) {
  return d3{B[0] * v.x + B[1] * v.y + B[2] * v.z, B[3] * v.x + B[4] * v.y + B[5] * v.z,
            B[6] * v.x + B[7] * v.y + B[8] * v.z};
}
DEM_HD d3 unit_of(d3 v) { return v / norm(v); }

// isContactBVolume(OBC, OBC) (OBC.cpp:226-363): shortest distance of the
// axes, projections of the two rectangles, then ellipse against circle
DEM_HD bool obc_overlap(const ConvexGeo& A, const ConvexGeo& B) {
  double r1, hh1, r2, hh2;
  d3 e1, e2l;
  obc_of(A, r1, hh1, e1);
  obc_of(B, r2, hh2, e2l);
  const double h1 = hh1 / 2., h2 = hh2 / 2.;
  const d3 eZ = basis_times(A.B, e1);
  const d3 e2 = basis_times(B.B, e2l);
  const d3 xPt = B.o - A.o;
  const d3 eX = unit_of(cross(e2, eZ));
  const d3 eY = unit_of(cross(eZ, eX));
  const double x = dot(eX, xPt), y = dot(eY, xPt), z = dot(eZ, xPt);
  const double ey = dot(eY, e2), ez = dot(eZ, e2);
  if (fabs(x) >= r1 + r2) return false;
  {
    const double s2 = y / ey;
    const double s1 = z + s2 * ez;
    if (fabs(s1) < h1 && fabs(s2) < h2) return true;
  }
  {
    const double fey = fabs(ey) + 1.e-5, fez = fabs(ez) + 1.e-5;
    if (fabs(y) > r1 + h2 * fey + r2 * fez) return false;
    if (fabs(z) > h1 + h2 * fez + r2 * fey) return false;
    if (fabs(y * ez - z * ey) > r2 + h1 * fey + r1 * fez) return false;
    if (fabs(y * ey + z * ez) > h2 + h1 * fez + r1 * fey) return false;
  }
  if (fabs(ez) < 0.99 && fabs(ez) > 0.01) {
    if (obc_ellipse_apart(x, y + h2 * ey, y - h2 * ey, ez, ey, r2, r1)) return false;
    const d3 eY2 = unit_of(cross(eX, e2));
    const double y2 = -dot(eY2, xPt);
    const double ey2 = dot(eY2, eZ);
    if (obc_ellipse_apart(-x, y2 + h1 * ey2, y2 - h1 * ey2, ez, ey2, r1, r2)) return false;
  }
  return true;
}

DEM_HD bool bv_overlap(const ConvexGeo& A, const ConvexGeo& B) {
  return A.opt.bv == 1 ? obb_overlap(A, B) : obc_overlap(A, B);
}

// A search under way: Johnson's GJK (Convex.cpp:536-627), one iteration per
// call, so that a wave can hand a lane whose search has ended the next pair.
struct GjkState {
  d3 v, w, d;  // current nearest point; last support point and direction (Nesterov)
  double dist;
  unsigned bits, all_bits;
  int it;
  bool accel;
};
DEM_HD void gjk_begin(const ConvexGeo& A, const Tf& a2w, const ConvexGeo& B, const Tf& b2w, GjkState& g) {
  const d3 zero{0., 0., 0.};
  g.v = tf_apply(a2w, support(A, zero)) - tf_apply(b2w, support(B, zero));
  g.w = g.d = g.v;
  g.accel = A.opt.accel != 0;
  g.dist = norm(g.v);
  g.bits = g.all_bits = 0u;
  g.it = 0;
}
// 1: go on; 0: the search has ended (g.dist, kept points in W); 2: the
// distance is proven larger than sep (>= 0)
DEM_HD int gjk_step(const ConvexGeo& A, const Tf& a2w, const ConvexGeo& B, const Tf& b2w, const GjkWork& W, double sep,
                    GjkState& g) {
  if (!(g.bits < 15u && g.dist > kEps2 && g.it < 1000)) return 0;
  ++g.it;
  // the first free slot
  const int f = __builtin_ctz(~g.bits);
  d3 P, Q;
  const int go = gjk_search(A, a2w, B, b2w, A.opt, g.it, g.v, g.dist, sep, g.d, g.w, g.accel, P, Q);
  if (go != 1) return go;
  if (j_degenerate(W, g.all_bits, g.w)) return 0;
  work_put(W, 3 * f, g.w);
  work_put(W, 12 + 3 * f, P);
  work_put(W, 24 + 3 * f, Q);
  g.all_bits = g.bits | (1u << f);
  if (!j_closest(W, g.bits, g.all_bits, f, g.w, g.v)) return 0;
  g.dist = norm(g.v);
  return 1;
}

// closest_points with Johnson's sub-distance (Convex.cpp:536-627), the
// tolerance and acceleration of A.opt; witness points in the local frames;
// returns the distance (sep >= 0: *separated set when the distance is
// proven larger than sep; the witness points are then not computed)
DEM_HD double gjk_johnson_closest(const ConvexGeo& A, const Tf& a2w, const ConvexGeo& B, const Tf& b2w,
                                  const GjkWork& W, d3& pa, d3& pb, int& iters, double sep, bool* separated) {
  GjkState g;
  gjk_begin(A, a2w, B, b2w, g);
  int go;
  while ((go = gjk_step(A, a2w, B, b2w, W, sep, g)) == 1) {
  }
  iters = g.it;
  if (go == 2) {
    if (separated) *separated = true;
    return g.dist;
  }
  j_points(W, g.bits, pa, pb);
  return g.dist;
}

// The GJK distance the system's options choose: the signed-volume
// sub-distance (GJK_SV) or Johnson's; johnson: Johnson's whatever the
// options (the ContactError recovery, RigidBodyWithCrust.cpp:545).
DEM_HD double gjk_closest(const ConvexGeo& A, const Tf& a2w, const ConvexGeo& B, const Tf& b2w, d3& pa, d3& pb,
                          int& iters, double sep = -1., bool* separated = nullptr, bool johnson = false) {
#if defined(__HIP_DEVICE_COMPILE__)
  const GjkWork W = A.work;
#else
  double area[kGjkWork];
  const GjkWork W{area, 1};
#endif
  if (A.opt.sv && !johnson) return gjk_sv_closest(A, a2w, B, b2w, W, pa, pb, iters, sep, separated);
  return gjk_johnson_closest(A, a2w, B, b2w, W, pa, pb, iters, sep, separated);
}

// General ClosestPoint path.  Returns 1 with the contact features (the
// caller tests d < 0), 0 when the circumscribed spheres (or, with the
// option, the bounding volumes) do not meet, -1 on ContactError (the
// crust-shrunk bodies intersect).
DEM_HD int closest_gjk(const ConvexGeo& A, const ConvexGeo& B, d3& P, d3& ov, double& d, int* iters = nullptr) {
  d3 gcagcb = A.o - B.o;
  if (!(norm(gcagcb) < A.circR + B.circR)) return 0;
  if (A.opt.bv && !bv_overlap(A, B)) return 0;
  Tf a2w = tf_scaled(A, A.scaling), b2w = tf_scaled(B, B.scaling);
  d3 pa, pb;
  int it;
  double distance = gjk_closest(A, a2w, B, b2w, pa, pb, it);
  if (iters) *iters = it;
  if (distance < kEps) return -1;
  pa = tf_apply(a2w, pa);
  pb = tf_apply(b2w, pb);
  d3 ba = pa - pb;
  P = pa / 2.0 + pb / 2.0;
  d3 o = ba / distance;
  round_small(o);
  o *= A.crust + B.crust - distance;
  ov = o;
  d = distance - (A.crust + B.crust);
  return 1;
}

// ClosestPoint_ErreurHandling(factor 10): false if still intersecting
DEM_HD bool recover_gjk(const ConvexGeo& A, const ConvexGeo& B, d3& P, d3& ov, double& d, int* iters = nullptr) {
  d3 sa, sb;
  double* as[3] = {&sa.x, &sa.y, &sa.z};
  double* bs[3] = {&sb.x, &sb.y, &sb.z};
  const double ae[3] = {A.bext.x, A.bext.y, A.bext.z}, be[3] = {B.bext.x, B.bext.y, B.bext.z};
  for (int a = 0; a < 3; ++a) {
    double x = ae[a] < kEps ? 1. : (ae[a] - 10. * A.crust) / ae[a];
    *as[a] = x > 0.5 ? x : 0.5;
    double y = be[a] < kEps ? 1. : (be[a] - 10. * B.crust) / be[a];
    *bs[a] = y > 0.5 ? y : 0.5;
  }
  Tf a2w = tf_scaled(A, sa), b2w = tf_scaled(B, sb);
  d3 pa, pb;
  int it;
  double distance = gjk_closest(A, a2w, B, b2w, pa, pb, it, -1., nullptr, true);
  if (iters) *iters = it;
  if (distance < kEps) return false;
  pa = tf_apply(a2w, pa);
  pb = tf_apply(b2w, pb);
  d3 ba = pa - pb;
  ba /= norm(ba);
  P = pa / 2.0 + pb / 2.0;
  double imposed = 1. * (A.crust + B.crust);
  ov = imposed * ba;
  d = -imposed;
  return true;
}

// The transforms of one attempt of the general ClosestPoint path: attempt 0
// crust-shrunk (closest_gjk), attempt 1 with the bodies shrunk by ten crusts
// (recover_gjk, the ContactError recovery).  False when the circumscribed
// spheres (or the bounding volumes) do not meet.
DEM_HD bool gjk_frames(const ConvexGeo& A, const ConvexGeo& B, int attempt, Tf& a2w, Tf& b2w) {
  d3 sa = A.scaling, sb = B.scaling;
  if (attempt == 0) {
    d3 gcagcb = A.o - B.o;
    if (!(norm(gcagcb) < A.circR + B.circR)) return false;
    if (A.opt.bv && !bv_overlap(A, B)) return false;
  } else {
    double* as[3] = {&sa.x, &sa.y, &sa.z};
    double* bs[3] = {&sb.x, &sb.y, &sb.z};
    const double ae[3] = {A.bext.x, A.bext.y, A.bext.z}, be[3] = {B.bext.x, B.bext.y, B.bext.z};
    for (int a = 0; a < 3; ++a) {
      double x = ae[a] < kEps ? 1. : (ae[a] - 10. * A.crust) / ae[a];
      *as[a] = x > 0.5 ? x : 0.5;
      double y = be[a] < kEps ? 1. : (be[a] - 10. * B.crust) / be[a];
      *bs[a] = y > 0.5 ? y : 0.5;
    }
  }
  a2w = tf_scaled(A, sa);
  b2w = tf_scaled(B, sb);
  return true;
}

// The contact features of an attempt from its search's distance and witness
// points (local frames): 1 with the features (d may be >= 0), 2 with the
// recovered features, -1 when the shrunk bodies intersect.
DEM_HD int gjk_features(const Tf& a2w, const Tf& b2w, int attempt, double crusts, double distance, d3 pa, d3 pb, d3& P,
                        d3& ov, double& d) {
  if (distance < kEps) return -1;
  pa = tf_apply(a2w, pa);
  pb = tf_apply(b2w, pb);
  d3 ba = pa - pb;
  P = pa / 2.0 + pb / 2.0;
  if (attempt == 0) {
    d3 o = ba / distance;
    round_small(o);
    o *= crusts - distance;
    ov = o;
    d = distance - crusts;
    return 1;
  }
  ba /= norm(ba);
  double imposed = 1. * crusts;
  ov = imposed * ba;
  d = -imposed;
  return 2;
}

// One attempt of the general ClosestPoint path (gjk_frames, the search,
// gjk_features); 0 when the pair is no contact (attempt 0); -1 on attempt 0:
// go on with attempt 1; on attempt 1: ContactError.
// early: attempt 0 stops as soon as the pair is proven farther apart than
// the crusts (no contact; the iteration count is then not the full run's,
// so a caller collecting statistics passes false).
DEM_HD int gjk_attempt(const ConvexGeo& A, const ConvexGeo& B, int attempt, d3& P, d3& ov, double& d,
                       int& iters, bool early = false) {
  Tf a2w, b2w;
  if (!gjk_frames(A, B, attempt, a2w, b2w)) return 0;
  const double crusts = A.crust + B.crust;
  d3 pa, pb;
  bool separated = false;
  double distance =
      gjk_closest(A, a2w, B, b2w, pa, pb, iters, early && attempt == 0 ? crusts : -1., &separated, attempt != 0);
  if (separated) return 0;
  return gjk_features(a2w, b2w, attempt, crusts, distance, pa, pb, P, ov, d);
}

// --- kinematics of non-spherical bodies --------------------------------------
DEM_HD d3 ang_acc3(d3 tbf, double cf, d3 I, d3 om) {
  return d3{tbf.x / (cf * I.x) + om.y * om.z * (I.y - I.z) / I.x, tbf.y / (cf * I.y) + om.z * om.x * (I.z - I.x) / I.y,
            tbf.z / (cf * I.z) + om.x * om.y * (I.x - I.y) / I.z};
}
DEM_HD void ssprk3_3(d3& vrot, d3 tbf, double cf, d3 I, double dt) {
  d3 K1 = ang_acc3(tbf, cf, I, vrot);
  K1 *= dt;
  d3 K2 = ang_acc3(tbf, cf, I, vrot + K1);
  K2 *= dt;
  d3 K3 = ang_acc3(tbf, cf, I, vrot + 0.25 * (K1 + K2));
  K3 *= dt;
  vrot += (K1 + K2 + 4. * K3) / 6.;
}
// basis <- R(q) basis
DEM_HD void compose_left(double* B, quat q) {
  const double qx = q.v.x, qy = q.v.y, qz = q.v.z, qw = q.w;
  for (int i = 0; i < 3; ++i) {
    double px = qy * B[6 + i] - qz * B[3 + i] + qw * B[i];
    double py = qz * B[i] - qx * B[6 + i] + qw * B[3 + i];
    double pz = qx * B[3 + i] - qy * B[i] + qw * B[6 + i];
    double pw = -qx * B[i] - qy * B[3 + i] - qz * B[6 + i];
    B[i] = qy * pz - qz * py - pw * qx + qw * px;
    B[3 + i] = qz * px - qx * pz - pw * qy + qw * py;
    B[6 + i] = qx * py - qy * px - pw * qz + qw * pz;
  }
}

}  // namespace dem

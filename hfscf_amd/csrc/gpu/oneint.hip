// One-electron integrals on the GPU: overlap S, kinetic T and nuclear attraction V of a single
// molecule, and their first-derivative contractions for the RHF gradient. They replace what hfscf
// computes on the CPU in OSOverlap, OSKinetic and OSNuclear and their first derivatives (hfscf:
// src/integrals/hfscf_osoverlap.cpp:10, hfscf_osnuclear.cpp:17-83, hfscf_osoverlapderiv1.cpp:8,
// hfscf_oskineticderiv1.cpp:8, hfscf_osnuclearderiv1.cpp:15): S and T from the 1-D overlap
// recursion, V from the McMurchie-Davidson Hermite coefficients E^{ij}_t and the Hermite Coulomb
// integrals R_tuv (Boys values from the device table), derivatives by the shifts
// d/dA_x |a> = 2 alpha |a + 1_x> - a_x |a - 1_x>.
//
// One kernel per pair class (la lb), everything unrolled so that the tables are registers. Sixteen
// lanes take a shell pair; a lane's item is a primitive pair and a slice of the nuclei. The sum
// over nuclei is taken in the Hermite basis, V_ab = sum_tuv E^{ab}_tuv (sum_C -Z_C R_tuv(P - C)), so
// a nucleus costs its R_tuv and one multiply-add per tuv, and the expansion to the components
// happens once per item. In the gradient the same Hermite sums give the derivatives with respect to
// A and to P (A and B together), and a nucleus's own derivative is one more contraction of R with
// the primitive pair's Hermite density. All blocks are Cartesian; the spherical basis enters by
// one transformation of the matrices (densities before, integrals after).
//
// Bound: FP64 VALU of R_tuv (the Boys step and the recursion). Measured per call, with the host's
// copies: (H2O)16 / cc-pVDZ S, T, V 0.54 ms (3.2 with one lane per pair and nucleus on tables in
// scratch); (H2O)8 / cc-pVDZ gradient terms 0.27 ms (7.9).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "boys.hpp"
#include "cart.hpp"
#include "context.hpp"
#include "coop.hpp"
#include "oneint.hpp"
#include "rys_grad.hpp"

namespace hfg {

namespace {

constexpr int kOneLanes = 16;   // lanes per shell pair
constexpr int kOneBlock = 64;   // threads per workgroup: four shell pairs
constexpr int kOneLdsAtoms = 1024;  // gradient sums of up to this many nuclei in LDS
// A primitive pair with exp(-ab/p |AB|^2) c_a c_b below this adds nothing to a double (the integrals
// are at most a few hundred times it): about half of a water cluster's primitive pairs. Not with coordinates
// beyond kOneFar or infinite, where the other factors overflow and the pair's NaN shows in the results.
constexpr double kOneTiny = 1e-40, kOneFar = 1e30;

HFG_HD int rsize(int n) { return (n + 1) * (n + 2) * (n + 3) / 6; }
HFG_HD int ridx(int t, int u, int v) {
    const int s = t + u + v;
    return s * (s + 1) * (s + 2) / 6 + (s - t) * (s - t + 1) / 2 + v;
}

// R_tuv(p, PC), t + u + v <= N (numbered as the Cartesian components of cart.hpp), by the recursion over the auxiliary order from
// R^(m)_000 = (-2p)^m F_m(p |PC|^2), one order at a time.
template <int N>
HFG_INLINE void hermite_r(double p, const double* pc, const double* tab, double* R) {
    double F[N + 1];
    boys_eval<N, double>(p * (pc[0] * pc[0] + pc[1] * pc[1] + pc[2] * pc[2]), tab, 1.0, F);
    double f = 1.0;
    sfor<N + 1>([&](auto m) {
        F[m] *= f;
        f *= -2.0 * p;
    });
    double prev[rsize(N)];
    prev[0] = F[N];
    sfor<N>([&](auto k) {
        constexpr int m = N - 1 - k;
        double cur[rsize(N - m)];
        cur[0] = F[m];
        sfor<rsize(N - m) - 1>([&](auto x0) {
            constexpr int x = x0 + 1, d = gdir(x), x1 = gminus(x, d), n1 = gexp(x1, d);
            double v = pc[d] * prev[x1];
            if constexpr (n1 > 0) v += (double)n1 * prev[gminus(x1, d)];
            cur[x] = v;
        });
        sfor<rsize(N - m)>([&](auto x) { prev[x] = cur[x]; });
    });
    sfor<rsize(N)>([&](auto x) { R[x] = prev[x]; });
}

// Hermite coefficients E^{ij}_t of one direction, i <= IM, j <= JM.
template <int IM, int JM>
struct Herm {
    static constexpr int NT = IM + JM + 1;
    double e[IM + 1][JM + 1][NT];
    HFG_INLINE void build(double o2p, double pa, double pb) {
        sfor<IM + 1>([&](auto i) {
            sfor<JM + 1>([&](auto j) {
                sfor<i + j + 1>([&](auto t) {
                    if constexpr (i == 0 && j == 0) {
                        e[0][0][0] = 1.0;
                    } else {
                        constexpr int si = i > 0 ? i - 1 : 0, sj = i > 0 ? (int)j : j - 1;
                        constexpr int top = si + sj;
                        double v = 0.0;
                        if constexpr (t > 0) v += o2p * e[si][sj][t - 1];
                        if constexpr (t <= top) v += (i > 0 ? pa : pb) * e[si][sj][t];
                        if constexpr (t + 1 <= top) v += (double)(t + 1) * e[si][sj][t + 1];
                        e[i][j][t] = v;
                    }
                });
            });
        });
    }
    // coefficient t of (i, j), 0 outside
    template <int I, int J, int T>
    HFG_INLINE double at() const {
        if constexpr (I < 0 || J < 0 || T < 0 || T > I + J)
            return 0.0;
        else
            return e[I][J][T];
    }
};

// 1-D overlaps s(i, j), i <= IM, j <= JM, of one direction.
template <int IM, int JM>
struct Overlap1 {
    double s[IM + 1][JM + 1];
    HFG_INLINE void build(double s00, double o2p, double pa, double pb) {
        s[0][0] = s00;
        sfor<IM>([&](auto i) {
            double v = pa * s[i][0];
            if constexpr (i > 0) v += (double)(int)i * o2p * s[i - 1][0];
            s[i + 1][0] = v;
        });
        sfor<JM>([&](auto j) {
            sfor<IM + 1>([&](auto i) {
                double v = pb * s[i][j];
                if constexpr (j > 0) v += (double)(int)j * o2p * s[i][j - 1];
                if constexpr (i > 0) v += (double)(int)i * o2p * s[i - 1][j];
                s[i][j + 1] = v;
            });
        });
    }
    // kinetic factor -1/2 <i| d2/dx2 |j> with the ket's exponent b
    template <int I, int J>
    HFG_INLINE double kin(double b) const {
        double v = b * (double)(2 * J + 1) * s[I][J] - 2.0 * b * b * s[I][J + 2];
        if constexpr (J > 1) v -= 0.5 * (double)(J * (J - 1)) * s[I][J - 2];
        return v;
    }
};

struct PrimPair {
    double a, b, p, P[3], PA[3], PB[3], K;  // K = exp(-ab/p |AB|^2) c_a c_b
};

HFG_INLINE PrimPair prim_pair(const OneArgs& g, const OneShell& A, const OneShell& B, int i, int j) {
    const double* ra = g.xyz + 3 * A.atom;
    const double* rb = g.xyz + 3 * B.atom;
    PrimPair pp;
    pp.a = g.alpha[A.po + i];
    pp.b = g.alpha[B.po + j];
    pp.p = pp.a + pp.b;
    const double ip = 1.0 / pp.p;
    double r2 = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        pp.P[d] = (pp.a * ra[d] + pp.b * rb[d]) * ip;
        pp.PA[d] = pp.P[d] - ra[d];
        pp.PB[d] = pp.P[d] - rb[d];
        r2 += (ra[d] - rb[d]) * (ra[d] - rb[d]);
    }
    pp.K = exp(-pp.a * pp.b * ip * r2) * g.coef[A.po + i] * g.coef[B.po + j];
    return pp;
}

// Slices of the nuclei per primitive pair, so that a shell pair's items fill its sixteen lanes.
HFG_INLINE int nuclear_slices(int nprim) { return nprim >= 48 ? 1 : nprim >= 4 ? 4 : kOneLanes; }

template <int LA, int LB>
__global__ __launch_bounds__(kOneBlock) void oneint_kernel(OneArgs g, const int2* __restrict__ pairs, int npairs) {
    constexpr int L = LA + LB, ca = ncart(LA), cb = ncart(LB), nab = ca * cb;
    const int k = blockIdx.x * (kOneBlock / kOneLanes) + threadIdx.x / kOneLanes, ln = threadIdx.x & (kOneLanes - 1);
    if (k >= npairs) return;  // whole groups of lanes: the shuffles below stay within a group
    const OneShell A = g.sh[pairs[k].x], B = g.sh[pairs[k].y];
    double Sb[nab], Tk[nab], Vb[nab];
    sfor<nab>([&](auto x) { Sb[x] = Tk[x] = Vb[x] = 0.0; });
    const int nprim = A.np * B.np, nsl = nuclear_slices(nprim);
    for (int x = ln; x < nprim * nsl; x += kOneLanes) {
        const int pr = x / nsl, sl = x - pr * nsl, i = pr / B.np;
        const PrimPair pp = prim_pair(g, A, B, i, pr - i * B.np);
        if (!(fabs(pp.K) >= g.tiny) && pp.K == pp.K) continue;  // a NaN is evaluated
        const double o2p = 0.5 / pp.p;
        if (sl == 0) {
            Overlap1<LA, LB + 2> s[3];
            const double s00 = sqrt(M_PI / pp.p);
            sfor<3>([&](auto d) { s[d].build(d == 2 ? s00 * pp.K : s00, o2p, pp.PA[d], pp.PB[d]); });
            sfor<nab>([&](auto ab) {
                constexpr int ga = ncum(LA - 1) + ab / cb, gb = ncum(LB - 1) + ab % cb;
                constexpr int ax = gexp(ga, 0), ay = gexp(ga, 1), az = gexp(ga, 2);
                constexpr int bx = gexp(gb, 0), by = gexp(gb, 1), bz = gexp(gb, 2);
                const double sx = s[0].s[ax][bx], sy = s[1].s[ay][by], sz = s[2].s[az][bz];
                Sb[ab] += sx * sy * sz;
                Tk[ab] += s[0].template kin<ax, bx>(pp.b) * sy * sz + sx * s[1].template kin<ay, by>(pp.b) * sz +
                          sx * sy * s[2].template kin<az, bz>(pp.b);
            });
        }
        double h[rsize(L)];  // sum_C -Z_C R_tuv
        sfor<rsize(L)>([&](auto t) { h[t] = 0.0; });
        for (int c = sl; c < g.natom; c += nsl) {
            const double pc[3] = {pp.P[0] - g.xyz[3 * c], pp.P[1] - g.xyz[3 * c + 1], pp.P[2] - g.xyz[3 * c + 2]};
            const double z = g.Z[c];
            double R[rsize(L)];
            hermite_r<L>(pp.p, pc, g.boys, R);
            sfor<rsize(L)>([&](auto t) { h[t] -= z * R[t]; });
        }
        const double pre = 4.0 * M_PI * o2p * pp.K;  // 2 pi / p
        Herm<LA, LB> E[3];
        sfor<3>([&](auto d) { E[d].build(o2p, pp.PA[d], pp.PB[d]); });
        sfor<nab>([&](auto ab) {
            constexpr int ga = ncum(LA - 1) + ab / cb, gb = ncum(LB - 1) + ab % cb;
            constexpr int nx = gexp(ga, 0) + gexp(gb, 0) + 1, ny = gexp(ga, 1) + gexp(gb, 1) + 1,
                          nz = gexp(ga, 2) + gexp(gb, 2) + 1;
            double v = 0.0;
            sfor<nx>([&](auto t) {
                sfor<ny>([&](auto u) {
                    double w = 0.0;
                    sfor<nz>([&](auto q) { w += E[2].e[gexp(ga, 2)][gexp(gb, 2)][q] * h[ridx(t, u, q)]; });
                    v += E[0].e[gexp(ga, 0)][gexp(gb, 0)][t] * E[1].e[gexp(ga, 1)][gexp(gb, 1)][u] * w;
                });
            });
            Vb[ab] += pre * v;
        });
    }
    // the group's sums, each element written by one lane to both triangles
    const int oa = g.cart_off[pairs[k].x], ob = g.cart_off[pairs[k].y];
    sfor<nab>([&](auto ab) {
        double s = Sb[ab], t = Tk[ab], v = Vb[ab];
#pragma unroll
        for (int o = kOneLanes / 2; o > 0; o >>= 1) {
            s += __shfl_xor(s, o);
            t += __shfl_xor(t, o);
            v += __shfl_xor(v, o);
        }
        if ((ab & (kOneLanes - 1)) == ln) {
            const size_t e = (size_t)(oa + ab / cb) * g.ncart + ob + ab % cb;
            const size_t f = (size_t)(ob + ab % cb) * g.ncart + oa + ab / cb;
            g.S[e] = s;
            g.S[f] = s;
            g.T[e] = t;
            g.T[f] = t;
            g.V[e] = v;
            g.V[f] = v;
        }
    });
}

// Gradient terms 2 D_ab d(T + V)_ab/dX - 2 Q_ab dS_ab/dX of the shell pairs, D and Q Cartesian and
// symmetric: a pair of two shells counts twice for its mirror. The workgroup's sums per nucleus
// live in LDS (in grad itself beyond kOneLdsAtoms nuclei); the lanes start at different nuclei, so
// their LDS additions fall on different addresses.
template <int LA, int LB>
__global__ __launch_bounds__(kOneBlock) void oneint_grad_kernel(OneArgs g, const int2* __restrict__ pairs, int npairs,
                                                                const double* __restrict__ D, const double* __restrict__ Q,
                                                                double* grad) {
    constexpr int L = LA + LB, ca = ncart(LA), cb = ncart(LB), nab = ca * cb;
    extern __shared__ double gs[];
    const bool lds = g.natom <= kOneLdsAtoms;
    auto add = [&](int e, double v) {
        if (lds)
            atomicAdd(&gs[e], v);
        else
            unsafeAtomicAdd(&grad[e], v);
    };
    if (lds)
        for (int x = threadIdx.x; x < 3 * g.natom; x += kOneBlock) gs[x] = 0.0;
    __syncthreads();
    const int ln = threadIdx.x & (kOneLanes - 1), per = kOneBlock / kOneLanes;
    for (int k = blockIdx.x * per + threadIdx.x / kOneLanes; k < npairs; k += gridDim.x * per) {
        const int sa = pairs[k].x, sb = pairs[k].y;
        const OneShell A = g.sh[sa], B = g.sh[sb];
        // weights of the block (larger shell index, smaller) as it is stored; read again at each use,
        // which leaves the registers to the d pairs' tables
        const double f0 = sa == sb ? 2.0 : 4.0;
        const bool in_order = sa >= sb;
        const size_t w0 = in_order ? (size_t)g.cart_off[sa] * g.ncart + g.cart_off[sb]
                                   : (size_t)g.cart_off[sb] * g.ncart + g.cart_off[sa];
        const int wr = in_order ? g.ncart : 1, wc = in_order ? 1 : g.ncart;
        auto weight = [&](const double* M, int ab) { return f0 * M[w0 + (size_t)(ab / cb) * wr + (ab % cb) * wc]; };
        double gA[3] = {0.0, 0.0, 0.0}, gB[3] = {0.0, 0.0, 0.0};
        const int nprim = A.np * B.np, nsl = nuclear_slices(nprim);
        for (int x = ln; x < nprim * nsl; x += kOneLanes) {
            const int pr = x / nsl, sl = x - pr * nsl, i = pr / B.np;
            const PrimPair pp = prim_pair(g, A, B, i, pr - i * B.np);
            if (!(fabs(pp.K) >= g.tiny) && pp.K == pp.K) continue;  // a NaN is evaluated
            const double o2p = 0.5 / pp.p, ta = 2.0 * pp.a;
            if (sl == 0) {
                Overlap1<LA + 1, LB + 2> s[3];
                const double s00 = sqrt(M_PI / pp.p);
                sfor<3>([&](auto d) { s[d].build(d == 2 ? s00 * pp.K : s00, o2p, pp.PA[d], pp.PB[d]); });
                sfor<nab>([&](auto ab) {
                    constexpr int ga = ncum(LA - 1) + ab / cb, gb = ncum(LB - 1) + ab % cb;
                    double sv[3], tv[3], ds[3], dt[3];
                    const double wd = weight(D, ab), wq = weight(Q, ab);
                    sfor<3>([&](auto d) {
                        constexpr int ia = gexp(ga, d), jb = gexp(gb, d);
                        sv[d] = s[d].s[ia][jb];
                        tv[d] = s[d].template kin<ia, jb>(pp.b);
                        ds[d] = ta * s[d].s[ia + 1][jb];
                        dt[d] = ta * s[d].template kin<ia + 1, jb>(pp.b);
                        if constexpr (ia > 0) {
                            ds[d] -= (double)ia * s[d].s[ia - 1][jb];
                            dt[d] -= (double)ia * s[d].template kin<ia - 1, jb>(pp.b);
                        }
                    });
                    sfor<3>([&](auto d) {
                        constexpr int e1 = (d + 1) % 3, e2 = (d + 2) % 3;
                        const double dS = ds[d] * sv[e1] * sv[e2];
                        const double dT = dt[d] * sv[e1] * sv[e2] + ds[d] * (tv[e1] * sv[e2] + sv[e1] * tv[e2]);
                        const double v = wd * dT - wq * dS;
                        gA[d] += v;
                        gB[d] -= v;
                    });
                });
            }
            // Hermite density of the primitive pair
            const double pre = 4.0 * M_PI * o2p * pp.K;
            Herm<LA + 1, LB> E[3];
            sfor<3>([&](auto d) { E[d].build(o2p, pp.PA[d], pp.PB[d]); });
            double w[rsize(L)];
            sfor<rsize(L)>([&](auto t) { w[t] = 0.0; });
            sfor<nab>([&](auto ab) {
                constexpr int ga = ncum(LA - 1) + ab / cb, gb = ncum(LB - 1) + ab % cb;
                const double f = pre * weight(D, ab);
                sfor<gexp(ga, 0) + gexp(gb, 0) + 1>([&](auto t) {
                    const double ft = f * E[0].e[gexp(ga, 0)][gexp(gb, 0)][t];
                    sfor<gexp(ga, 1) + gexp(gb, 1) + 1>([&](auto u) {
                        const double fu = ft * E[1].e[gexp(ga, 1)][gexp(gb, 1)][u];
                        sfor<gexp(ga, 2) + gexp(gb, 2) + 1>(
                            [&](auto q) { w[ridx(t, u, q)] += fu * E[2].e[gexp(ga, 2)][gexp(gb, 2)][q]; });
                    });
                });
            });
            double h[rsize(L + 1)];  // sum_C -Z_C R_tuv
            sfor<rsize(L + 1)>([&](auto t) { h[t] = 0.0; });
            const int cnt = (g.natom - sl + nsl - 1) / nsl;
            int c = cnt > 0 ? sl + nsl * ((int)threadIdx.x % cnt) : 0;
            for (int n = 0; n < cnt; ++n) {
                const double pc[3] = {pp.P[0] - g.xyz[3 * c], pp.P[1] - g.xyz[3 * c + 1], pp.P[2] - g.xyz[3 * c + 2]};
                const double z = g.Z[c];
                double R[rsize(L + 1)];
                hermite_r<L + 1>(pp.p, pc, g.boys, R);
                double dc[3] = {0.0, 0.0, 0.0};
                sfor<rsize(L)>([&](auto t) { sfor<3>([&](auto d) { dc[d] += w[t] * R[gplus(t, d)]; }); });
                sfor<rsize(L + 1)>([&](auto t) { h[t] -= z * R[t]; });
#pragma unroll
                for (int d = 0; d < 3; ++d) add(3 * c + d, z * dc[d]);
                c += nsl;
                if (c >= g.natom) c = sl;
            }
            // d/dP, and d/dA by the shifts of the bra; d/dB = d/dP - d/dA
            sfor<3>([&](auto d) {
                double dp = 0.0, da = 0.0;
                sfor<rsize(L)>([&](auto t) { dp += w[t] * h[gplus(t, d)]; });
                sfor<nab>([&](auto ab) {
                    constexpr int ga = ncum(LA - 1) + ab / cb, gb = ncum(LB - 1) + ab % cb;
                    constexpr int e1 = (d + 1) % 3, e2 = (d + 2) % 3;
                    constexpr int ia = gexp(ga, d), jb = gexp(gb, d);
                    double v = 0.0;
                    sfor<ia + jb + 2>([&](auto t) {
                        double ed = ta * E[d].template at<ia + 1, jb, t>();
                        if constexpr (ia > 0) ed -= (double)ia * E[d].template at<ia - 1, jb, t>();
                        double q1 = 0.0;
                        sfor<gexp(ga, e1) + gexp(gb, e1) + 1>([&](auto u) {
                            double q2 = 0.0;
                            sfor<gexp(ga, e2) + gexp(gb, e2) + 1>([&](auto q) {
                                constexpr int tu[3] = {d == 0 ? (int)t : e1 == 0 ? (int)u : (int)q,
                                                       d == 1 ? (int)t : e1 == 1 ? (int)u : (int)q,
                                                       d == 2 ? (int)t : e1 == 2 ? (int)u : (int)q};
                                q2 += E[e2].e[gexp(ga, e2)][gexp(gb, e2)][q] * h[ridx(tu[0], tu[1], tu[2])];
                            });
                            q1 += E[e1].e[gexp(ga, e1)][gexp(gb, e1)][u] * q2;
                        });
                        v += ed * q1;
                    });
                    da += weight(D, ab) * v;
                });
                da *= pre;
                gA[d] += da;
                gB[d] += dp - da;
            });
        }
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int o = kOneLanes / 2; o > 0; o >>= 1) {
                gA[d] += __shfl_xor(gA[d], o);
                gB[d] += __shfl_xor(gB[d], o);
            }
        if (ln < 3) {
            const double va = ln == 0 ? gA[0] : ln == 1 ? gA[1] : gA[2], vb = ln == 0 ? gB[0] : ln == 1 ? gB[1] : gB[2];
            add(3 * A.atom + ln, va);
            add(3 * B.atom + ln, vb);
        }
    }
    __syncthreads();
    if (lds)
        for (int x = threadIdx.x; x < 3 * g.natom; x += kOneBlock) unsafeAtomicAdd(&grad[x], gs[x]);
}

// Output-basis matrices from the Cartesian ones (blockIdx.y: S, T, V): one thread per element.
__global__ __launch_bounds__(256) void from_cart_kernel(const double* __restrict__ Mc, int nc, const SphTerms* __restrict__ terms,
                                                        int n, double* __restrict__ M) {
    const double* src = Mc + (size_t)blockIdx.y * nc * nc;
    double* dst = M + (size_t)blockIdx.y * n * n;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < n * n; e += gridDim.x * 256) {
        const int i = e / n, j = e - i * n;
        const SphTerms ti = terms[i], tj = terms[j];
        double v = 0.0;
        for (int x = 0; x < ti.n; ++x)
            for (int y = 0; y < tj.n; ++y) v += ti.w[x] * tj.w[y] * src[(size_t)ti.c[x] * nc + tj.c[y]];
        dst[e] = v;
    }
}

constexpr int kClassLa[6] = {2, 2, 2, 1, 1, 0}, kClassLb[6] = {2, 1, 0, 1, 0, 0};

// Shell pairs by class, L(x) >= L(y); first[k]..first[k + 1] are those of class k.
std::vector<int2> pairs_by_class(const hfg_ctx* c, int* first) {
    std::vector<int> of_l[3];
    for (int s = 0; s < c->nshell; ++s) of_l[c->L[s]].push_back(s);
    std::vector<int2> out;
    out.reserve((size_t)c->nshell * (c->nshell + 1) / 2);
    for (int k = 0; k < 6; ++k) {
        first[k] = (int)out.size();
        const bool same = kClassLa[k] == kClassLb[k];
        for (int a : of_l[kClassLa[k]])
            for (int b : of_l[kClassLb[k]]) {
                if (same && b > a) break;
                out.push_back(make_int2(a, b));
            }
    }
    first[6] = (int)out.size();
    return out;
}

// The classes as (la, lb, index, stream): (ss|, the longest, on the main stream, the others on two
// side streams of about its length.
#define HFG_ONE_CLASSES(X) X(1, 0, 4, 1) X(1, 1, 3, 2) X(0, 0, 5, 0) X(2, 2, 0, 1) X(2, 0, 2, 2) X(2, 1, 1, 2)

// The main stream and the two side streams that the classes run on, forked here.
struct OneStreams {
    hipStream_t s[3];
    hfg_ctx* c;
    hipError_t fork(hfg_ctx* ctx) {
        c = ctx;
        s[0] = c->stream;
        s[1] = c->side[0];
        s[2] = c->nside > 1 ? c->side[1] : c->side[0];
        hipError_t e = hipEventRecord(c->ev_fork, s[0]);
        for (int k = 1; k < 3 && e == hipSuccess; ++k) e = hipStreamWaitEvent(s[k], c->ev_fork, 0);
        return e;
    }
    hipError_t join() {
        hipError_t e = hipGetLastError();
        for (int k = 0; k < std::min(2, c->nside) && e == hipSuccess; ++k) {
            e = hipEventRecord(c->ev_join[k], c->side[k]);
            if (e == hipSuccess) e = hipStreamWaitEvent(s[0], c->ev_join[k], 0);
        }
        return e;
    }
};

}  // namespace

// S, T, V over the Cartesian functions (g.S, g.T, g.V).
static hipError_t launch_oneint(hfg_ctx* c, const OneArgs& g, const int2* pairs, const int* first) {
    constexpr int per = kOneBlock / kOneLanes;
    OneStreams st;
    if (hipError_t e = st.fork(c)) return e;
#define HFG_RUN(A, B, K, S)                                                                                       \
    if (const int n = first[K + 1] - first[K])                                                                    \
        hipLaunchKernelGGL((oneint_kernel<A, B>), dim3((n + per - 1) / per), dim3(kOneBlock), 0, st.s[S], g,       \
                           pairs + first[K], n);
    HFG_ONE_CLASSES(HFG_RUN)
#undef HFG_RUN
    return st.join();
}

static hipError_t launch_oneint_grad(hfg_ctx* c, const OneArgs& g, const int2* pairs, const int* first, const double* D,
                                     const double* Q, double* grad) {
    constexpr int per = kOneBlock / kOneLanes;
    OneStreams st;
    if (hipError_t e = st.fork(c)) return e;
    const size_t lds = g.natom <= kOneLdsAtoms ? 3 * sizeof(double) * g.natom : 0;
    // at most 1024 workgroups per class, so that their flushes stay few
#define HFG_RUN(A, B, K, S)                                                                                         \
    if (const int n = first[K + 1] - first[K])                                                                      \
        hipLaunchKernelGGL((oneint_grad_kernel<A, B>), dim3(std::min((n + per - 1) / per, 1024)), dim3(kOneBlock), lds, \
                           st.s[S], g, pairs + first[K], n, D, Q, grad);
    HFG_ONE_CLASSES(HFG_RUN)
#undef HFG_RUN
    return st.join();
}

}  // namespace hfg

namespace {

int one_fail(hfg_ctx* c, int code, const char* msg) {
    c->err = msg;
    return code;
}

}  // namespace

namespace hfg {

int one_upload(hfg_ctx* c, hfg::OneArgs& g) {
    if (!c->have_basis || !c->have_geom) return one_fail(c, HFG_ERR_ARG, "basis and geometry must be set first");
    if (c->batch || c->mols.size() != 1) return one_fail(c, HFG_ERR_ARG, "one-electron integrals: single-molecule contexts only");
    if ((int)c->Zn.size() != c->natom)
        return one_fail(c, HFG_ERR_ARG, "one-electron integrals: hfg_set_geometry was given no nuclear charges");
    std::vector<hfg::OneShell> sh(c->nshell);
    for (int s = 0; s < c->nshell; ++s)
        sh[s] = hfg::OneShell{c->L[s], c->nprim[s], c->prim_off[s], c->atom[s]};
    HFG_CHECK(c, hipSetDevice(c->device));
    HFG_CHECK(c, c->d_one_sh.upload(sh, c->stream));
    HFG_CHECK(c, c->d_one_alpha.upload(c->alpha, c->stream));
    HFG_CHECK(c, c->d_one_coef.upload(c->coef, c->stream));
    HFG_CHECK(c, c->d_one_xyz.upload(c->xyz, c->stream));
    HFG_CHECK(c, c->d_one_Z.upload(c->Zn, c->stream));
    g = hfg::OneArgs{};
    g.sh = c->d_one_sh.p;
    g.alpha = c->d_one_alpha.p;
    g.coef = c->d_one_coef.p;
    g.xyz = c->d_one_xyz.p;
    g.Z = c->d_one_Z.p;
    g.boys = c->d_boys.p;
    g.natom = c->natom;
    g.ncart = c->ncart;
    g.cart_off = c->d_cart_off.p;
    const bool near = std::all_of(c->xyz.begin(), c->xyz.end(), [](double x) { return std::fabs(x) < hfg::kOneFar; });
    g.tiny = near ? hfg::kOneTiny : 0.0;
    return HFG_OK;
}

}  // namespace hfg

extern "C" {

int hfg_oneint(hfg_ctx* c, double* S, double* T, double* V) {
    if (!c) return HFG_ERR_ARG;
    hfg::OneArgs g;
    if (int r = hfg::one_upload(c, g)) return r;
    int first[7];
    const std::vector<int2> pairs = hfg::pairs_by_class(c, first);
    HFG_CHECK(c, c->d_one_pairs.upload(pairs, c->stream));
    const size_t nn = (size_t)c->nbf * c->nbf, cc = (size_t)c->ncart * c->ncart;
    HFG_CHECK(c, c->d_one_buf.ensure(3 * cc + (c->pure ? 3 * nn : 0)));
    g.S = c->d_one_buf.p;
    g.T = g.S + cc;
    g.V = g.T + cc;
    HFG_CHECK(c, hfg::launch_oneint(c, g, c->d_one_pairs.p, first));
    const double* res = g.S;  // a Cartesian basis has them already
    std::vector<hfg::SphTerms> terms(c->pure ? c->nbf : 0);
    if (c->pure) {
        for (int s = 0; s < c->nshell; ++s)
            for (int k = 0; k < hfg::nfun(c->L[s], true); ++k) {
                hfg::SphTerms t = hfg::sph_terms(c->L[s], k);
                for (int x = 0; x < t.n; ++x) t.c[x] += c->cart_off[s];
                terms[c->pure_off[s] + k] = t;
            }
        HFG_CHECK(c, c->d_one_terms.upload(terms, c->stream));
        double* dst = g.S + 3 * cc;
        hipLaunchKernelGGL(hfg::from_cart_kernel, dim3((unsigned)std::min<size_t>(1024, (nn + 255) / 256), 3), dim3(256), 0,
                           c->stream, g.S, c->ncart, c->d_one_terms.p, c->nbf, dst);
        HFG_CHECK(c, hipGetLastError());
        res = dst;
    }
    double* out[3] = {S, T, V};
    for (int k = 0; k < 3; ++k)
        if (out[k]) HFG_CHECK(c, hipMemcpyAsync(out[k], res + k * nn, nn * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HFG_CHECK(c, hipStreamSynchronize(c->stream));
    return HFG_OK;
}

int hfg_oneint_gradient(hfg_ctx* c, const double* D, const double* Q, double* grad) {
    if (!c) return HFG_ERR_ARG;
    if (!D || !Q || !grad) return one_fail(c, HFG_ERR_ARG, "hfg_oneint_gradient: null argument");
    hfg::OneArgs g;
    if (int r = hfg::one_upload(c, g)) return r;
    int first[7];
    const std::vector<int2> pairs = hfg::pairs_by_class(c, first);
    HFG_CHECK(c, c->d_one_pairs.upload(pairs, c->stream));
    const size_t nn = (size_t)c->nbf * c->nbf, cc = (size_t)c->ncart * c->ncart;
    const int nout = 3 * c->natom;
    HFG_CHECK(c, c->d_one_buf.ensure(2 * nn + nout + (c->pure ? 2 * cc : 0)));
    double* dD = c->d_one_buf.p;
    double* dQ = dD + nn;
    double* dg = dQ + nn;
    HFG_CHECK(c, hipMemcpyAsync(dD, D, nn * sizeof(double), hipMemcpyHostToDevice, c->stream));
    HFG_CHECK(c, hipMemcpyAsync(dQ, Q, nn * sizeof(double), hipMemcpyHostToDevice, c->stream));
    HFG_CHECK(c, hipMemcpyAsync(dg, grad, nout * sizeof(double), hipMemcpyHostToDevice, c->stream));
    if (c->pure) {
        double* cart = dg + nout;
        for (int k = 0; k < 2; ++k)
            HFG_CHECK(c, hfg::launch_to_cart(k ? dQ : dD, c->d_mols.p, c->d_mol_cart.p, 1, c->max_ncart, c->d_cart_terms.p,
                                             cart + k * cc, c->stream));
        dD = cart;
        dQ = cart + cc;
    }
    HFG_CHECK(c, hfg::launch_oneint_grad(c, g, c->d_one_pairs.p, first, dD, dQ, dg));
    HFG_CHECK(c, hipMemcpyAsync(grad, dg, nout * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HFG_CHECK(c, hipStreamSynchronize(c->stream));
    return HFG_OK;
}

}  // extern "C"

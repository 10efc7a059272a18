// Second-derivative integrals contracted with the Coulomb and exchange densities, one kernel per
// angular-momentum class, by Rys quadrature (hfg_hessian_2e; hess2e.hip sets up and launches).
//
// A work item is a shell quartet (ab|cd) and a range of its primitive quartets. At a Rys node an
// integral is a product of three 1-D integrals, and a derivative acts on one direction's factor
// only, so with ten 1-D values per direction (I, its first derivatives with respect to A, B, C and
// the six second ones) every one of the 45 derivatives over (A, B, C) x (x, y, z) is one
// product; D follows from translational invariance. A workgroup of three wavefronts works on S
// primitive quartets ("slots") and RC nodes at a time:
//   a. per (slot, node, direction), one lane runs the 2-D recursion G(n, m) in registers;
//   b. per (slot, node, direction, m), one lane transfers from n to (a, b) and forms the six bra
//      values (I, A, B, AA, AB, BB);
//   c. per (slot, node, direction, a b), one lane transfers from m to (c, d) and stores the ten
//      values of every (a, b, c, d) of the direction as one 80-byte record;
//   d. wavefront k takes axis k: the six second derivatives along it and its nine products with the
//      next axis, 15 of the 45. Its lanes hold the Cartesian component quartets (several slots side
//      by side in the classes with few) and sum the unweighted derivatives over the item; the
//      classes with more than three component quartets per lane weight them at once instead.
// At the item's end the sums are weighted, reduced over the wavefront, expanded to the 12 x 12 block
// of the four centres and added to one of several copies of the result.
//
// One lane per component quartet forming Hermite convolutions and triple sums of its own lengths
// (the form before) issued 1.8 scalar instructions per vector instruction and took 1.18 s on (H2O)4 /
// cc-pVDZ; this form takes 27 ms (water 50 -> 0.76 ms). Bound: the LDS reads of step d in the classes with many
// components; in the s and p classes, which take most of the time ((ps|ps) 10 ms, (ss|ss) 7 alone), the load latency
// and the item's end, two block expansions and 156 global atomics per item, of which every shell quartet has one
// at least (59 million L2 atomic requests per call there, TCC_ATOMIC).
#pragma once
#include "common.hpp"
#include "oneint.hpp"
#include "rys.hpp"

namespace hfg {

constexpr int kHessBlock = 192;
constexpr int kHessRounds = 16;  // rounds of S primitive quartets per work item, at most

struct HessPair {
    int sa, sb;   // shells, L(sa) >= L(sb)
    int off, np;  // primitive pairs [off, off + np): np counts the significant ones (set on the device)
};

// Work items of one class: bra pairs [b0, b0 + nb) against ket pairs [k0, k0 + nk) (or, when tri, the
// pairs k <= b of one range), each shell quartet in `chunks` items; item0 is the segment's first item.
struct HessSegment {
    int b0, nb, k0, nk, tri, chunks;
    long long item0;
};

struct HessArgs {
    const OneShell* sh;
    const double* alpha;
    const double* coef;
    const double* xyz;
    const double* rys;
    HessPair* pairs;
    double4* hp0;         // {p, P}
    double4* hp1;         // {K, alpha, beta, 1/2p}, K = exp(-ab/p |AB|^2) c_a c_b sqrt(2 pi^2.5) / p
    const int* cart_off;  // first Cartesian function of each shell
    int ncart, natom, npairs;
    const double* Dc;     // ncart x ncart density over the Cartesian functions
    double prim_cut;      // primitive quartets with |prefactor| below it are skipped
    double kmin;          // primitive pairs with |K| below it reach it with none
    double* H;            // copies of {HC, HX}, each (3 natom)^2, upper triangles
    int copies;
    const HessSegment* segs;
    int nsegs;
    long long nitems;
    unsigned long long* queue;
};

template <int LA, int LB, int LC, int LD>
struct RysHessShape {
    static constexpr int L = LA + LB + LC + LD;
    static constexpr int NR = (L + 2) / 2 + 1;
    static constexpr int NN = LA + LB + 3, NM = LC + LD + 3;
    static constexpr int NAB = (LA + 1) * (LB + 1), NCD = (LC + 1) * (LD + 1), NX = NAB * NCD;
    static constexpr int ca = ncart(LA), cb = ncart(LB), cc = ncart(LC), cd = ncart(LD);
    static constexpr int NCOMP = ca * cb * cc * cd;
    static constexpr int ND = ca * cb + cc * cd + ca * cc + ca * cd + cb * cc + cb * cd;
    // step c's records over step a's G, step b's values; doubles per direction and node
    static constexpr int TS = 10 * NX > NN * NM ? 10 * NX : NN * NM + (NN * NM) % 2, JS = 6 * NAB * NM;
    static constexpr int kPool = 6600;  // three workgroups on a CU's 160 KB of LDS
    static constexpr int RC = 3 * NR * (TS + JS) <= kPool ? NR : 3 * (NR + 1) / 2 * (TS + JS) <= kPool ? (NR + 1) / 2 : 1;
    static constexpr int RD = 3 * RC;
    static constexpr int fit = kPool / (RD * (TS + JS));
    static constexpr int ncpad = NCOMP > 32 ? 64 : NCOMP > 16 ? 32 : NCOMP > 8 ? 16 : NCOMP > 4 ? 8 : NCOMP > 2 ? 4 : NCOMP;
    static constexpr int side = 64 / ncpad;  // slots side by side in a wavefront
    static constexpr int S = fit >= 32 ? 32 : fit >= 16 ? 16 : fit >= 8 ? 8 : fit >= 4 ? 4 : fit >= 2 ? 2 : 1;
    static constexpr int CR = (NCOMP + 63) / 64;    // component quartets per lane
    static constexpr bool kLate = CR <= 2;          // weight at the item's end
};

// One primitive pair per lane, a wavefront per shell pair: the significant ones are stored first to
// last without gaps and counted.
__global__ void hess_prim_kernel(HessArgs g);

// Sums 32 values over the wavefront; afterwards lane l holds value 16 b5 + 8 b4 + 4 b3 + 2 b2 + b1 of
// its bits (each exchange step leaves a lane with half of the values).
HFG_INLINE double hess_reduce32(double* v) {
    const int lane = threadIdx.x & 63;
    sfor<5>([&](auto step) {
        constexpr int n = 16 >> step, o = 32 >> step;
        const bool up = lane & o;
        sfor<n>([&](auto k) {
            const double send = up ? v[k] : v[k + n], keep = up ? v[k + n] : v[k];
            v[k] = keep + __shfl_xor(send, o);
        });
    });
    return v[0] + __shfl_xor(v[0], 1);
}

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(kHessBlock) void rys_hess_kernel(HessArgs g) {
    using Sh = RysHessShape<LA, LB, LC, LD>;
    constexpr int S = Sh::S, NR = Sh::NR, RC = Sh::RC, RD = Sh::RD, NN = Sh::NN, NM = Sh::NM, NAB = Sh::NAB,
                  NCD = Sh::NCD, NCOMP = Sh::NCOMP, TS = Sh::TS, JS = Sh::JS;
    constexpr int ca = Sh::ca, cb = Sh::cb, cc = Sh::cc, cd = Sh::cd;
    __shared__ __align__(16) double Tb[S * RD * TS];
    __shared__ double Jb[S * RD * JS];
    __shared__ double Db[Sh::ND];
    __shared__ int2 cinfo[NCOMP];  // 1-D record indices, density-block indices
    __shared__ double M[2][81];    // the item's 9 x 9 blocks over (A, B, C) x (x, y, z)
    __shared__ double sz[S][3];    // 2 alpha, 2 beta, 2 gamma
    __shared__ int act[S];
    __shared__ long long next_item;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int c = tid; c < NCOMP; c += kHessBlock) {
        const int ia = c / (cb * cc * cd), ib = (c / (cc * cd)) % cb, ic = (c / cd) % cc, id = c % cd;
        int x = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int o = ((cart_exp(LA, ia, d) * (LB + 1) + cart_exp(LB, ib, d)) * (LC + 1) + cart_exp(LC, ic, d)) * (LD + 1) +
                          cart_exp(LD, id, d);
            x |= o << (8 * d);
        }
        cinfo[c] = make_int2(x, ia | (ib << 3) | (ic << 6) | (id << 9));
    }
    const int n3 = 3 * g.natom;
    for (;;) {
        __syncthreads();  // the previous item's end has read M and next_item
        if (tid == 0) next_item = (long long)atomicAdd(g.queue, 1ull);
        __syncthreads();
        const long long item = next_item;
        if (item >= g.nitems) break;
        int sg = 0;
        while (sg + 1 < g.nsegs && g.segs[sg + 1].item0 <= item) ++sg;
        const HessSegment seg = g.segs[sg];
        const long long rel = item - seg.item0;
        const int chunk = (int)(rel % seg.chunks);
        const long long qi = rel / seg.chunks;
        int ib_, ik_;
        if (seg.tri) {  // pair index qi of the triangle k <= b
            ib_ = (int)((sqrt(8.0 * (double)qi + 1.0) - 1.0) * 0.5);
            while ((long long)(ib_ + 1) * (ib_ + 2) / 2 <= qi) ++ib_;
            while ((long long)ib_ * (ib_ + 1) / 2 > qi) --ib_;
            ik_ = (int)(qi - (long long)ib_ * (ib_ + 1) / 2);
        } else {
            ib_ = (int)(qi / seg.nk);
            ik_ = (int)(qi - (long long)ib_ * seg.nk);
        }
        const int P = seg.b0 + ib_, Q = seg.k0 + ik_;
        const HessPair bp = g.pairs[P], kp = g.pairs[Q];
        const int nprim = bp.np * kp.np;
        const int first = chunk * (S * kHessRounds), last = min(nprim, first + S * kHessRounds);
        if (first >= last) continue;  // uniform over the workgroup
        const OneShell A = g.sh[bp.sa], B = g.sh[bp.sb], C = g.sh[kp.sa], D = g.sh[kp.sb];
        const double* ra = g.xyz + 3 * A.atom;
        const double* rb = g.xyz + 3 * B.atom;
        const double* rc = g.xyz + 3 * C.atom;
        const double* rd_ = g.xyz + 3 * D.atom;
        {
            const int oa = g.cart_off[bp.sa], ob = g.cart_off[bp.sb], oc = g.cart_off[kp.sa], od = g.cart_off[kp.sb];
            constexpr int n1 = ca * cb, n2 = n1 + cc * cd, n3_ = n2 + ca * cc, n4 = n3_ + ca * cd, n5 = n4 + cb * cc;
            for (int e = tid; e < Sh::ND; e += kHessBlock) {
                int r, c;
                if (e < n1) {
                    r = oa + e / cb;
                    c = ob + e % cb;
                } else if (e < n2) {
                    r = oc + (e - n1) / cd;
                    c = od + (e - n1) % cd;
                } else if (e < n3_) {
                    r = oa + (e - n2) / cc;
                    c = oc + (e - n2) % cc;
                } else if (e < n4) {
                    r = oa + (e - n3_) / cd;
                    c = od + (e - n3_) % cd;
                } else if (e < n5) {
                    r = ob + (e - n4) / cc;
                    c = oc + (e - n4) % cc;
                } else {
                    r = ob + (e - n5) / cd;
                    c = od + (e - n5) % cd;
                }
                Db[e] = g.Dc[(size_t)r * g.ncart + c];
            }
        }
        double deg = 8.0;
        if (bp.sa == bp.sb) deg *= 0.5;
        if (kp.sa == kp.sb) deg *= 0.5;
        if (P == Q) deg *= 0.5;
        const double *Dab = Db, *Dcd = Dab + ca * cb, *Dac = Dcd + cc * cd, *Dad = Dac + ca * cc, *Dbc = Dad + ca * cd,
                     *Dbd = Dbc + cb * cc;
        auto weights = [&](int ci, double& gC, double& gX) {
            const int ia = ci & 7, ib = (ci >> 3) & 7, ic = (ci >> 6) & 7, id = ci >> 9;
            gC = deg * 2.0 * Dab[ia * cb + ib] * Dcd[ic * cd + id];
            gX = -deg * 0.5 * (Dac[ia * cc + ic] * Dbd[ib * cd + id] + Dad[ia * cd + id] * Dbc[ib * cc + ic]);
        };
        constexpr int NACC = Sh::kLate ? Sh::CR : 2;  // sets of 15: per component, or Coulomb and exchange
        double acc[NACC][15];
#pragma unroll
        for (int i = 0; i < NACC; ++i)
#pragma unroll
            for (int k = 0; k < 15; ++k) acc[i][k] = 0.0;
        for (int p0 = first; p0 < last; p0 += S)
            for (int r0 = 0; r0 < NR; r0 += RC) {
                // a. quadrature and 2-D recursion
                for (int v = tid; v < S * RD; v += kHessBlock) {
                    const int s = v / RD, rd = v - s * RD, d = rd / RC, r = r0 + rd - d * RC;
                    const int idx = p0 + s;
                    int ok = 0;
                    if (idx < last) {
                        const int ip = idx / kp.np, jp = idx - ip * kp.np;
                        const double4 a0 = g.hp0[bp.off + ip], a1 = g.hp1[bp.off + ip];
                        const double4 b0 = g.hp0[kp.off + jp], b1 = g.hp1[kp.off + jp];
                        const double p = a0.x, qe = b0.x;
                        const double rs = rsqrt(p + qe);
                        const double pfac = a1.x * b1.x * rs;
                        if (fabs(pfac) >= g.prim_cut) {
                            ok = 1;
                            if (r < NR) {  // a last group of nodes may be partly filled
                                const double PQ[3] = {a0.y - b0.y, a0.z - b0.z, a0.w - b0.w};
                                const double ipq = rs * rs, rp = qe * ipq, rq = p * ipq;
                                double u, wt;
                                rys_point<NR>(g.rys, p * rp * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]), r, u, wt);
                                const double pq = d == 0 ? PQ[0] : d == 1 ? PQ[1] : PQ[2];
                                const double pa = (d == 0 ? a0.y : d == 1 ? a0.z : a0.w) - ra[d];
                                const double qc = (d == 0 ? b0.y : d == 1 ? b0.z : b0.w) - rc[d];
                                rys_2d<NN, NM>(d == 2 ? pfac * wt : 1.0, pa - u * rp * pq, qc + u * rq * pq,
                                               a1.w * (1.0 - u * rp), b1.w * (1.0 - u * rq), 0.5 * u * ipq,
                                               Tb + (s * RD + rd) * TS);
                            }
                            if (rd == 0) {
                                sz[s][0] = 2.0 * a1.y;
                                sz[s][1] = 2.0 * a1.z;
                                sz[s][2] = 2.0 * b1.y;
                            }
                        }
                    }
                    if (rd == 0) act[s] = ok;
                }
                __syncthreads();
                // b. n -> (a, b) with the bra derivatives
                for (int v = tid; v < S * RD * NM; v += kHessBlock) {
                    const int sr = v / NM, m = v - sr * NM, s = sr / RD, d = (sr - s * RD) / RC;
                    if (!act[s]) continue;
                    const double AB = ra[d] - rb[d], za = sz[s][0], zb = sz[s][1];
                    const double* G = Tb + sr * TS + m * NN;
                    double h[LB + 3][NN];  // (b, n)
                    sfor<NN>([&](auto n) { h[0][n] = G[n]; });
                    sfor<LB + 2>([&](auto b) {
                        sfor<NN - 1 - b>([&](auto n) { h[b + 1][n] = h[b][n + 1] + AB * h[b][n]; });
                    });
                    double* J = Jb + sr * JS + m;
                    sfor<LA + 1>([&](auto i) {
                        sfor<LB + 1>([&](auto j) {
                            double dA = za * h[j][i + 1], dB = zb * h[j + 1][i];
                            double dAA = za * za * h[j][i + 2] - za * (double)(2 * i + 1) * h[j][i];
                            double dBB = zb * zb * h[j + 2][i] - zb * (double)(2 * j + 1) * h[j][i];
                            double dAB = za * zb * h[j + 1][i + 1];
                            if constexpr (i > 0) {
                                dA -= (double)(int)i * h[j][i - 1];
                                dAB -= zb * (double)(int)i * h[j + 1][i - 1];
                            }
                            if constexpr (j > 0) {
                                dB -= (double)(int)j * h[j - 1][i];
                                dAB -= za * (double)(int)j * h[j - 1][i + 1];
                            }
                            if constexpr (i > 0 && j > 0) dAB += (double)(i * j) * h[j - 1][i - 1];
                            if constexpr (i > 1) dAA += (double)(i * (i - 1)) * h[j][i - 2];
                            if constexpr (j > 1) dBB += (double)(j * (j - 1)) * h[j - 2][i];
                            constexpr int ab = i * (LB + 1) + j;
                            J[ab * NM] = h[j][i];
                            J[(NAB + ab) * NM] = dA;
                            J[(2 * NAB + ab) * NM] = dB;
                            J[(3 * NAB + ab) * NM] = dAA;
                            J[(4 * NAB + ab) * NM] = dAB;
                            J[(5 * NAB + ab) * NM] = dBB;
                        });
                    });
                }
                __syncthreads();
                // c. m -> (c, d) with the ket derivatives; records {I, A, B, C, AA, AB, BB, AC, BC, CC}
                for (int v = tid; v < S * RD * NAB; v += kHessBlock) {
                    const int sr = v / NAB, ab = v - sr * NAB, s = sr / RD, d = (sr - s * RD) / RC;
                    if (!act[s]) continue;
                    const double CD = rc[d] - rd_[d], zc = sz[s][2];
                    const double* J = Jb + sr * JS + ab * NM;
                    double* T = Tb + sr * TS + ab * NCD * 10;
                    sfor<6>([&](auto op) {
                        constexpr int n = op == 0 ? NM : op < 3 ? NM - 1 : NM - 2;  // values of m in use
                        double h[LD + 1][NM];
                        sfor<n>([&](auto m) { h[0][m] = J[op * NAB * NM + m]; });
                        sfor<LD>([&](auto l) {
                            sfor<n - 1 - l>([&](auto m) { h[l + 1][m] = h[l][m + 1] + CD * h[l][m]; });
                        });
                        sfor<LC + 1>([&](auto i) {
                            sfor<LD + 1>([&](auto j) {
                                double* t = T + (i * (LD + 1) + j) * 10;
                                constexpr int slot0 = op < 3 ? (int)op : op + 1;  // I A B . AA AB BB
                                t[slot0] = h[j][i];
                                if constexpr (op < 3) {
                                    double dC = zc * h[j][i + 1];
                                    if constexpr (i > 0) dC -= (double)(int)i * h[j][i - 1];
                                    t[op == 0 ? 3 : op + 6] = dC;
                                }
                                if constexpr (op == 0) {
                                    double dCC = zc * zc * h[j][i + 2] - zc * (double)(2 * i + 1) * h[j][i];
                                    if constexpr (i > 1) dCC += (double)(i * (i - 1)) * h[j][i - 2];
                                    t[9] = dCC;
                                }
                            });
                        });
                    });
                }
                __syncthreads();
                // d. the wavefront's 15 derivatives of the component quartets
                const int ay = wave == 2 ? 0 : wave + 1, az = wave == 0 ? 2 : wave - 1;
                auto add = [&](int s, int xyz, double* out) {
                    const double2* Tx = reinterpret_cast<const double2*>(
                        Tb + (s * RD + wave * RC) * TS + 10 * ((xyz >> (8 * wave)) & 255));
                    const double2* Ty = reinterpret_cast<const double2*>(
                        Tb + (s * RD + ay * RC) * TS + 10 * ((xyz >> (8 * ay)) & 255));
                    const double* Tz = Tb + (s * RD + az * RC) * TS + 10 * ((xyz >> (8 * az)) & 255);
#pragma unroll
                    for (int r = 0; r < RC; ++r) {
                        if (NR % RC != 0 && r0 + r >= NR) break;
                        const double2 xa = Tx[r * (TS / 2)], xb = Tx[r * (TS / 2) + 1], xc = Tx[r * (TS / 2) + 2],
                                      xd = Tx[r * (TS / 2) + 3], xe = Tx[r * (TS / 2) + 4];
                        const double2 ya = Ty[r * (TS / 2)], yb = Ty[r * (TS / 2) + 1];
                        const double z = Tz[r * TS];
                        const double yz = ya.x * z;
                        out[0] += xc.x * yz;
                        out[1] += xc.y * yz;
                        out[2] += xd.x * yz;
                        out[3] += xd.y * yz;
                        out[4] += xe.x * yz;
                        out[5] += xe.y * yz;
                        const double x1 = xa.y * z, x2 = xb.x * z, x3 = xb.y * z;
                        out[6] += x1 * ya.y;
                        out[7] += x1 * yb.x;
                        out[8] += x1 * yb.y;
                        out[9] += x2 * ya.y;
                        out[10] += x2 * yb.x;
                        out[11] += x2 * yb.y;
                        out[12] += x3 * ya.y;
                        out[13] += x3 * yb.x;
                        out[14] += x3 * yb.y;
                    }
                };
                if constexpr (Sh::CR == 1) {
                    const int c = lane & (Sh::ncpad - 1);
                    if (c < NCOMP) {
                        const int xyz = cinfo[c].x;
                        for (int s = lane / Sh::ncpad; s < S; s += Sh::side)
                            if (act[s]) add(s, xyz, acc[0]);
                    }
                } else if constexpr (Sh::kLate) {
                    for (int s = 0; s < S; ++s)
                        if (act[s])
#pragma unroll
                            for (int i = 0; i < NACC; ++i)
                                if (lane + 64 * i < NCOMP) add(s, cinfo[lane + 64 * i].x, acc[i]);
                } else {
                    for (int s = 0; s < S; ++s)
                        if (act[s])
                            for (int c = lane; c < NCOMP; c += 64) {
                                double t[15];
#pragma unroll
                                for (int k = 0; k < 15; ++k) t[k] = 0.0;
                                const int2 ci = cinfo[c];
                                add(s, ci.x, t);
                                double gC, gX;
                                weights(ci.y, gC, gX);
#pragma unroll
                                for (int k = 0; k < 15; ++k) {
                                    acc[0][k] += gC * t[k];
                                    acc[1][k] += gX * t[k];
                                }
                            }
                }
                __syncthreads();  // the slots' tables are rewritten by the next round
            }
        // the wavefront's sums into the 9 x 9 blocks
        {
            double v[32];
            if constexpr (Sh::kLate) {
#pragma unroll
                for (int k = 0; k < 32; ++k) v[k] = 0.0;
#pragma unroll
                for (int i = 0; i < NACC; ++i) {
                    const int c = Sh::CR == 1 ? (lane & (Sh::ncpad - 1)) : lane + 64 * i;
                    if (c < NCOMP) {
                        double gC, gX;
                        weights(cinfo[c].y, gC, gX);
#pragma unroll
                        for (int k = 0; k < 15; ++k) {
                            v[k] += gC * acc[i][k];
                            v[16 + k] += gX * acc[i][k];
                        }
                    }
                }
            } else {
#pragma unroll
                for (int k = 0; k < 15; ++k) {
                    v[k] = acc[0][k];
                    v[16 + k] = acc[1][k];
                }
            }
            v[15] = v[31] = 0.0;
            const double sum = hess_reduce32(v);
            const int k = ((lane >> 1) & 15), part = lane >> 5;
            // bits 5..1 of the lane name the value: bit 5 the part, bits 4..1 the derivative
            if (!(lane & 1) && k < 15) {
                const int ay = wave == 2 ? 0 : wave + 1;
                int x1, x2;
                if (k < 6) {  // AA AB BB AC BC CC
                    const int c1 = k == 0 || k == 1 || k == 3 ? 0 : k == 2 || k == 4 ? 1 : 2;
                    const int c2 = k == 0 ? 0 : k < 3 ? 1 : 2;
                    x1 = 3 * c1 + wave;
                    x2 = 3 * c2 + wave;
                } else {
                    x1 = 3 * ((k - 6) / 3) + wave;
                    x2 = 3 * ((k - 6) % 3) + ay;
                }
                M[part][x1 * 9 + x2] = sum;
                M[part][x2 * 9 + x1] = sum;
            }
        }
        __syncthreads();
        // the 12 x 12 block of the four centres (the D rows and columns -(A + B + C)), its upper
        // triangle, into this workgroup's copy of the upper triangles of HC and HX
        if (tid < 156) {
            const int part = tid / 78;
            int y1 = 0, e = tid - part * 78;
            while (e >= 12 - y1) {
                e -= 12 - y1;
                ++y1;
            }
            const int y2 = y1 + e;
            double v = 0.0;
            for (int c1 = 0; c1 < 3; ++c1) {
                if (y1 < 9 && c1 != y1 / 3) continue;
                for (int c2 = 0; c2 < 3; ++c2) {
                    if (y2 < 9 && c2 != y2 / 3) continue;
                    const double t = M[part][(3 * c1 + y1 % 3) * 9 + 3 * c2 + y2 % 3];
                    v += (y1 < 9) == (y2 < 9) ? t : -t;
                }
            }
            const int atoms[4] = {A.atom, B.atom, C.atom, D.atom};
            const int r = atoms[y1 / 3] * 3 + y1 % 3, c = atoms[y2 / 3] * 3 + y2 % 3;
            if (y1 != y2 && r == c) v *= 2.0;  // both orders fall on the diagonal
            double* H = g.H + ((size_t)(blockIdx.x % g.copies) * 2 + part) * n3 * n3;
            unsafeAtomicAdd(&H[(size_t)min(r, c) * n3 + max(r, c)], v);
        }
    }
}

template <int LA, int LB, int LC, int LD>
hipError_t launch_rys_hess_class(const HessArgs& g, hipStream_t s);

}  // namespace hfg

// FP64 adjoint gradient kernel of the classes from L = kRysGradMinL, by Rys quadrature.
//
// The register kernel (grad_impl.hpp) gives a lane a whole shell quartet; from L = 4 its VRR
// tables and shifted integrals no longer fit the registers (2.7-13 KB of scratch per lane), and the
// program kernel (coop_grad.hpp) from L = 7 runs one primitive quartet at a time with a barrier
// per recursion level. At a Rys node an integral is a product of three 1-D integrals, so the data
// between the recursion and the contraction is one table per direction, small enough for LDS, and
// every step is wide:
//   a. per primitive quartet ("slot", S of them at a time), node and direction, one lane runs the
//      2-D recursion G(n, m) in registers;
//   b. per (slot, node, direction, m), one lane transfers from n to (a, b) and forms the bra
//      values I, dI/dA, dI/dB (2 alpha I(a+1) - a I(a-1));
//   c. per (slot, node, direction, a b), one lane transfers from m to (c, d) and stores I, dI/dA,
//      dI/dB, dI/dC of every (a, b, c, d) of the direction as one 32-byte record;
//   d. a wavefront takes a slot: its lanes share the Cartesian component quartets, each reading
//      three records per node and adding the nine derivatives weighted with the Cartesian
//      two-particle density. The sums stay in registers while consecutive slots belong to one shell
//      quartet and are then reduced over the wavefront into the per-atom sums.
// The spherical basis enters only through the density, transformed to Cartesian functions
// once per gradient, so one kernel per class serves both basis types.
//
// Bound: LDS reads of step d (six 16-byte reads per component quartet and node against 15 FP64
// operations) and, in the classes with few components, the load latency of step a. Measured per whole
// gradient when every class from L = 4 moved here: (H2O)16 / cc-pVDZ 292 -> 171 ms (the (dp|dd), (dd|dp),
// (dd|dd) launches 83 ms each -> 4.5, 1.3, 0.1 ms; (dp|pp) 60 -> 28, (dd|pp) 45 -> 4.8, (dp|dp) 50 ->
// 2.8 ms, each among the other launches), water / 6-31G* 13.7 -> 1.45 ms; with the register kernel kept for
// many (dp|ps), (ds|pp), (ds|ds) and (dd|ss) quartets (grad_on_rys) (H2O)16 148 ms.
#pragma once
#include "grad_impl.hpp"
#include "rys.hpp"

namespace hfg {

struct RysGradArgs {
    GradArgs g;
    const double* rys;        // quadrature tables
    const double* Dc;         // densities over the Cartesian functions, concatenated
    const int* cart_off;      // global shell -> first Cartesian function in its molecule
    const MolCart* mol_cart;  // per molecule
};


constexpr int kRysChunk = 64;  // shell quartets enumerated at a time

template <int LA, int LB, int LC, int LD>
struct RysGradShape {
    static constexpr int L = LA + LB + LC + LD;
    static constexpr int NR = (L + 1) / 2 + 1;
    static constexpr int NN = LA + LB + 2, NM = LC + LD + 2;
    static constexpr int NAB = (LA + 1) * (LB + 1), NCD = (LC + 1) * (LD + 1), NX = NAB * NCD;
    static constexpr int ca = ncart(LA), cb = ncart(LB), cc = ncart(LC), cd = ncart(LD);
    static constexpr int NCOMP = ca * cb * cc * cd;
    static constexpr int ND = ca * cb + cc * cd + ca * cc + ca * cd + cb * cc + cb * cd;
    static constexpr int RD = 3 * NR;
    static constexpr int TS = RD * (4 * NX > NN * NM ? 4 * NX : NN * NM);  // step c records over step a's G
    static constexpr int JS = RD * 3 * NAB * NM;
    static_assert(TS % 2 == 0, "records are read as 16-byte halves");
    static constexpr int SLOT = TS + JS + ND;
    // slots at a time: as many (a power of two) as keep two workgroups on a CU's 160 KB of LDS
    static constexpr int S = 8 * SLOT <= 8600 ? 8 : 4 * SLOT <= 8600 ? 4 : 2 * SLOT <= 8600 ? 2 : 1;
    static constexpr int WPS = S >= 4 ? 1 : 4 / S;  // wavefronts per slot
};

// Sums v[0..8] over the wavefront and adds them to the atoms' sums (x, y, z of A, B, C, and D by
// translational invariance): eight values are halved together, each exchange step leaving a lane
// with half of them.
HFG_INLINE void rys_flush(const double* v, const int4 at, double* gsum) {
    const int lane = threadIdx.x & 63;
    double w[4], x[2], y;
    const bool h5 = lane & 32, h4 = lane & 16, h3 = lane & 8;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const double send = h5 ? v[k] : v[k + 4], keep = h5 ? v[k + 4] : v[k];
        w[k] = keep + __shfl_xor(send, 32);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const double send = h4 ? w[k] : w[k + 2], keep = h4 ? w[k + 2] : w[k];
        x[k] = keep + __shfl_xor(send, 16);
    }
    {
        const double send = h3 ? x[0] : x[1], keep = h3 ? x[1] : x[0];
        y = keep + __shfl_xor(send, 8);
    }
    for (int o = 4; o > 0; o >>= 1) y += __shfl_xor(y, o);
    double z = v[8];
    for (int o = 32; o > 0; o >>= 1) z += __shfl_xor(z, o);
    // lanes 0, 8, .., 56 hold values 0..7 (bits 5, 4, 3 of the lane = bits 2, 1, 0 of the value)
    const int k = lane == 1 ? 8 : ((h5 ? 4 : 0) + (h4 ? 2 : 0) + (h3 ? 1 : 0));
    if ((lane & 7) == 0 || lane == 1) {
        const double val = lane == 1 ? z : y;
        const int c = k / 3, d = k - 3 * c;
        atomicAdd(&gsum[(c == 0 ? at.x : c == 1 ? at.y : at.z) * 3 + d], val);
        atomicAdd(&gsum[at.w * 3 + d], -val);
    }
}

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void rys_grad_kernel(RysGradArgs ra) {
    using Sh = RysGradShape<LA, LB, LC, LD>;
    constexpr int S = Sh::S, NR = Sh::NR, RD = Sh::RD, NN = Sh::NN, NM = Sh::NM, NAB = Sh::NAB, NCD = Sh::NCD,
                  NX = Sh::NX, ND = Sh::ND;
    constexpr int ca = Sh::ca, cb = Sh::cb, cc = Sh::cc, cd = Sh::cd;
    __shared__ __align__(16) double Tb[S * Sh::TS];
    __shared__ double Jb[S * Sh::JS];
    __shared__ double Db[S * ND];
    __shared__ int2 cinfo[Sh::NCOMP];  // 1-D record indices, density-block indices
    __shared__ double gsum[kMaxAtoms * 3];
    __shared__ int rowpre[kMaxRows + 1];
    __shared__ int next_item;
    // the chunk's shell quartets
    __shared__ int qpre[kRysChunk + 1];  // primitive quartets before each
    __shared__ int4 qprim[kRysChunk];    // bra and ket primitive offset and stride
    __shared__ int qnk[kRysChunk];       // ket primitive pairs
    __shared__ int4 qao[kRysChunk];      // first Cartesian functions
    __shared__ int4 qat[kRysChunk];      // atoms
    __shared__ double qgeo[kRysChunk][7];  // A - B, C - D, degeneracy
    // the slots
    __shared__ int sq[S], sstaged[S];  // shell quartet (-1: none, or cut), the one its density blocks are of
    __shared__ double sz[S][3];        // 2 alpha, 2 beta, 2 gamma
    const GradArgs& a = ra.g;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int c = tid; c < Sh::NCOMP; c += 256) {
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
    for (;;) {
        __syncthreads();  // the previous item's flush has read gsum and next_item
        if (tid == 0) next_item = atomicAdd(a.queue, 1);
        __syncthreads();
        const int item = next_item;
        if (item >= a.nitems) break;
        const WorkItem w = a.items[item];
        const MolDev md = a.mols[w.mol];
        const MolCart mc = ra.mol_cart[w.mol];
        const double* __restrict__ Dm = ra.Dc + mc.off;
        const int natom3 = md.natom * 3;
        for (int k = tid; k < natom3; k += 256) gsum[k] = 0.0;
        const int nrows = w.r1 - w.r0;
        const int bpo = a.bp_off[w.P], kpo = a.bp_off[w.Q], kn = a.bp_cnt[w.Q];
        const bool same = (w.P == w.Q);
        for (int r = tid; r < nrows; r += 256) {
            const int i = w.r0 + r;
            int c = ket_count(a.psmean + kpo, kn, a.psmean[bpo + i], a.tol);
            if (same) c = min(c, i + 1);
            rowpre[r + 1] = max(0, min(c, w.c1) - w.c0);
        }
        __syncthreads();
        if (tid == 0) {
            rowpre[0] = 0;
            for (int r = 0; r < nrows; ++r) rowpre[r + 1] += rowpre[r];
        }
        __syncthreads();
        const int total = rowpre[nrows];
        for (int base = 0; base < total; base += kRysChunk) {
            // the chunk's shell quartets, one per lane of the first wavefront
            if (tid < kRysChunk) {
                int n = 0;
                if (base + tid < total) {
                    int i, j;
                    locate(base + tid, rowpre, nrows, w, i, j);
                    const PairDev bp = a.pairs[bpo + i];
                    const PairDev kp = a.pairs[kpo + j];
                    n = bp.np * kp.np;
                    qprim[tid] = make_int4(bp.off, bp.pstride, kp.off, kp.pstride);
                    qnk[tid] = kp.np;
                    const int* co = ra.cart_off + md.shell0;
                    const int* sat = a.shell_atom + md.shell0;
                    qao[tid] = make_int4(co[bp.sa], co[bp.sb], co[kp.sa], co[kp.sb]);
                    qat[tid] = make_int4(sat[bp.sa], sat[bp.sb], sat[kp.sa], sat[kp.sb]);
                    double deg = 8.0;
                    if (bp.sa == bp.sb) deg *= 0.5;
                    if (kp.sa == kp.sb) deg *= 0.5;
                    if (same && i == j) deg *= 0.5;
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        qgeo[tid][d] = bp.AB[d];
                        qgeo[tid][3 + d] = kp.AB[d];
                    }
                    qgeo[tid][6] = deg;
                }
                int s = n;
                for (int o = 1; o < 64; o <<= 1) {
                    const int t = __shfl_up(s, o);
                    if (lane >= o) s += t;
                }
                qpre[tid + 1] = s;
                if (tid == 0) qpre[0] = 0;
            }
            if (tid < S) sstaged[tid] = -1;
            __syncthreads();
            const int nprim = qpre[kRysChunk];
            double acc[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) acc[k] = 0.0;
            int pend = -1;  // shell quartet of acc
            for (int p0 = 0; p0 < nprim; p0 += S) {
                // a. quadrature and 2-D recursion
                for (int v = tid; v < S * RD; v += 256) {
                    const int s = v / RD, rd = v - s * RD, d = rd / NR, r = rd - d * NR;
                    const int idx = p0 + s;
                    int q = -1;
                    if (idx < nprim) {
                        int lo = 0, hi = kRysChunk;  // largest q with qpre[q] <= idx
                        while (hi - lo > 1) {
                            const int mid = (lo + hi) >> 1;
                            if (qpre[mid] <= idx)
                                lo = mid;
                            else
                                hi = mid;
                        }
                        q = lo;
                        const int4 pr = qprim[q];
                        const int rem = idx - qpre[q], ip = rem / qnk[q], jp = rem - ip * qnk[q];
                        const int ia = pr.x + ip * pr.y, ib = pr.z + jp * pr.w;
                        const double4 a0 = a.pp0[ia], a1 = a.pp1[ia], a2 = a.pp2[ia];
                        const double4 b0 = a.pp0[ib], b1 = a.pp1[ib], b2 = a.pp2[ib];
                        const double p = a0.x, qe = b0.x;
                        const double rs = rsqrt(p + qe);
                        const double pfac = a1.w * b1.w * rs;
                        if (fabs(pfac) < a.prim_cut) {
                            q = -1;
                        } else {
                            const double PQ[3] = {a0.y - b0.y, a0.z - b0.z, a0.w - b0.w};
                            const double ipq = rs * rs, rp = qe * ipq, rq = p * ipq;
                            double u, wt;
                            rys_point<NR>(ra.rys, p * rp * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]), r, u, wt);
                            const double pq = d == 0 ? PQ[0] : d == 1 ? PQ[1] : PQ[2];
                            const double pa = d == 0 ? a1.x : d == 1 ? a1.y : a1.z;
                            const double qc = d == 0 ? b1.x : d == 1 ? b1.y : b1.z;
                            rys_2d<NN, NM>(d == 2 ? pfac * wt : 1.0, pa - u * rp * pq, qc + u * rq * pq,
                                           a2.x * (1.0 - u * rp), b2.x * (1.0 - u * rq), 0.5 * u * ipq,
                                           Tb + s * Sh::TS + rd * (NN * NM));
                            if (rd == 0) {
                                sz[s][0] = 2.0 * a2.y;
                                sz[s][1] = 2.0 * a2.z;
                                sz[s][2] = 2.0 * b2.y;
                            }
                        }
                    }
                    if (rd == 0) sq[s] = q;
                }
                __syncthreads();
                // b. n -> (a, b) with the bra derivatives
                for (int v = tid; v < S * RD * NM; v += 256) {
                    const int s = v / (RD * NM), x = v - s * (RD * NM), rd = x / NM, m = x - rd * NM;
                    const int q = sq[s];
                    if (q < 0) continue;
                    const double AB = qgeo[q][rd / NR], za = sz[s][0], zb = sz[s][1];
                    const double* G = Tb + s * Sh::TS + rd * (NN * NM) + m * NN;
                    double h[LB + 2][NN];  // (n, b)
                    sfor<NN>([&](auto n) { h[0][n] = G[n]; });
                    sfor<LB + 1>([&](auto b) {
                        sfor<NN - 1 - b>([&](auto n) { h[b + 1][n] = h[b][n + 1] + AB * h[b][n]; });
                    });
                    double* J = Jb + s * Sh::JS + rd * (3 * NAB * NM) + m;
                    sfor<LA + 1>([&](auto i) {
                        sfor<LB + 1>([&](auto j) {
                            double dA = za * h[j][i + 1], dB = zb * h[j + 1][i];
                            if constexpr (i > 0) dA -= (double)(int)i * h[j][i - 1];
                            if constexpr (j > 0) dB -= (double)(int)j * h[j - 1][i];
                            constexpr int ab = i * (LB + 1) + j;
                            J[ab * NM] = h[j][i];
                            J[(NAB + ab) * NM] = dA;
                            J[(2 * NAB + ab) * NM] = dB;
                        });
                    });
                }
                // the density blocks of slots that moved to another shell quartet
                for (int v = tid; v < S * ND; v += 256) {
                    const int s = v / ND, e = v - s * ND;
                    const int q = sq[s];
                    if (q < 0 || q == sstaged[s]) continue;
                    const int4 o = qao[q];
                    constexpr int n1 = ca * cb, n2 = n1 + cc * cd, n3 = n2 + ca * cc, n4 = n3 + ca * cd, n5 = n4 + cb * cc;
                    int r, c;
                    if (e < n1) {
                        r = o.x + e / cb;
                        c = o.y + e % cb;
                    } else if (e < n2) {
                        r = o.z + (e - n1) / cd;
                        c = o.w + (e - n1) % cd;
                    } else if (e < n3) {
                        r = o.x + (e - n2) / cc;
                        c = o.z + (e - n2) % cc;
                    } else if (e < n4) {
                        r = o.x + (e - n3) / cd;
                        c = o.w + (e - n3) % cd;
                    } else if (e < n5) {
                        r = o.y + (e - n4) / cc;
                        c = o.z + (e - n4) % cc;
                    } else {
                        r = o.y + (e - n5) / cd;
                        c = o.w + (e - n5) % cd;
                    }
                    Db[v] = Dm[(size_t)r * mc.n + c];
                }
                __syncthreads();
                if (tid < S && sq[tid] >= 0) sstaged[tid] = sq[tid];
                // c. m -> (c, d) with the ket derivative
                for (int v = tid; v < S * RD * NAB; v += 256) {
                    const int s = v / (RD * NAB), x = v - s * (RD * NAB), rd = x / NAB, ab = x - rd * NAB;
                    const int q = sq[s];
                    if (q < 0) continue;
                    const double CD = qgeo[q][3 + rd / NR], zc = sz[s][2];
                    const double* J = Jb + s * Sh::JS + rd * (3 * NAB * NM) + ab * NM;
                    double2* T = reinterpret_cast<double2*>(Tb + s * Sh::TS + (rd * NX + ab * NCD) * 4);
                    double h[3][LD + 1][NM];  // (m, d) of I, dI/dA, dI/dB
                    sfor<3>([&](auto k) {
                        constexpr int n = k == 0 ? NM : NM - 1;
                        sfor<n>([&](auto m) { h[k][0][m] = J[k * NAB * NM + m]; });
                        sfor<LD>([&](auto l) {
                            sfor<n - 1 - l>([&](auto m) { h[k][l + 1][m] = h[k][l][m + 1] + CD * h[k][l][m]; });
                        });
                    });
                    sfor<LC + 1>([&](auto i) {
                        sfor<LD + 1>([&](auto j) {
                            double dC = zc * h[0][j][i + 1];
                            if constexpr (i > 0) dC -= (double)(int)i * h[0][j][i - 1];
                            constexpr int x2 = (i * (LD + 1) + j) * 2;
                            T[x2] = make_double2(h[0][j][i], h[1][j][i]);
                            T[x2 + 1] = make_double2(h[2][j][i], dC);
                        });
                    });
                }
                __syncthreads();
                // d. contraction with the two-particle density
                constexpr int kPerWave = S >= 4 ? S / 4 : 1;
                for (int t = 0; t < kPerWave; ++t) {
                    const int s = S >= 4 ? wave * kPerWave + t : wave / Sh::WPS;
                    const int q = sq[s];
                    if (q < 0) continue;
                    if (q != pend) {
                        if (pend >= 0) rys_flush(acc, qat[pend], gsum);
#pragma unroll
                        for (int k = 0; k < 9; ++k) acc[k] = 0.0;
                        pend = q;
                    }
                    const double deg = qgeo[q][6];
                    const double* Dab = Db + s * ND;
                    const double *Dcd = Dab + ca * cb, *Dac = Dcd + cc * cd, *Dad = Dac + ca * cc, *Dbc = Dad + ca * cd,
                                 *Dbd = Dbc + cb * cc;
                    const double2* T = reinterpret_cast<const double2*>(Tb + s * Sh::TS);
                    for (int c = lane + 64 * (S >= 4 ? 0 : wave % Sh::WPS); c < Sh::NCOMP; c += 64 * Sh::WPS) {
                        const int2 ci = cinfo[c];
                        const int ia = ci.y & 7, ib = (ci.y >> 3) & 7, ic = (ci.y >> 6) & 7, id = ci.y >> 9;
                        const double gam = deg * (2.0 * Dab[ia * cb + ib] * Dcd[ic * cd + id] -
                                                  0.5 * (Dac[ia * cc + ic] * Dbd[ib * cd + id] + Dad[ia * cd + id] * Dbc[ib * cc + ic]));
                        const double2* Tx = T + 2 * (ci.x & 255);
                        const double2* Ty = T + 2 * (NR * NX + ((ci.x >> 8) & 255));
                        const double2* Tz = T + 2 * (2 * NR * NX + (ci.x >> 16));
#pragma unroll
                        for (int r = 0; r < NR; ++r) {
                            const double2 x0 = Tx[2 * r * NX], x1 = Tx[2 * r * NX + 1];
                            const double2 y0 = Ty[2 * r * NX], y1 = Ty[2 * r * NX + 1];
                            const double2 z0 = Tz[2 * r * NX], z1 = Tz[2 * r * NX + 1];
                            const double gx = gam * x0.x, gy = gam * y0.x;
                            const double yz = gy * z0.x, xz = gx * z0.x, xy = gx * y0.x;
                            acc[0] += yz * x0.y;
                            acc[3] += yz * x1.x;
                            acc[6] += yz * x1.y;
                            acc[1] += xz * y0.y;
                            acc[4] += xz * y1.x;
                            acc[7] += xz * y1.y;
                            acc[2] += xy * z0.y;
                            acc[5] += xy * z1.x;
                            acc[8] += xy * z1.y;
                        }
                    }
                }
                __syncthreads();  // the slots' tables are rewritten by the next round
            }
            if (pend >= 0) rys_flush(acc, qat[pend], gsum);
            __syncthreads();  // the chunk's quartets are rewritten
        }
        __syncthreads();
        double* out = a.slab + w.gslab;
        for (int k = tid; k < natom3; k += 256) out[k] = gsum[k];
    }
}

template <int LA, int LB, int LC, int LD>
hipError_t launch_rys_grad_class(const RysGradArgs& a, LaunchShape sh, hipStream_t s);

// The Rys launch of a class with L >= kRysGradMinL over nitems work items.
hipError_t launch_rys_grad(int la, int lb, int lc, int ld, const RysGradArgs& a, int nitems, LaunchShape sh, hipStream_t s);

// Densities over the Cartesian functions, Dc = T D T^T per molecule (T the map of a Cartesian
// function's terms), max_ncart the largest molecule's Cartesian function count.
hipError_t launch_to_cart(const double* D, const MolDev* mols, const MolCart* mc, int nmol, int max_ncart,
                          const CartTerms* terms, double* Dc, hipStream_t s);

}  // namespace hfg

// FP64 J/K (and ERI export) kernel of the classes of high angular momentum, by Rys quadrature.
//
// The register kernel (jk_impl.hpp) gives a lane a whole shell quartet and spills from L = 5 (0.2-4 KB
// per lane), and a small molecule has too few quartets to fill wavefronts with; the program kernel
// (coop.hpp) from L = 7 runs one primitive quartet at a time with a barrier per recursion level.
// Here S primitive quartets ("slots") go through a workgroup together, as in the gradient's Rys
// kernel (rys_grad.hpp): 2-D recursion per (slot, node, direction), transfer to (a, b), transfer to
// (c, d), each spread over the lanes with the 1-D tables in LDS; then a wavefront takes its slots,
// its lanes holding the Cartesian component quartets and summing the products of three 1-D integrals
// over the nodes and over consecutive primitive quartets of one shell quartet. When the shell
// quartet changes, the sums go through hfscf's element screen into LDS and the wavefront digests
// them, one lane per element of the six J/K blocks, into tiles over the Cartesian functions; the
// item's end transforms the tiles to the output basis on their way to the slab. Digestion is linear,
// so a shell quartet whose primitives fall to several wavefronts is digested in parts (the
// Cartesian diagonal that hfscf takes from its screen is added by the part with the first one).
//
// Bound: the latency of a round (four barriers, the loads of step a and its index arithmetic; FP64 is 7 to 17 %
// of the VALU instructions), about 0.4 ns per primitive quartet over the device. By LDS one workgroup fits a
// CU for (dd|dd) (134 KB) and (dd|dp) (84 KB), two to four for the other classes. A workgroup walks its work
// item in series, 2 to 3 us per round of S primitive quartets, which limits the items that L = 4 and 5 run here.
// Per class against the other kernels in context.hpp (jk_on_rys). Per build, when they replaced the
// register and program kernels: (H2O)8 8.5 -> 6.4 ms, C12H26 / 6-31G** 8.2 -> 5.5, (H2O)16 34.5 -> 28.7.
#pragma once
#include "coop.hpp"
#include "rys.hpp"

namespace hfg {

struct RysJkArgs {
    JkArgs j;
    const double* rys;        // quadrature tables
    const double* Dc;         // densities over the Cartesian functions, concatenated
    const int* cart_off;      // global shell -> first Cartesian function in its molecule
    const MolCart* mol_cart;  // per molecule
    int pure;
};

template <int LA, int LB, int LC, int LD>
struct RysJkShape {
    static constexpr int L = LA + LB + LC + LD;
    static constexpr int NR = L / 2 + 1;
    static constexpr int NN = LA + LB + 1, NM = LC + LD + 1;
    static constexpr int NAB = (LA + 1) * (LB + 1), NCD = (LC + 1) * (LD + 1), NX = NAB * NCD;
    static constexpr int ca = ncart(LA), cb = ncart(LB), cc = ncart(LC), cd = ncart(LD);
    static constexpr int NCOMP = ca * cb * cc * cd;
    static constexpr int ND = ca * cb + cc * cd + ca * cc + ca * cd + cb * cc + cb * cd;
    static constexpr int RD = 3 * NR;
    static constexpr int TS = RD * (NX > NN * NM ? NX : NN * NM);  // step c's values over step a's G
    static constexpr int JS = RD * NAB * NM;
    static constexpr int S = 8 * (TS + JS + ND) <= 4200 ? 8 : 4;
    static constexpr int CR = (NCOMP + 63) / 64;  // component quartets per lane
    // Cartesian functions of the largest block (kBlockFuncs output functions)
    static constexpr int fmax(int l) { return l == 0 ? kBlockFuncs : l == 1 ? 15 : 18; }
    static constexpr int NT = fmax(LA) * fmax(LB) + fmax(LC) * fmax(LD) + fmax(LA) * fmax(LC) + fmax(LA) * fmax(LD) +
                              fmax(LB) * fmax(LC) + fmax(LB) * fmax(LD);
};

constexpr int kRysJkChunk = 64;  // shell quartets enumerated at a time

HFG_INLINE void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Writes a shell quartet's integrals to the packed vector at every canonical element's index, once
// per element as export_block (jk_impl.hpp); `ao` the shells' first output functions, I the
// Cartesian block.
template <int LA, int LB, int LC, int LD>
HFG_INLINE void export_quartet(bool pure, const double* I, int4 ao, bool same_pair, double* out) {
    constexpr int cb = ncart(LB), cc = ncart(LC), cd = ncart(LD);
    const int na = pure ? 2 * LA + 1 : ncart(LA), nb = pure ? 2 * LB + 1 : cb, nc = pure ? 2 * LC + 1 : cc,
              nd = pure ? 2 * LD + 1 : cd;
    auto tri = [](long long x, long long y) { return x >= y ? x * (x + 1) / 2 + y : y * (y + 1) / 2 + x; };
    for (int e = threadIdx.x & 63; e < na * nb * nc * nd; e += 64) {
        const int u = e % nd, r = (e / nd) % nc, q = (e / (nd * nc)) % nb, p = e / (nd * nc * nb);
        const int fi = ao.x + p, fj = ao.y + q, fk = ao.z + r, fl = ao.w + u;
        const long long ij = tri(fi, fj), kl = tri(fk, fl);
        if ((ao.x == ao.y && fi < fj) || (ao.z == ao.w && fk < fl) || (same_pair && ij < kl)) continue;
        double v = 0.0;
        if (pure) {
            const SphTerms ta = sph_terms(LA, p), tb = sph_terms(LB, q), tc = sph_terms(LC, r), td = sph_terms(LD, u);
            // unrolled over the at most three terms of each index, which keeps them in registers
            auto each = [](const SphTerms& t, auto&& fn) {
                sfor<3>([&](auto x) {
                    if (x < t.n) fn(t.c[x], t.w[x]);
                });
            };
            each(ta, [&](int x, double wx) {
                each(tb, [&](int y, double wy) {
                    each(tc, [&](int z, double wz) {
                        each(td, [&](int t, double wt) { v += wx * wy * wz * wt * I[((x * cb + y) * cc + z) * cd + t]; });
                    });
                });
            });
        } else {
            v = I[e];
        }
        out[tri(ij, kl)] = v;
    }
}

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void rys_jk_kernel(RysJkArgs ra) {
    using Sh = RysJkShape<LA, LB, LC, LD>;
    constexpr int S = Sh::S, NR = Sh::NR, RD = Sh::RD, NN = Sh::NN, NM = Sh::NM, NAB = Sh::NAB, NCD = Sh::NCD,
                  NX = Sh::NX, ND = Sh::ND, NCOMP = Sh::NCOMP, CR = Sh::CR, kPerWave = S / 4;
    constexpr int ca = Sh::ca, cb = Sh::cb, cc = Sh::cc, cd = Sh::cd;
    constexpr int n1 = ca * cb, n2 = n1 + cc * cd, n3 = n2 + ca * cc, n4 = n3 + ca * cd, n5 = n4 + cb * cc;
    __shared__ double Tb[S * Sh::TS];
    __shared__ double Jb[S * Sh::JS];
    __shared__ double Db[S * ND];
    __shared__ double Ib[4][NCOMP];
    __shared__ double tiles[Sh::NT];
    __shared__ int rowpre[kMaxRows + 1];
    __shared__ int next_item;
    // the chunk's shell quartets
    __shared__ int qpre[kRysJkChunk + 1];   // primitive quartets before each
    __shared__ int4 qprim[kRysJkChunk];     // bra and ket primitive offset and stride
    __shared__ int qnk[kRysJkChunk];        // ket primitive pairs
    __shared__ int4 qao[kRysJkChunk];       // first Cartesian functions (output functions for an export)
    __shared__ int4 qslot[kRysJkChunk];     // positions of the shells in their blocks
    __shared__ int4 qsq[kRysJkChunk];       // bra and ket offset of sqrt|(pq|pq)|, element screen, same pair
    __shared__ double qgeo[kRysJkChunk][7];  // A - B, C - D, permutational weight
    // the slots
    __shared__ int sq[S], sact[S], sstaged[S];  // shell quartet (-1: none), whether it is evaluated, density blocks
    const JkArgs& a = ra.j;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // the lane's component quartets: 1-D value indices
    int cinfo[CR];
#pragma unroll
    for (int i = 0; i < CR; ++i) {
        const int c = min(lane + 64 * i, NCOMP - 1);
        const int ia = c / (cb * cc * cd), ib = (c / (cc * cd)) % cb, ic = (c / cd) % cc, id = c % cd;
        int x = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d)
            x |= (((cart_exp(LA, ia, d) * (LB + 1) + cart_exp(LB, ib, d)) * (LC + 1) + cart_exp(LC, ic, d)) * (LD + 1) +
                  cart_exp(LD, id, d))
                 << (8 * d);
        cinfo[i] = x;
    }
    const bool dscreen = a.dtol > 0.0;
    for (;;) {
        __syncthreads();  // the previous item's flush has read the tiles and next_item
        if (tid == 0) next_item = atomicAdd(a.queue, 1);
        __syncthreads();
        const int item = next_item;
        if (item >= a.nitems) break;
        const WorkItem w = a.items[item];
        const MolDev md = a.mols[w.mol];
        const MolCart mc = ra.mol_cart[w.mol];
        const double* __restrict__ Dm = ra.Dc + mc.off;
        const float* __restrict__ dm = a.dmax + md.dm_off;
        // the blocks' Cartesian widths and the tiles over them
        const int na = ra.pure ? 2 * LA + 1 : ca, nb = ra.pure ? 2 * LB + 1 : cb, nc = ra.pure ? 2 * LC + 1 : cc,
                  nd = ra.pure ? 2 * LD + 1 : cd;
        const int gA = a.blk_nf[w.A], gB = a.blk_nf[w.B], gC = a.blk_nf[w.C], gD = a.blk_nf[w.D];
        const int fA = gA / na * ca, fB = gB / nb * cb, fC = gC / nc * cc, fD = gD / nd * cd;
        const int t1 = fA * fB, t2 = t1 + fC * fD, t3 = t2 + fA * fC, t4 = t3 + fA * fD, t5 = t4 + fB * fC,
                  ntile = t5 + fB * fD;
        for (int k = tid; k < ntile; k += 256) tiles[k] = 0.0;
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
        for (int base = 0; base < total; base += kRysJkChunk) {
            // the chunk's shell quartets, one per lane of the first wavefront; a density-screened one
            // has no primitives
            if (tid < kRysJkChunk) {
                int n = 0;
                const int off = base + (a.eri_out ? (tid & 15) * 4 + (tid >> 4) : tid);
                if (off < total) {
                    int i, j;
                    locate(off, rowpre, nrows, w, i, j);
                    const PairDev bp = a.pairs[bpo + i];
                    const PairDev kp = a.pairs[kpo + j];
                    if (!dscreen || density_bound(bp, kp, dm, md.nshell) >= a.dtol) n = bp.np * kp.np;
                    qprim[tid] = make_int4(bp.off, bp.pstride, kp.off, kp.pstride);
                    qnk[tid] = kp.np;
                    const int* co = ra.cart_off + md.shell0;
                    qao[tid] = a.eri_out ? make_int4(bp.ao_a, bp.ao_b, kp.ao_a, kp.ao_b)
                                         : make_int4(co[bp.sa], co[bp.sb], co[kp.sa], co[kp.sb]);
                    qslot[tid] = make_int4(bp.slot_a, bp.slot_b, kp.slot_a, kp.slot_b);
                    qsq[tid] = make_int4(bp.sq_off, kp.sq_off, a.elem_tol > 0.0 && bp.sq_min * kp.sq_min < a.elem_tol,
                                         same && i == j);
                    double s = 1.0;
                    if (bp.sa == bp.sb) s *= 0.5;
                    if (kp.sa == kp.sb) s *= 0.5;
                    if (same && i == j) s *= 0.5;
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        qgeo[tid][d] = bp.AB[d];
                        qgeo[tid][3 + d] = kp.AB[d];
                    }
                    qgeo[tid][6] = s;
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
            // The slots take the chunk's primitive quartets in order. An export instead gives every
            // wavefront sixteen shell quartets of its own, so that one sums a quartet alone, in a fixed
            // order, and writes it once.
            const bool own = a.eri_out != nullptr;
            int nprim = qpre[kRysJkChunk];
            if (own) {
                int rounds = 0;
                for (int v = 0; v < 4; ++v) rounds = max(rounds, (qpre[16 * v + 16] - qpre[16 * v] + kPerWave - 1) / kPerWave);
                nprim = rounds * S;
            }
            double acc[CR];
#pragma unroll
            for (int i = 0; i < CR; ++i) acc[i] = 0.0;
            int pend = -1, pslot = 0;  // shell quartet of acc, a slot with its density blocks
            bool pfirst = false;       // whether acc includes its first primitive quartet
            // digests (or exports) acc, the whole wavefront together
            auto flush = [&]() __attribute__((always_inline)) {
                const int4 qs = qsq[pend];
                double* I = Ib[wave];
#pragma unroll
                for (int i = 0; i < CR; ++i) {
                    const int c = lane + 64 * i;
                    if (c < NCOMP) {
                        double v = acc[i];
                        const int ab = c / (cc * cd), kl = c - ab * (cc * cd);
                        // hfscf's element screen (hfscf: src/integrals/hfscf_oseri.cpp:152-158)
                        if (qs.z) v *= a.psq[qs.x + ab] * a.psq[qs.y + kl] >= a.elem_tol ? 1.0 : 0.0;
                        // and its Cartesian diagonal, taken from the screen (:214-218)
                        if (LA == LC && LB == LD && !ra.pure && a.elem_tol > 0.0 && qs.w && ab == kl) {
                            const double s = a.psq[qs.x + ab];
                            v = pfirst ? s * s : 0.0;
                        }
                        I[c] = v;
                    }
                    acc[i] = 0.0;
                }
                wave_fence();
                if (a.eri_out) {
                    export_quartet<LA, LB, LC, LD>(ra.pure, I, qao[pend], qs.w, a.eri_out);
                    wave_fence();
                    return;
                }
                const int4 sl = qslot[pend];
                const double s = qgeo[pend][6];
                const double* D = Db + pslot * ND;
                for (int e = lane; e < ND; e += 64) {
                    int r, c, i0, s1, m1, s2, m2, d0, t;  // value (r, c) of a block: sum over m1 x m2
                    double f = s;
                    if (e < n1) {
                        r = e / cb;
                        c = e - r * cb;
                        i0 = e * (cc * cd);
                        m1 = cc, s1 = cd, m2 = cd, s2 = 1, d0 = n1;
                        t = (sl.x * ca + r) * fB + sl.y * cb + c;
                        f += s;
                    } else if (e < n2) {
                        r = (e - n1) / cd;
                        c = e - n1 - r * cd;
                        i0 = e - n1;
                        m1 = ca, s1 = cb * cc * cd, m2 = cb, s2 = cc * cd, d0 = 0;
                        t = t1 + (sl.z * cc + r) * fD + sl.w * cd + c;
                        f += s;
                    } else if (e < n3) {
                        r = (e - n2) / cc;
                        c = e - n2 - r * cc;
                        i0 = r * (cb * cc * cd) + c * cd;
                        m1 = cb, s1 = cc * cd, m2 = cd, s2 = 1, d0 = n5;
                        t = t2 + (sl.x * ca + r) * fC + sl.z * cc + c;
                    } else if (e < n4) {
                        r = (e - n3) / cd;
                        c = e - n3 - r * cd;
                        i0 = r * (cb * cc * cd) + c;
                        m1 = cb, s1 = cc * cd, m2 = cc, s2 = cd, d0 = n4;
                        t = t3 + (sl.x * ca + r) * fD + sl.w * cd + c;
                    } else if (e < n5) {
                        r = (e - n4) / cc;
                        c = e - n4 - r * cc;
                        i0 = r * (cc * cd) + c * cd;
                        m1 = ca, s1 = cb * cc * cd, m2 = cd, s2 = 1, d0 = n3;
                        t = t4 + (sl.y * cb + r) * fC + sl.z * cc + c;
                    } else {
                        r = (e - n5) / cd;
                        c = e - n5 - r * cd;
                        i0 = r * (cc * cd) + c;
                        m1 = ca, s1 = cb * cc * cd, m2 = cc, s2 = cd, d0 = n2;
                        t = t5 + (sl.y * cb + r) * fD + sl.w * cd + c;
                    }
                    double v = 0.0;
                    for (int x = 0; x < m1; ++x)
                        for (int y = 0; y < m2; ++y) v += D[d0 + x * m2 + y] * I[i0 + x * s1 + y * s2];
                    atomicAdd(&tiles[t], f * v);
                }
                wave_fence();
            };
            for (int p0 = 0; p0 < nprim; p0 += S) {
                // a. quadrature and 2-D recursion
                for (int v = tid; v < S * RD; v += 256) {
                    const int s = v / RD, rd = v - s * RD, d = rd / NR, r = rd - d * NR;
                    const int wv = 16 * (s / kPerWave);  // the slot's wavefront's first shell quartet (export)
                    const int idx = own ? qpre[wv] + p0 / S * kPerWave + s % kPerWave : p0 + s;
                    int q = -1, ok = 0;
                    if (idx < (own ? qpre[wv + 16] : nprim)) {
                        int lo = 0, hi = kRysJkChunk;  // largest q with qpre[q] <= idx
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
                        const double4 a0 = a.pp0[ia], a1 = a.pp1[ia], b0 = a.pp0[ib], b1 = a.pp1[ib];
                        const double p = a0.x, qe = b0.x;
                        const double rs = rsqrt(p + qe);
                        const double pfac = a1.w * b1.w * rs;
                        if (fabs(pfac) >= a.prim_cut) {
                            ok = 1;
                            const double PQ[3] = {a0.y - b0.y, a0.z - b0.z, a0.w - b0.w};
                            const double ipq = rs * rs, rp = qe * ipq, rq = p * ipq;
                            double u, wt;
                            rys_point<NR>(ra.rys, p * rp * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]), r, u, wt);
                            const double pq = d == 0 ? PQ[0] : d == 1 ? PQ[1] : PQ[2];
                            const double pa = d == 0 ? a1.x : d == 1 ? a1.y : a1.z;
                            const double qc = d == 0 ? b1.x : d == 1 ? b1.y : b1.z;
                            rys_2d<NN, NM>(d == 2 ? pfac * wt : 1.0, pa - u * rp * pq, qc + u * rq * pq,
                                           a.pp2[ia].x * (1.0 - u * rp), a.pp2[ib].x * (1.0 - u * rq), 0.5 * u * ipq,
                                           Tb + s * Sh::TS + rd * (NN * NM));
                        }
                    }
                    if (rd == 0) {
                        sq[s] = q;
                        sact[s] = ok;
                    }
                }
                __syncthreads();
                // b. n -> (a, b)
                for (int v = tid; v < S * RD * NM; v += 256) {
                    const int s = v / (RD * NM), x = v - s * (RD * NM), rd = x / NM, m = x - rd * NM;
                    if (!sact[s]) continue;
                    const double AB = qgeo[sq[s]][rd / NR];
                    const double* G = Tb + s * Sh::TS + rd * (NN * NM) + m * NN;
                    double h[LB + 1][NN];  // (b, n)
                    sfor<NN>([&](auto n) { h[0][n] = G[n]; });
                    sfor<LB>([&](auto b) {
                        sfor<NN - 1 - b>([&](auto n) { h[b + 1][n] = h[b][n + 1] + AB * h[b][n]; });
                    });
                    double* J = Jb + s * Sh::JS + rd * (NAB * NM) + m;
                    sfor<LA + 1>([&](auto i) { sfor<LB + 1>([&](auto j) { J[(i * (LB + 1) + j) * NM] = h[j][i]; }); });
                }
                // the density blocks of slots that moved to another shell quartet
                if (!a.eri_out)
                    for (int v = tid; v < S * ND; v += 256) {
                        const int s = v / ND, e = v - s * ND;
                        const int q = sq[s];
                        if (q < 0 || q == sstaged[s]) continue;
                        const int4 o = qao[q];
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
                // c. m -> (c, d)
                for (int v = tid; v < S * RD * NAB; v += 256) {
                    const int s = v / (RD * NAB), x = v - s * (RD * NAB), rd = x / NAB, ab = x - rd * NAB;
                    if (!sact[s]) continue;
                    const double CD = qgeo[sq[s]][3 + rd / NR];
                    const double* J = Jb + s * Sh::JS + rd * (NAB * NM) + ab * NM;
                    double* T = Tb + s * Sh::TS + rd * NX + ab * NCD;
                    double h[LD + 1][NM];  // (d, m)
                    sfor<NM>([&](auto m) { h[0][m] = J[m]; });
                    sfor<LD>([&](auto l) {
                        sfor<NM - 1 - l>([&](auto m) { h[l + 1][m] = h[l][m + 1] + CD * h[l][m]; });
                    });
                    sfor<LC + 1>([&](auto i) { sfor<LD + 1>([&](auto j) { T[i * (LD + 1) + j] = h[j][i]; }); });
                }
                __syncthreads();
                // d. the wavefront's slots
                for (int t = 0; t < kPerWave; ++t) {
                    const int s = wave * kPerWave + t;
                    const int q = sq[s];
                    if (q < 0) continue;
                    if (q != pend) {
                        if (pend >= 0) flush();
                        pend = q;
                        pfirst = false;
                    }
                    pslot = s;
                    if (own || p0 + s == qpre[q]) pfirst = true;
                    if (!sact[s]) continue;
                    const double* T = Tb + s * Sh::TS;
#pragma unroll
                    for (int i = 0; i < CR; ++i) {
                        const double* Tx = T + (cinfo[i] & 255);
                        const double* Ty = T + NR * NX + ((cinfo[i] >> 8) & 255);
                        const double* Tz = T + 2 * NR * NX + (cinfo[i] >> 16);
#pragma unroll
                        for (int r = 0; r < NR; ++r) acc[i] += Tx[r * NX] * Ty[r * NX] * Tz[r * NX];
                    }
                }
                // the density blocks of a slot are replaced in the next round: a pending shell quartet
                // that this wavefront does not continue there is digested now
                if (pend >= 0 && !own) {
                    const int nx = p0 + S + wave * kPerWave;  // the wavefront's next slot
                    if (nx >= nprim || nx >= qpre[pend + 1]) {
                        flush();
                        pend = -1;
                    }
                }
                __syncthreads();  // the slots' tables are rewritten by the next round
            }
            if (pend >= 0) flush();
            __syncthreads();  // the chunk's quartets are rewritten
        }
        if (a.eri_out) continue;  // an export has no tiles (the item may have no slab)
        // the tiles in the output basis
        double* out = a.slab + w.slab;
        auto put = [&](const double* tile, int fc, auto lr, auto lc, int nr, int ncol) {
            if (!ra.pure) {
                for (int k = tid; k < nr * ncol; k += 256) out[k] = tile[k];
            } else {
                constexpr int Lr = lr, Lc = lc;
                for (int k = tid; k < nr * ncol; k += 256) {
                    const int r = k / ncol, c = k - r * ncol;
                    const int sr = r / (2 * Lr + 1), sc = c / (2 * Lc + 1);
                    const SphTerms tr = sph_terms(Lr, r - sr * (2 * Lr + 1)), tc = sph_terms(Lc, c - sc * (2 * Lc + 1));
                    double v = 0.0;
                    sfor<3>([&](auto x) {
                        sfor<3>([&](auto y) {
                            if (x < tr.n && y < tc.n)
                                v += tr.w[x] * tc.w[y] * tile[(sr * ncart(Lr) + tr.c[x]) * fc + sc * ncart(Lc) + tc.c[y]];
                        });
                    });
                    out[k] = v;
                }
            }
            out += nr * ncol;
        };
        put(tiles, fB, ic<LA>{}, ic<LB>{}, gA, gB);
        put(tiles + t1, fD, ic<LC>{}, ic<LD>{}, gC, gD);
        put(tiles + t2, fC, ic<LA>{}, ic<LC>{}, gA, gC);
        put(tiles + t3, fD, ic<LA>{}, ic<LD>{}, gA, gD);
        put(tiles + t4, fC, ic<LB>{}, ic<LC>{}, gB, gC);
        put(tiles + t5, fD, ic<LB>{}, ic<LD>{}, gB, gD);
    }
}

template <int LA, int LB, int LC, int LD>
hipError_t launch_rys_jk_class(const RysJkArgs& a, LaunchShape sh, hipStream_t s);

// The Rys launch of a J/K class over nitems work items.
hipError_t launch_rys_jk(int la, int lb, int lc, int ld, const RysJkArgs& a, int nitems, LaunchShape sh, hipStream_t s);

}  // namespace hfg

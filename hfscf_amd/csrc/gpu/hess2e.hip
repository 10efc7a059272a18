// Two-electron part of the RHF Hessian at a fixed density on the GPU: hfscf's
//   m_hessianC(X1, X2)  =  sum_ijkl D_ij D_kl 2 d2(ij|kl)/dX1 dX2
//   m_hessianEx(X1, X2) = -sum_ijkl D_ij D_kl   d2(ik|jl)/dX1 dX2
// (hfscf: src/hessian/hfscf_hessian_ints.cpp:20-313). hfscf evaluates the second-derivative
// integrals with its chained recursions into six N^4 tensors per direction pair
// (src/integrals/hfscf_oserideriv2qq.cpp:28-749, hfscf_oserideriv2pq.cpp:23-799) and contracts
// them afterwards; here they are contracted with the density as they are made and never stored
// (rys_hess.hpp). This file prepares the shell pairs and work items and launches the classes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "context.hpp"
#include "rys_grad.hpp"
#include "rys_hess.hpp"

namespace hfg {

namespace {

// Pair classes by angular momenta, in the order that makes bra >= ket canonical.
constexpr int kPairLa[6] = {0, 1, 1, 2, 2, 2}, kPairLb[6] = {0, 0, 1, 0, 1, 2};

#define HFG_FOR_HESS(X)                                                                             \
    X(0, 0, 0, 0) X(1, 0, 0, 0) X(1, 0, 1, 0) X(1, 1, 0, 0) X(1, 1, 1, 0) X(1, 1, 1, 1)             \
    X(2, 0, 0, 0) X(2, 0, 1, 0) X(2, 0, 1, 1) X(2, 0, 2, 0) X(2, 1, 0, 0) X(2, 1, 1, 0)             \
    X(2, 1, 1, 1) X(2, 1, 2, 0) X(2, 1, 2, 1) X(2, 2, 0, 0) X(2, 2, 1, 0) X(2, 2, 1, 1)             \
    X(2, 2, 2, 0) X(2, 2, 2, 1) X(2, 2, 2, 2)

}  // namespace

#define HFG_DECL(A, B, C, D) \
    template <>              \
    hipError_t launch_rys_hess_class<A, B, C, D>(const HessArgs&, hipStream_t);
HFG_FOR_HESS(HFG_DECL)
#undef HFG_DECL

namespace {

hipError_t launch_rys_hess(int P, int Q, const HessArgs& g, hipStream_t s) {
    const int la = kPairLa[P], lb = kPairLb[P], lc = kPairLa[Q], ld = kPairLb[Q];
#define HFG_CASE(A, B, C, D) \
    if (la == A && lb == B && lc == C && ld == D) return launch_rys_hess_class<A, B, C, D>(g, s);
    HFG_FOR_HESS(HFG_CASE)
#undef HFG_CASE
    return hipErrorInvalidValue;
}

// Primitive quartets of one work item of class (P | Q).
int item_prims(int P, int Q) {
    const int la = kPairLa[P], lb = kPairLb[P], lc = kPairLa[Q], ld = kPairLb[Q];
#define HFG_CASE(A, B, C, D) \
    if (la == A && lb == B && lc == C && ld == D) return RysHessShape<A, B, C, D>::S * kHessRounds;
    HFG_FOR_HESS(HFG_CASE)
#undef HFG_CASE
    return 1;
}

// Sum of the copies' upper triangles, mirrored: out = {HC, HX}.
__global__ __launch_bounds__(256) void hess_sum_kernel(const double* __restrict__ H, int copies, int n3,
                                                       double* __restrict__ out) {
    const int nn = n3 * n3;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < 2 * nn; e += gridDim.x * 256) {
        const int part = e / nn, r = (e - part * nn) / n3, c = e - part * nn - r * n3;
        const int u = part * nn + min(r, c) * n3 + max(r, c);
        double v = 0.0;
        for (int k = 0; k < copies; ++k) v += H[(size_t)k * 2 * nn + u];
        out[e] = v;
    }
}

}  // namespace

__global__ __launch_bounds__(64) void hess_prim_kernel(HessArgs g) {
    const int k = blockIdx.x, lane = threadIdx.x;
    const HessPair pr = g.pairs[k];
    const OneShell A = g.sh[pr.sa], B = g.sh[pr.sb];
    double ra[3], rb[3], r2 = 0.0;
    for (int d = 0; d < 3; ++d) {
        ra[d] = g.xyz[3 * A.atom + d];
        rb[d] = g.xyz[3 * B.atom + d];
        r2 += (ra[d] - rb[d]) * (ra[d] - rb[d]);
    }
    int np = 0;
    for (int base = 0; base < A.np * B.np; base += 64) {
        const int x = base + lane;
        bool keep = false;
        double a = 1.0, b = 1.0, p = 2.0, K = 0.0;
        if (x < A.np * B.np) {
            const int i = x / B.np, j = x - i * B.np;
            a = g.alpha[A.po + i];
            b = g.alpha[B.po + j];
            p = a + b;
            // sqrt(2 pi^2.5)
            K = exp(-a * b / p * r2) * g.coef[A.po + i] * g.coef[B.po + j] * 5.9149671727956128778 / p;
            keep = fabs(K) >= g.kmin;
        }
        const unsigned long long mask = __ballot(keep);
        if (keep) {
            const int o = pr.off + np + __popcll(mask & ((1ull << lane) - 1));
            g.hp0[o] = make_double4(p, (a * ra[0] + b * rb[0]) / p, (a * ra[1] + b * rb[1]) / p, (a * ra[2] + b * rb[2]) / p);
            g.hp1[o] = make_double4(K, a, b, 0.5 / p);
        }
        np += __popcll(mask);
    }
    if (lane == 0) g.pairs[k].np = np;
}

}  // namespace hfg

extern "C" {

int hfg_hessian_2e(hfg_ctx* c, const double* D, double* HC, double* HX) {
    if (!c) return HFG_ERR_ARG;
    if (!D || !HC || !HX) {
        c->err = "hfg_hessian_2e: null argument";
        return HFG_ERR_ARG;
    }
    hfg::OneArgs one;
    if (int r = hfg::one_upload(c, one)) return r;
    const int n = c->nbf, nc = c->ncart, n3 = 3 * c->natom;
    const size_t nn = (size_t)n * n, nh = (size_t)n3 * n3;
    // shell pairs by class, most primitive pairs first, and each class's runs of equal primitive counts
    std::vector<hfg::HessPair> pairs;
    struct Run {
        int first, count, nprim;
    };
    std::vector<Run> runs[6];
    int nprims = 0;
    for (int P = 0; P < 6; ++P) {
        std::vector<hfg::HessPair> v;
        for (int x = 0; x < c->nshell; ++x)
            for (int y = 0; y <= x; ++y) {
                const int a = c->L[x] >= c->L[y] ? x : y, b = a == x ? y : x;
                if (c->L[a] == hfg::kPairLa[P] && c->L[b] == hfg::kPairLb[P]) v.push_back(hfg::HessPair{a, b, 0, 0});
            }
        auto prims = [&](const hfg::HessPair& p) { return c->nprim[p.sa] * c->nprim[p.sb]; };
        std::stable_sort(v.begin(), v.end(), [&](const auto& p, const auto& q) { return prims(p) > prims(q); });
        for (hfg::HessPair& p : v) {
            if (runs[P].empty() || runs[P].back().nprim != prims(p)) runs[P].push_back(Run{(int)pairs.size(), 0, prims(p)});
            ++runs[P].back().count;
            p.off = nprims;
            nprims += prims(p);
            pairs.push_back(p);
        }
    }
    // the items of every class: heavy runs first
    std::vector<hfg::HessSegment> segs;
    struct Launch {
        int P, Q, seg0, nseg;
        long long items;
    };
    std::vector<Launch> launches;
    for (int P = 5; P >= 0; --P)
        for (int Q = P; Q >= 0; --Q) {
            Launch l{P, Q, (int)segs.size(), 0, 0};
            const int per = hfg::item_prims(P, Q);
            for (size_t x = 0; x < runs[P].size(); ++x)
                for (size_t y = P == Q ? x : 0; y < runs[Q].size(); ++y) {
                    const Run &b = runs[P][x], &k = runs[Q][y];
                    hfg::HessSegment s{b.first, b.count, k.first, k.count, P == Q && x == y, 0, l.items};
                    s.chunks = std::max(1, (int)(((long long)b.nprim * k.nprim + per - 1) / per));
                    const long long q = s.tri ? (long long)b.count * (b.count + 1) / 2 : (long long)b.count * k.count;
                    l.items += q * s.chunks;
                    segs.push_back(s);
                }
            l.nseg = (int)segs.size() - l.seg0;
            if (l.items) launches.push_back(l);
        }
    // D, the Cartesian density, and the copies of the result that the workgroups add into
    const int copies = (int)std::max<size_t>(1, std::min<size_t>(64, ((size_t)1 << 20) / (2 * nh)));
    HFG_CHECK(c, c->d_one_buf.ensure(nn + (size_t)nc * nc + 2 * nh * (copies + 1)));
    HFG_CHECK(c, c->d_hess_pairs.upload(pairs, c->stream));
    HFG_CHECK(c, c->d_hess_segs.upload(segs, c->stream));
    HFG_CHECK(c, c->d_hess_prims.ensure(2 * (size_t)std::max(nprims, 1)));
    HFG_CHECK(c, c->d_hess_queue.ensure(32));
    double* dD = c->d_one_buf.p;
    double* dDc = dD + nn;
    double* dH = dDc + (size_t)nc * nc;
    HFG_CHECK(c, hipMemcpyAsync(dD, D, nn * sizeof(double), hipMemcpyHostToDevice, c->stream));
    HFG_CHECK(c, hipMemsetAsync(dH, 0, 2 * nh * copies * sizeof(double), c->stream));
    HFG_CHECK(c, hipMemsetAsync(c->d_hess_queue.p, 0, 32 * sizeof(unsigned long long), c->stream));
    if (c->pure)
        HFG_CHECK(c, hfg::launch_to_cart(dD, c->d_mols.p, c->d_mol_cart.p, 1, c->max_ncart, c->d_cart_terms.p, dDc, c->stream));
    hfg::HessArgs g{};
    g.sh = one.sh;
    g.alpha = one.alpha;
    g.coef = one.coef;
    g.xyz = one.xyz;
    g.rys = c->rys;
    g.pairs = c->d_hess_pairs.p;
    g.hp0 = c->d_hess_prims.p;
    g.hp1 = c->d_hess_prims.p + nprims;
    g.cart_off = c->d_cart_off.p;
    g.ncart = nc;
    g.natom = c->natom;
    g.npairs = (int)pairs.size();
    g.Dc = c->pure ? dDc : dD;
    g.prim_cut = c->opt.integral_tol / 1e4;
    // |K_ab K_cd| / sqrt(p + q) <= |K_ab| max(|K| / sqrt(p)), widened against rounding
    g.kmin = c->prim_mq > 0.0 ? g.prim_cut / c->prim_mq * (1.0 - 1e-12) : 0.0;
    g.H = dH;
    g.copies = copies;
    hipLaunchKernelGGL(hfg::hess_prim_kernel, dim3((unsigned)pairs.size()), dim3(64), 0, c->stream, g);
    HFG_CHECK(c, hipGetLastError());
    // the classes on the side streams in turn
    HFG_CHECK(c, hipEventRecord(c->ev_fork, c->stream));
    for (int k = 0; k < c->nside; ++k) HFG_CHECK(c, hipStreamWaitEvent(c->side[k], c->ev_fork, 0));
    for (size_t l = 0; l < launches.size(); ++l) {
        hfg::HessArgs b = g;
        b.segs = c->d_hess_segs.p + launches[l].seg0;
        b.nsegs = launches[l].nseg;
        b.nitems = launches[l].items;
        b.queue = c->d_hess_queue.p + l;
        HFG_CHECK(c, hfg::launch_rys_hess(launches[l].P, launches[l].Q, b, c->side[l % c->nside]));
    }
    for (int k = 0; k < c->nside; ++k) {
        HFG_CHECK(c, hipEventRecord(c->ev_join[k], c->side[k]));
        HFG_CHECK(c, hipStreamWaitEvent(c->stream, c->ev_join[k], 0));
    }
    double* dout = dH + 2 * nh * copies;
    hipLaunchKernelGGL(hfg::hess_sum_kernel, dim3((unsigned)std::max<size_t>(1, std::min<size_t>(1024, (2 * nh + 255) / 256))),
                       dim3(256), 0, c->stream, dH, copies, n3, dout);
    HFG_CHECK(c, hipGetLastError());
    HFG_CHECK(c, hipMemcpyAsync(HC, dout, nh * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HFG_CHECK(c, hipMemcpyAsync(HX, dout + nh, nh * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HFG_CHECK(c, hipStreamSynchronize(c->stream));
    return HFG_OK;
}

}  // extern "C"

// Host build of the rules that choose a class's kernel (context.hpp), for test_class_routes.py.
#include "../hfscf_amd/csrc/gpu/context.hpp"
#include "../hfscf_amd/csrc/gpu/grad_impl.hpp"

extern "C" int jk_runs_rys(int la, int lb, int lc, int ld, int mixed, int coop_min_l, long long quartets,
                           double longest_item, double heaviest_quartet) {
    hfg_ctx c;
    c.opt = hfg_options{};
    c.opt.coop_min_l = coop_min_l;
    hfg::ClassWork cw{};
    cw.la = la;
    cw.lb = lb;
    cw.lc = lc;
    cw.ld = ld;
    cw.quartets = quartets;
    cw.longest_item = longest_item;
    cw.heaviest_quartet = heaviest_quartet;
    return hfg::jk_on_rys(&c, cw, mixed != 0);
}

extern "C" int grad_first_prim(int k, int np) { return hfg::first_prim(k, np); }

// One-electron integrals of a single molecule on the GPU (S, T, V and their gradient terms).
#pragma once
#include <hip/hip_runtime.h>

struct hfg_ctx;

namespace hfg {

// A shell for the one-electron kernels: angular momentum, primitive count, offset of its
// exponents / normalised coefficients, atom.
struct OneShell {
    int L, np, po, atom;
};

struct OneArgs {
    const OneShell* sh;
    const double* alpha;
    const double* coef;
    const double* xyz;    // natom x 3, bohr
    const double* Z;      // nuclear charges
    const double* boys;   // the Boys table
    const int* cart_off;  // shell -> first Cartesian function
    int natom, ncart;
    double tiny;  // primitive pairs with a prefactor below it are skipped
    double* S;  // ncart x ncart outputs over the Cartesian functions (device)
    double* T;
    double* V;
};

// Device copies of the context's single molecule (shells, exponents, normalised coefficients,
// geometry, charges) into g; an HFG_ error code (message in the context) if it has none.
int one_upload(hfg_ctx* c, OneArgs& g);

}  // namespace hfg

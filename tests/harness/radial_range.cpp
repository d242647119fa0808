// Host driver of qg_radial.hpp under the address sanitizer: the table is an allocation of its own, so a
// value read outside it ends the run.  Prints the values at rel = xi - xi_min given in argv (in units of
// the table's step; "-inf" and "nan" too) for a table of n = argv[1] values 1, 2, 3, ...
#include <cstdio>
#include <cstdlib>
#include "../../qumasun_amd/csrc/qg_radial.hpp"

int main(int argc, char** argv) {
    const int n = std::atoi(argv[1]);
    double* v = new double[n];
    for (int k = 0; k < n; ++k) v[k] = 1.0 + k;
    for (int k = 2; k < argc; ++k) std::printf("%.17g\n", qg::radial_by_rel(0.25 * std::strtod(argv[k], nullptr), v, n, 0.25));
    delete[] v;
}

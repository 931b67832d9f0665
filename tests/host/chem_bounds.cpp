// calc_T of a mechanism table handed in as raw bytes, compiled with checks of
// every array index: prints the viscosity of one mixture, or stops at the
// first index outside its array.  Arguments: the table's file, T, then rho
// Y_k of eight species.  Test infrastructure only.
#define SHCFD_HD inline
#define __device__
#define __host__
#include <cstdio>
#include <cstdlib>

#include "../../shared_cfd_amd/csrc/shcfd_chem.h"

int main(int argc, char** argv) {
    static shcfd_mech m;
    FILE* f = argc == 11 ? std::fopen(argv[1], "rb") : nullptr;
    if (!f || std::fread(&m, sizeof(m), 1, f) != 1 || m.ns != 8) return 2;
    std::fclose(f);
    double rel[8], rho, E, T = std::atof(argv[2]);
    for (int k = 0; k < 8; k++) rel[k] = std::atof(argv[3 + k]);
    shcfd::chem::rho_rel2abs<8>(&m, 1.01325e5, T, rel, rho, E);
    shcfd::chem::ThermoOut<8> o;
    if (shcfd::chem::calc_t<8>(&m, rel, rho, E, T, o) < 0) return 3;
    std::printf("%.17g\n", o.mu);
    return 0;
}

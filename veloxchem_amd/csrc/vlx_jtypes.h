// Interface of the Coulomb build through Hermite densities (j_kernels.h) with the driver.
#pragma once

#include "vlx_types.h"

// Work item: bra entries [i0, i0 + JBLOCK) against ket entries [k0, k1).
struct JItem {
    int i0, k0, k1;
};
constexpr int j_nherm(int l) { return (l + 1) * (l + 2) * (l + 3) / 6; }
constexpr int JBLOCK = 256;
constexpr int j_row(int l) { return 4 + j_nherm(l); }  // doubles of an entry: zeta, P, H

struct JArgs {
    const double* bra;      // rows [entry][j_row(LAB)] of the bra rank
    const unsigned char* bra_bin;
    const double* ket;
    double* jp;             // [entry][j_nherm(LAB)]
    const JItem* items;
    const double* boys_tab; // for L = LAB + LCD
    const int* ket_cnt;     // entries of the ket list with bin <= b, 16 bins
    double omega2;
    int nbra, nitems, ithreshold;
};
// largest LAB + LCD: up to 165 values of R^0 per lane, past which they leave the registers (27 waters
// def2-TZVP, J: 71 ms up to 6 with the class kernels above it, 32 ms up to 8)
constexpr int J_LMAX = 8;

// Per-primitive steps of one pair class: its pairs and primitives, each primitive's pair, each pair's
// first entry in the list of its Hermite rank.
struct JPrep {
    const PairInfo* pairs;
    const PrimPair* prims;
    const int* pair_of;
    const int* entry0;
    int nprims, nao;
    const double* D;
    double* rows;
    double* jp;
    double factor;
    double* F;
};
void vlx_launch_j_density(int la, int lb, const JPrep& a, hipStream_t s);
void vlx_launch_j_fock(int la, int lb, const JPrep& a, hipStream_t s);
void vlx_launch_j(int lab, int lcd, const JArgs& a, hipStream_t s);

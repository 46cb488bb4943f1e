// angle_operands.hpp — which DST kernel a call takes, and the key of its cached
// operands (standard C++ only).
#pragma once

#include <algorithm>
#include <vector>

namespace bfpn {

// Whether FP32 planes run on the matrix cores: they hold planes of at most
// 32 x 32 directions and address a launch's planes with 32-bit offsets
// (launch_angle_mfma); other grids take the vector kernel.
inline bool angle_on_matrix_cores(int Nmu, int Nom, long long planes) {
    return Nmu <= 32 && Nom <= 32 && planes < (1LL << 30) && planes * Nmu * Nom < (1LL << 31);
}

// Whether FP64 planes run a line per thread (bases padded and blocked) or a value
// per thread.  Lines are the faster from 3 directions on (8 x 2 24 against 35 us,
// 21 x 21 nodes x 500 groups), but thin planes are mostly their padding to four:
// 1 x 20 directions 94 against 68 us, 27 x 2 211 against 142, 29 x 3 293 against
// 232.  Not where the value kernel's LDS columns fall on few banks: 1 x 16 56
// against 122 us, 2 x 24 142 against 302, 1 x 32 241 against 441.
inline bool angle_by_lines(int Nmu, int Nom) {
    const int least = std::min(Nmu, Nom), most = std::max(Nmu, Nom);
    const bool few_banks = most % 8 == 0 && most > 8;
    const bool thin = (least <= 2 && most > 4 * least) || (Nom == 3 && Nmu > 24);
    return most <= 32 && (!thin || few_banks);
}

// Everything the operands of one call are built from.  The kernel belongs to
// it: it depends on the number of planes, which the tables do not, and each
// kernel reads the bases in an order of its own.
inline std::vector<double> angle_operand_key(bool fp64, bool matrix_cores, int Ng, int Nmu, int Nom,
                                             double du, double dv, double dt, double rho,
                                             const double* sig_tr) {
    std::vector<double> key = {fp64 ? 1.0 : 0.0, matrix_cores ? 1.0 : 0.0, double(Ng), double(Nmu),
                               double(Nom), du, dv, dt, rho};
    key.insert(key.end(), sig_tr, sig_tr + Ng);
    return key;
}

}  // namespace bfpn

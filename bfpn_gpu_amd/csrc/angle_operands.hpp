// angle_operands.hpp — which DST kernel a call takes, and the key of its cached
// operands (standard C++ only).
#pragma once

#include <vector>

namespace bfpn {

// Whether FP32 planes run on the matrix cores: they hold planes of at most
// 32 x 32 directions and address a launch's planes with 32-bit offsets
// (launch_angle_mfma); other grids take the vector kernel.
inline bool angle_on_matrix_cores(int Nmu, int Nom, long long planes) {
    return Nmu <= 32 && Nom <= 32 && planes < (1LL << 30) && planes * Nmu * Nom < (1LL << 31);
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

// Host-visible interface of the linear RK4 stepper (linear_rk4.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace lime {

struct LinearArgs {
  int m, rows, nsteps, n_e;
  double dt;
  const double2* gen;      // [m][m] generator G
  const double2* eops;     // [n_e][m] or NULL
  double2* x;              // [rows][m] state vectors, updated in place
  double2* states;         // [nsteps][rows][m]
  double2* obs;            // [nsteps][rows][n_e] or NULL
};
size_t linear_workspace_bytes(int m);
hipError_t linear_run(const LinearArgs& a, void* work, hipStream_t stream);

}  // namespace lime

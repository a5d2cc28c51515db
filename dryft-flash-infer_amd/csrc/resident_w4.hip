// Resident-activation GEMM instances of FmtW4.
#include "resident.h"

int qlx::resident_w4a16(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream) {
  return resident_run<FmtW4>("linear_resident", a, m, n, k, plan, stream);
}

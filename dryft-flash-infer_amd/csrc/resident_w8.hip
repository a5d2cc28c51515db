// Resident-activation GEMM instances of FmtW8.
#include "resident.h"

int qlx::resident_w8a16(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream) {
  return resident_run<FmtW8>("linear_resident", a, m, n, k, plan, stream);
}

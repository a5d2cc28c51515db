// Resident-activation GEMM instances of FmtFP8.
#include "resident.h"

int qlx::resident_fp8(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream) {
  return resident_run<FmtFP8>("linear_resident", a, m, n, k, plan, stream);
}

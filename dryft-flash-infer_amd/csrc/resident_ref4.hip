// Resident-activation GEMM instances of FmtRef<4>.
#include "resident.h"

int qlx::resident_ref4(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream) {
  return resident_run<FmtRef<4>>("linear_resident", a, m, n, k, plan, stream);
}

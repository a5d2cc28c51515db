// Resident-activation GEMM instances of FmtRef<8>.
#include "resident.h"

int qlx::resident_ref8(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream) {
  return resident_run<FmtRef<8>>("linear_resident", a, m, n, k, plan, stream);
}

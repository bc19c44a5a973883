// The solver's quotients (magic_solver.h) on the host, for
// tests/test_solver_math.py.
#include "../magic_master_amd/csrc/magic_solver.h"

extern "C" void quotients(const double *num, const double *den, const double *rcp, double *out, int n)
{
    for (int i = 0; i < n; i++) out[i] = magic::quot(num[i], den[i], rcp[i]);
}

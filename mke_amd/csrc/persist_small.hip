// The persistent solve with workgroups of 256 threads (see krylov_block).
#define PS_BS 256
#include "persist_run.h"

namespace phg {

int persist_solve_small(phg_matrix_s* A, PersistWork* w, int K, const double* B, double* X,
                        const phg_gmres_opts& o, bool diag, bool stall, int max_cycles,
                        int max_rounds, int* launches, double* ms, hipStream_t s)
{
    return solve(A, w, K, B, X, o, diag, stall, max_cycles, max_rounds, launches, ms, s);
}

}  // namespace phg

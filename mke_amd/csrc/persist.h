// Restarted GMRES as persistent launches (persist.hip): the
// workspace that a matrix keeps for it, and its entry.
#pragma once
#include <algorithm>

#include "krylov.h"
#include "persist_turns.h"
#include "phg_internal.h"

namespace phg {

// Exchange rows in uncached device memory from a process-lifetime pool.
struct XchChunk {
    unsigned long long* p = nullptr;
    size_t n = 0;
    int dev = -1;
};
struct XchRows {
    XchChunk c;
    XchRows() = default;
    XchRows(const XchRows&) = delete;
    XchRows& operator=(const XchRows&) = delete;
    ~XchRows() { give_back(); }
    unsigned long long* p() const { return c.p; }
    void give_back();
    hipError_t alloc(size_t count);
};

// A column's state between launches, and its summary for the host.
struct PState {
    double bnorm, beta, rel;
    int iters, cycles, converged, active;
};

constexpr int PERSIST_NOT_HERE = 2;  // the shape does not run here: nothing was done
// Launches found no CUs for their workgroups: to be continued elsewhere.
// w->host[q]: a column with active = 1 and cycles = 0 has not begun (x as it
// was if it is a start vector, else undefined), with cycles > 0 it continues
// from x with cycle number `cycles`; one with active = 0 is complete.
constexpr int PERSIST_NO_START = 3;

struct PersistWork {
    DevBuf<char> W;              // the vector that the products gather, per column
    DevBuf<PState> st;           // per column
    DevBuf<int> abort_dev;       // per column
    PState* host = nullptr;      // pinned: host_k states, then the abort flag
    int host_k = 0;
    XchRows xch;                 // two rings of ring_slots words
    size_t ring_slots = 0;
    int ring_k = 0, ring_g = 0;  // shape of the launches since the rings were cleared
    int parity = 0;
    hipEvent_t ev[2] = {nullptr, nullptr};  // around each launch
    PersistWork() = default;
    PersistWork(const PersistWork&) = delete;
    PersistWork& operator=(const PersistWork&) = delete;
    ~PersistWork();
};

PersistTurns& persist_turns(int dev);  // of the device's launches

// Workgroups of n rows: of 512 threads 1024 rows each, of 256 threads (half
// of those 1024 rows each) two where the rows past the last 1024 need both.
inline int persist_workgroups(int n, int threads)
{
    const int pair = KR_STRIDE / threads, rows = KR_STRIDE * KR_RPT;
    return n / rows * pair + std::min(pair, (n % rows + threads - 1) / threads);
}

// A x_q = b_q for the K columns of B and X (n x K, row-major), each column by
// itself; o as gmres_batch_solve_pc takes it, also with PHG_MGS.  diag:
// right-preconditioned with the inverse diagonal (FP64).  stall: a column
// stops when a whole cycle lowers its residual by less than 1 %.  A launch
// runs at most max_cycles restart cycles of the columns that fit the device
// together; columns that need more than max_rounds launches do not run here.
// The columns' results are left in w->host.  launches (summed count) and ms
// (summed duration) may be null.
int persist_solve(phg_matrix_s* A, PersistWork* w, int K, const double* B, double* X,
                  const phg_gmres_opts& o, bool diag, bool stall, int max_cycles, int max_rounds,
                  int* launches, double* ms, hipStream_t s);

}  // namespace phg

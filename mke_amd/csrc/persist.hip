// Restarted GMRES(m), m <= 32, as persistent launches: all workgroups of a
// launch are resident, a column of the right-hand side belongs to G
// workgroups of 512 or 1024 rows each, and a restart cycle keeps everything
// that it owns on the chip.  A thread holds its rows of the work vector and of
// the matrix in registers and of the basis in LDS and registers; only the
// vector that the next product gathers goes through memory, and the global
// sums of an Arnoldi step go through an exchange (persist_run.h) instead of
// kernel boundaries.
//
// What bounds it: the exchanges, about 2.7 us each among 161 workgroups and
// 1.7 us among 41, and the instructions between them.  Level 7 FP64 MGS 11.5
// us a step (57 us with a sum per basis vector, 25.0 -> 5.1 ms a solve), level
// 4 7 us (1.37 -> 0.29 ms a solve), 36,503 rows FP32 CGS2 6.25 -> 1.77 ms.
// A step has two exchanges: the dots <v_i, w> of all basis vectors
// in one, ||w|| and, for modified Gram-Schmidt, the dots of the updated w in
// the other.  The latter are the products <v_i, v_{j+1}> that make
// modified Gram-Schmidt a triangular solve in the dots (mgs_solve), instead
// of a chain of j + 1 sums that each wait for the one before.  CGS2 has a
// third for its second pass.
//
// Columns are independent: each group of G workgroups runs its own cycles
// and stops by itself, so the batched solves of small meshes (gmres_batch)
// run here as one launch.
#include <map>
#include <mutex>

#define PS_BS 512
#include "persist_run.h"

namespace phg {

// ------------------------------------------------------ exchange memory --
// The exchange rows live in uncached device memory (hipDeviceMallocUncached):
// an agent-scope store of a partial and the loads that see it go to the
// memory side, not through each XCD's L2 (2.3 instead of 2.8 us per single
// sum across 161 workgroups).  Uncached memory that a kernel has read is
// never freed while the process runs (an allocation made later at its
// address may read stale data): a workspace hands its rows back to this pool
// when it is destroyed, after its last solve has synchronised, and the next
// workspace on the device takes them.
namespace {
std::mutex& xch_pool_mutex()
{
    static std::mutex* m = new std::mutex();  // kept until exit, like the pool
    return *m;
}
std::vector<XchChunk>& xch_pool()
{
    static std::vector<XchChunk>* v = new std::vector<XchChunk>();  // kept until exit
    return *v;
}
}  // namespace

void XchRows::give_back()
{
    if (!c.p) return;
    std::lock_guard<std::mutex> g(xch_pool_mutex());
    xch_pool().push_back(c);
    c = XchChunk();
}

// at least count slots on the current device: the smallest pooled chunk
// that holds them, else a new allocation
hipError_t XchRows::alloc(size_t count)
{
    give_back();
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    {
        std::lock_guard<std::mutex> g(xch_pool_mutex());
        std::vector<XchChunk>& pool = xch_pool();
        size_t best = pool.size();
        for (size_t i = 0; i < pool.size(); ++i)
            if (pool[i].dev == dev && pool[i].n >= count &&
                (best == pool.size() || pool[i].n < pool[best].n))
                best = i;
        if (best < pool.size()) {
            c = pool[best];
            pool.erase(pool.begin() + (std::ptrdiff_t)best);
            return hipSuccess;
        }
    }
    void* q = nullptr;
    e = hipExtMallocWithFlags(&q, count * sizeof(unsigned long long), hipDeviceMallocUncached);
    if (e != hipSuccess) return e;
    c.p = (unsigned long long*)q;
    c.n = count;
    c.dev = dev;
    return hipSuccess;
}

PersistWork::~PersistWork()
{
    for (hipEvent_t e : ev)
        if (e) (void)hipEventDestroy(e);
    if (host) (void)hipHostFree(host);
}

PersistTurns& persist_turns(int dev)
{
    static std::mutex mu;
    static std::map<int, PersistTurns>* m = new std::map<int, PersistTurns>();  // kept until exit
    std::lock_guard<std::mutex> l(mu);
    auto it = m->find(dev);
    if (it == m->end()) {
        int cus = 0;
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        it = m->try_emplace(dev, cus).first;
    }
    return it->second;
}

void persist_destroy(PersistWork* w) { delete w; }

int persist_solve_small(phg_matrix_s* A, PersistWork* w, int K, const double* B, double* X,
                        const phg_gmres_opts& o, bool diag, bool stall, int max_cycles,
                        int max_rounds, int* launches, double* ms, hipStream_t s);

// Workgroups of 256 threads wherever all columns fit the device with them: a
// SIMD then runs one wavefront instead of two, and a step is instructions
// beside its exchanges; the results are the same bits.  Measured with 512 and
// with 256 threads: level 4 FP64 MGS 371 and 305 us a solve, 7 columns of
// 9,991 rows FP64 CGS2 1.03 and 0.85 ms, 36,503 rows FP32 CGS2 1.89 and
// 1.88 ms.  Columns that would need more launches than with 512 threads are
// faster with those.
int persist_solve(phg_matrix_s* A, PersistWork* w, int K, const double* B, double* X,
                  const phg_gmres_opts& o, bool diag, bool stall, int max_cycles, int max_rounds,
                  int* launches, double* ms, hipStream_t s)
{
    if ((long)persist_workgroups(A->n_rows, 256) * K <= KR_MAXG) {
        const int rc = persist_solve_small(A, w, K, B, X, o, diag, stall, max_cycles, max_rounds,
                                           launches, ms, s);
        if (rc != PERSIST_NOT_HERE) return rc;
    }
    return solve(A, w, K, B, X, o, diag, stall, max_cycles, max_rounds, launches, ms, s);
}

}  // namespace phg

// Host interface of the resident BiCGStab (pb_resident2d.hip): whole Krylov
// runs in one launch, the vectors held in registers.
#pragma once
#include <functional>

#include "pb_bicg2d.hpp"

namespace pb2d {

// Result record of a member's run, written by the launch.
struct ResOut {
  KState st;
  int abort;   // a bounded wait ran out: the run is void and is done by launches
  int pad;
};

// Launch records of a run, owned by the operator or batch it belongs to: the
// member table followed by the results, on the device and as a pinned mirror,
// and the counter that hands blocks their tiles.
struct ResRecords {
  void* dev = nullptr;
  void* host = nullptr;
  size_t bytes = 0;
  unsigned* ticket = nullptr;
  unsigned ticket_next = 0;
  void release();
};

// Device words of one operator's resident runs: the edge exchange, the
// partial records and their sums, all tagged.  One allocation, made at the
// first run that fits on the chip.
struct Resident {
  unsigned long long* words = nullptr;
  long halo_words = 0;   // of one exchange buffer (there are two)
  long rec_words = 0;
  unsigned epoch = 0;    // no tag above it has been used
  bool cleared = false;
  ResRecords records;    // of the operator's own runs
};

template <typename T>
struct ResJob {
  pb_op2d* op;
  const T* b;          // right-hand side
  const T* r0;         // b - A x0 (b itself for a zero guess)
  const double* x0;    // initial iterate, null: zero
  double* x;           // result
  double tol;
  int maxiter, legacy;
};

// The operator's Resident, made at the first call, still without device memory.
Resident* resident_of(pb_op2d* op);

// Run every job with the launch records ``rec`` of their owner, in as few
// launches as the operator kinds and the tiles resident at once allow.
// ``prepare`` issues on ``s`` what the jobs' inputs still need; it is called once
// the runs are known to fit.  Returns 1 with the final states in ``out`` when all
// of them ran, 0 when they do not apply here (grid too large to be resident, no
// free room or memory, or a wait ran out: the caller takes the launch-per-phase
// path), < 0 on an error.
template <typename T>
int resident_run(pb_ctx* ctx, ResRecords& rec, const ResJob<T>* jobs, int count, bool exact, hipStream_t s,
                 KState* out, const std::function<void()>& prepare = {});

void resident_free(pb_op2d* op);

}  // namespace pb2d

// fc3d_batch.hpp — what the batched solver shares with the single problem's.
#pragma once
#include <vector>

#include "fc3d_layout.hpp"
#include "fc3d_sweep.hpp"

namespace fc3d {

struct BatchProblem {
  int cptr_off;     // first entry of the problem's colour slice pointers
  int ncolours;
  int slice_begin;
  int slice_end;
  double norm_q;
};

// Numbers each problem's contacts from 0 in slot order: cbase per slice, ccol
// per plane entry (at most 65536 contacts a problem).
void number_contacts(const HostLayout& L, const std::vector<BatchProblem>& problems,
                     std::vector<int>* cbase, std::vector<unsigned short>* ccol);

// One FP64 solve of a small problem in one workgroup of two quads: the
// device block that goes in before the launch and comes back after it.
struct SmallSolve {
  BatchProblem problem;
  int order, counter;                  // the queue of one problem
  int info, iterations, fp32_iterations;
  double residual, incr;
};
int launch_small_solve(const SweepPtrs<double>& P, const int* cptr, const int* cbase,
                       const unsigned short* ccol, int nc, const DevParams* prm, SmallSolve* d,
                       hipStream_t s);

}  // namespace fc3d

// fc3d_batch_rule.hpp — when the batched solver gives a problem a quad of waves
// with the reactions in LDS (sweep_quads).  Host arithmetic only.
#pragma once

namespace fc3d {

// Slices that a sweep of the batch's problems steps through, one after the
// other: by a quad (every slice of every colour) and by four waves that take a
// colour's slices side by side.
struct QuadRule {
  long long quad = 0, four = 0;  // of all problems
  int quad_max = 0, four_max = 0;  // of the longest problem

  // colour c of the problem holds slices [cptr[c], cptr[c + 1])
  void add(const int* cptr, int ncolours) {
    int s = 0, f = 0;
    for (int c = 0; c < ncolours; c++) {
      s += cptr[c + 1] - cptr[c];
      f += (cptr[c + 1] - cptr[c] + 3) / 4;
    }
    quad += s;
    four += f;
    quad_max = quad_max > s ? quad_max : s;
    four_max = four_max > f ? four_max : f;
  }

  // A quad's step is the shorter (it gathers one slice while it solves another:
  // 7-10 us against 9-16 in FP64, 3-6 against 4-8 in FP32), but it takes one
  // slice where four waves take up to four.  Time of four waves / of a quad by
  // the ratio of the steps, over random pairs, piles and chains of 200-2048
  // contacts, 16 and 256 problems, FP64 and mixed: 1.0-1.15: 1.19-1.5; 1.3:
  // 0.99-1.36; 1.4: 1.00-1.27; 1.55: 0.88-1.18; 1.7: 0.8-0.9; 2 and more:
  // 0.33-0.97.  Both the longest problem, which a launch of few problems waits
  // for, and the sum, which a full chip works through, have to be below 1.4.
  bool quads() const { return 5 * quad_max <= 7 * four_max && 5 * quad <= 7 * four; }

  // Whether quads take the batch without a trial against one wave a problem.
  // While every problem has a quad of its own (slots: the quads that the device
  // holds) they are the faster ones: 1.1-1.6 of the one wave's rate, FP64 and
  // mixed; only at two steps a sweep (chains of 20 and 60 contacts), where a
  // solve is its start and its end, 0.89-1.1.  Beyond that, one wave a problem
  // has the higher throughput and the quads reach the end of the slow problems
  // sooner; a trial of a few sweeps sees only the former.  The end decides
  // while the longest problem's steps go round few times (rounds below) and the
  // problems' sweeps differ: to 1e-6 within 1000 sweeps quads have 1.1-1.4 of
  // the one wave's rate in FP64 and 0.98-1.4 mixed at 0.9-2.9 rounds (600-2048
  // problems), 0.80-1.2 at 3.9.  A loose tolerance (1e-3: down to 0.87 at 1.5
  // rounds, mixed, and 0.83 at 2), a small limit on the sweeps (100: 0.84 and
  // 0.73) or none to stop before it (30: 0.79 and 0.53) lets the problems end
  // together.
  bool no_trial(int problems, int slots, int max_iter, double tol) const {
    if (!quads() || quad_max < 6) return false;
    if (problems <= slots) return true;
    const double rounds = double(quad) / (double(slots) * quad_max);
    return tol > 0.0 && ((rounds <= 1.5 && tol <= 1e-4 && max_iter >= 400) ||
                         (rounds <= 3.0 && tol <= 1e-6 && max_iter >= 1000));
  }
};

}  // namespace fc3d

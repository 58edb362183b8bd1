"""The batched solver's choice between quads of waves and the other forms
(fc3d_batch_rule.hpp), on the CPU: batches given by the contacts of each colour
of their problems, on both sides of where the measured times cross."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <vector>
#include "fc3d_batch_rule.hpp"
int main() {
  int problems, max_iter;
  double tol;
  if (std::scanf("%d %d %lf", &problems, &max_iter, &tol) != 3) return 1;
  fc3d::QuadRule rule;
  for (int p = 0; p < problems; p++) {
    int n;
    if (std::scanf("%d", &n) != 1) return 1;
    std::vector<int> cptr(1, 5);  // (a problem's slices need not start at 0)
    for (int c = 0; c < n; c++) {
      int contacts;
      if (std::scanf("%d", &contacts) != 1) return 1;
      cptr.push_back(cptr.back() + (contacts + 63) / 64);
    }
    rule.add(cptr.data(), n);
  }
  std::printf("%d %d\\n", rule.quads(), rule.no_trial(problems, 512, max_iter, tol));
}
"""

P200 = [15] * 14               # 200 contacts of 80 spheres
P600 = [90] * 5 + [45] * 8     # 600 contacts of 240: 18 steps against 13
P1300 = [200] * 4 + [130] * 4 + [60] * 7   # 1300 of 520: 35 against 15
CHAIN60 = [30, 30]
CHAIN200 = [100, 100]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is needed to compile the rule")
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I",
                    os.path.join(REPO, "siconos_amd", "csrc", "hip"), str(d / "rule.cpp"), "-o",
                    str(d / "rule")], check=True)

    def ask(problems, max_iter=1000, tol=1e-6):
        text = f"{len(problems)} {max_iter} {tol}\n" + "\n".join(
            " ".join(map(str, [len(p), *p])) for p in problems)
        out = subprocess.run([str(d / "rule")], input=text, check=True, capture_output=True,
                             text=True).stdout.split()
        return out[0] == "1", out[1] == "1"
    return ask


@pytest.mark.parametrize("problems,quads,no_trial", [
    ([P200] * 16, True, True),
    ([P600] * 16, True, True),
    ([P1300] * 16, False, False),             # four waves take a colour's slices together
    ([CHAIN200] * 16, False, False),
    ([CHAIN60] * 16, True, False),            # two steps a sweep: the trial decides
    ([P1300] + [CHAIN60] * 200, False, False),  # the longest problem is waited for
    ([P200] * 4 + [CHAIN200] * 200, False, False),  # the sum fills the chip
    ([P200] * 512, True, True),
    ([P200] * 768, True, True),
    ([P200] * 1536, True, True),
    ([P200] * 1537, True, False),             # more than 3 rounds
    ([P200] + [CHAIN60] * 1500, True, True),  # (rounds count steps, not problems)
])
def test_form_of_a_batch(rule, problems, quads, no_trial):
    assert rule(problems) == (quads, no_trial)


def test_trial_where_every_problem_runs_as_long(rule):
    """Beyond a quad a problem, a limit on the sweeps or a tolerance that none
    or all reach soon lets the problems end together: the trial decides."""
    assert rule([P200] * 700, tol=1e-4) == (True, True)
    assert rule([P200] * 700, tol=1e-3) == (True, False)
    assert rule([P200] * 700, max_iter=399) == (True, False)
    assert rule([P200] * 700, tol=0.0) == (True, False)
    assert rule([P200] * 768, max_iter=400) == (True, True)
    assert rule([P200] * 769, max_iter=999) == (True, False)
    assert rule([P200] * 769, tol=1e-5) == (True, False)
    assert rule([P200] * 512, max_iter=30, tol=0.0) == (True, True)

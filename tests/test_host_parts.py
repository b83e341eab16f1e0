"""CPU checks of host code that has no entry point of its own, compiled here against stand-ins of
what it calls."""
import subprocess

from conftest import ROOT

CSRC = ROOT / "pagedattention-based-transformer-decoder-inference-framework_amd" / "csrc"


def run(tmp_path, code, *flags):
    (tmp_path / "t.cpp").write_text(code)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", f"-I{ROOT / 'include'}", *flags,
                    "-o", str(tmp_path / "t"), str(tmp_path / "t.cpp")], check=True)
    return subprocess.run([str(tmp_path / "t")], check=True, capture_output=True, text=True).stdout.split()


def test_step_put_keeps_no_place_behind_a_failed_launch(tmp_path):
    """Any launch of a step's words may fail: what the host believes of the logits' place is what the
    device holds, and the next step without logits clears it."""
    out = run(tmp_path, """
#include <cstdio>
#include <vector>
#include "step_put.hpp"
using namespace llm;
int main() {
  float mine = 0.f;
  for (int rows : {1, 128, 129, 300})
    for (int fails = 0; fails < 5; ++fails) {
      std::vector<int32_t> to(rows, -1), tokens(rows);
      for (int i = 0; i < rows; ++i) tokens[i] = 7 * i;
      float* place = nullptr;
      bool placed = false;
      int left = fails, launches = 0;
      const auto launch = [&](const StepPut& a) {
        if (left-- == 0) return 5;
        ++launches;
        for (int i = 0; i < a.n; ++i) a.to[i] = a.v[i];
        if (a.place) *a.place = a.logits;
        return 0;
      };
      const int rc = put_step(tokens.data(), rows, to.data(), &place, &mine, placed, launch);
      if (placed != (place != nullptr)) return 1;
      if (rc == 0 && (place != &mine || to != tokens || launches != (rows + 127) / 128)) return 2;
      if (rc != 0 && (rc != 5 || placed)) return 3;
      left = -1;
      if (put_step(nullptr, rows, to.data(), &place, nullptr, placed, launch) || place || placed) return 4;
      launches = 0;
      if (put_step(nullptr, rows, to.data(), &place, nullptr, placed, launch) || launches) return 5;
    }
  std::puts("ok");
}
""")
    assert out == ["ok"]

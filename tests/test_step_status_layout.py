"""The step status's layout: the face-list counters, cleared by plain stores of
one block, lie in no 128-byte line that other blocks of that launch read or
update."""
import pathlib
import subprocess


CSRC = pathlib.Path(__file__).resolve().parents[1] / "quasar_amd" / "csrc"

SOURCE = """
#include "qmhd_kernels.hpp"
#include <cstddef>
using qmhd::StepStatus;
constexpr std::size_t line(std::size_t at) { return at / 128; }
static_assert(alignof(StepStatus) % 128 == 0, "a line starts the status");
static_assert(line(offsetof(StepStatus, lists)) != line(offsetof(StepStatus, theta)), "");
static_assert(line(offsetof(StepStatus, lists)) != line(offsetof(StepStatus, live_theta1)), "");
static_assert(line(offsetof(StepStatus, lists)) != line(offsetof(StepStatus, divb_scale)), "");
static_assert(line(offsetof(StepStatus, lists)) != line(offsetof(StepStatus, max_rate)), "");
static_assert(line(offsetof(StepStatus, lists)) != line(offsetof(StepStatus, dt)), "");
static_assert(line(sizeof(StepStatus) - 1) == line(offsetof(StepStatus, lists)), "nothing shares the counters' line");
int main() {}
"""


def test_list_counters_have_a_line_of_their_own(tmp_path):
    src = tmp_path / "layout.cpp"
    src.write_text(SOURCE)
    done = subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-std=c++17", "-fsyntax-only",
                           f"-I{CSRC}", str(src)], capture_output=True, text=True)
    assert done.returncode == 0, done.stderr[-2000:]

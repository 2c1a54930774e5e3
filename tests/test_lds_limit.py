"""The dynamic LDS limit of a kernel is raised on every device that launches it, remembered only after success, and never
lowered (``csrc/lds_limit.h``, compiled here for the host)."""

import re
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "blksprs_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "lds_limit.h"

#define CHECK(cond) if (!(cond)) { std::printf("line %d: %s\n", __LINE__, #cond); return 1; }

int main() {
  bsa::LdsLimit limit;
  int calls = 0, answer = 0;
  auto set = [&] { ++calls; return answer; };
  // a second device is raised too, each one once
  CHECK(limit.raise(0, 70000, set) == 0 && calls == 1);
  CHECK(limit.raise(0, 70000, set) == 0 && calls == 1);
  CHECK(limit.raise(1, 70000, set) == 0 && calls == 2);
  CHECK(limit.raise(1, 70000, set) == 0 && calls == 2);
  // more than before is raised again, less is not
  CHECK(limit.raise(0, 90000, set) == 0 && calls == 3);
  CHECK(limit.raise(0, 80000, set) == 0 && calls == 3);
  CHECK(limit.raise(1, 80000, set) == 0 && calls == 4);
  // a failure is handed on and not remembered
  answer = 7;
  CHECK(limit.raise(2, 70000, set) == 7 && calls == 5);
  answer = 0;
  CHECK(limit.raise(2, 70000, set) == 0 && calls == 6);
  // a device beyond those that are tracked: every time
  CHECK(limit.raise(64, 70000, set) == 0 && limit.raise(64, 70000, set) == 0 && limit.raise(-1, 70000, set) == 0 && calls == 9);
  // several threads with different demands: what is set last is the largest
  for (int round = 0; round < 200; ++round) {
    bsa::LdsLimit shared;
    int attribute = 0;
    std::vector<std::thread> threads;
    for (int t = 0; t < 4; ++t)
      threads.emplace_back([&, t] { shared.raise(0, 70000 + 1000 * t, [&] { attribute = 70000 + 1000 * t; return 0; }); });
    for (auto &t : threads) t.join();
    CHECK(attribute == 73000);
  }
  return 0;
}
"""


def test_limit_is_kept_per_device_and_only_after_success(tmp_path):
    (tmp_path / "check.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{CSRC}", "check.cpp", "-o", "check"], cwd=tmp_path, check=True)
    done = subprocess.run([str(tmp_path / "check")], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout


def test_every_launch_raises_its_limit_that_way():
    """No source sets the attribute by itself, and none keeps a flag per process beside it."""
    for path in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")):
        uses = re.findall(r"\bhipFuncSetAttribute\(", path.read_text())
        assert len(uses) == (1 if path.name == "common.h" else 0), path.name

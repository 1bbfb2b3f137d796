"""One-time work per device (csrc/device_once.h), compiled with the host compiler: every device gets its own, concurrent
first callers see it finished, a failure is tried again.  And every function of the library that raises a kernel's limit
of dynamic LDS goes through it or does the work on each call: none keeps one flag for the whole process."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "llmxabe_amd", "csrc")

PROGRAM = r"""
#include <stdio.h>
#include <atomic>
#include <thread>
#include <vector>
#include "device_once.h"
#define REQUIRE(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
  xabe::DeviceOnce once;
  int calls[3] = {0, 0, 0};
  for (int round = 0; round < 2; ++round)
    for (int d = 0; d < 3; ++d) REQUIRE(once.run(d, [&] { ++calls[d]; return 0; }) == 0);
  REQUIRE(calls[0] == 1 && calls[1] == 1 && calls[2] == 1);
  int tries = 0;
  REQUIRE(once.run(7, [&] { ++tries; return 5; }) == 5);
  REQUIRE(once.run(7, [&] { ++tries; return 0; }) == 0);
  REQUIRE(once.run(7, [&] { ++tries; return 9; }) == 0 && tries == 2);
  int outside = 0;
  for (int i = 0; i < 2; ++i) REQUIRE(once.run(xabe::kMaxDevices, [&] { ++outside; return 0; }) == 0);
  REQUIRE(outside == 2);
  std::atomic<int> ran{0}, early{0};
  std::vector<std::thread> threads;
  for (int i = 0; i < 8; ++i)
    threads.emplace_back([&] {
      once.run(11, [&] { std::this_thread::sleep_for(std::chrono::milliseconds(50)); ++ran; return 0; });
      if (ran != 1) ++early;
    });
  for (auto& t : threads) t.join();
  REQUIRE(ran == 1 && early == 0);
  return 0;
}
"""


def test_once_per_device_with_threads_and_failures(tmp_path):
    src = tmp_path / "once.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "once"
    subprocess.check_call(["g++", "-std=c++17", "-pthread", "-I", CSRC, str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_no_configuration_is_kept_in_a_flag_of_the_process():
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".h")):
            text = open(os.path.join(CSRC, name)).read()
            assert not re.search(r"static\s+bool\s+\w+\s*=\s*false", text), name

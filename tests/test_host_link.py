"""The helper threads of the host transfers: a process that forks after a transfer (a host engine's
worker pool) must be able to leave the child, which has none of them, in the ordinary way."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include "host_link.h"
#include <signal.h>
#include <sys/wait.h>
#include <cstdlib>
using namespace csk;
static CrewOwner crew;
static char a[(1 << 20) + 77], b[17 << 16];
int main() {
  for (size_t i = 0; i < sizeof a; ++i) a[i] = (char)(i * 7 + i / 251);
  const CopyCrew::Job j{a, b, sizeof a, 0, sizeof b, true};
  if (!crew.ready() || !crew->begin(j)) return 2;
  crew->open_to(j.pieces());
  while (crew->work_one()) {}
  for (long i = 0; i < j.pieces(); ++i)
    while (!crew->done(i)) CopyCrew::relax();
  crew->end();
  if (std::memcmp(a, b, sizeof a)) return 3;
  usleep(100000);  // the helpers are asleep by now
  const pid_t p = fork();
  if (p == 0) std::exit(0);
  int st = 0;
  for (int i = 0; i < 100; ++i, usleep(50000))
    if (waitpid(p, &st, WNOHANG) == p) return st == 0 ? 0 : 4;
  kill(p, SIGKILL);
  return 5;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_forked_child_exits(tmp_path):
    src, exe = tmp_path / "fork_check.hip", tmp_path / "fork_check"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I" + os.path.join(ROOT, "coalsack_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                    str(src), "-o", str(exe), "-pthread"], check=True, capture_output=True, timeout=300)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0

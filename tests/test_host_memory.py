"""afid_amd/csrc/host_memory.h on the CPU: which buffers count as pinned memory
that a kernel may write, over allocations a made-up runtime reports."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# Two pinned allocations at equal host and device addresses with ordinary memory
# between them, one pinned at another device address, one of device memory.
PROGRAM = r"""
#include "host_memory.h"
#include <cstdio>
#include <cstdlib>
using namespace afid;
struct Row { uintptr_t base; size_t size; bool host; uintptr_t device; };
static const Row rows[] = {{0x10000, 0x1000, true, 0x10000},
                           {0x14000, 0x1000, true, 0x14000},
                           {0x20000, 0x1000, true, 0x90000},
                           {0x30000, 0x1000, false, 0x30000}};
int main(int argc, char **argv) {
  auto lookup = [](uintptr_t a, Allocation *o) {
    for (const Row &r : rows)
      if (a >= r.base && a < r.base + r.size) {
        o->host = r.host; o->base = r.base; o->size = r.size; o->device = r.device;
        return true;
      }
    return false;
  };
  uintptr_t device = 0;
  const HostKind k = host_kind((const void *)strtoull(argv[1], nullptr, 16), strtoull(argv[2], nullptr, 16), lookup, &device);
  printf("%s %llx\n", k == HostKind::ordinary ? "ordinary" : k == HostKind::pinned ? "pinned" : "other",
         (unsigned long long)device);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_memory")
    src, exe = d / "t.cpp", d / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{os.path.join(ROOT, 'afid_amd', 'csrc')}", str(src), "-o",
                    str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("p,n,want", [
    (0x10000, 0x1000, "pinned 10000"),     # all of one allocation
    (0x10008, 0x0ff8, "pinned 10008"),     # its end
    (0x20010, 0x0010, "pinned 90010"),     # at another device address
    (0x10000, 0x1001, "other 0"),          # one byte too long
    (0x10008, 0x4808, "other 0"),          # into the next one, unmapped memory between them
    (0x0fff8, 0x0100, "other 0"),          # begins before it
    (0x30000, 0x0100, "other 0"),          # not the host's
    (0x40000, 0x0100, "ordinary 0"),
    (0x0f000, 0x0100, "ordinary 0"),
])
def test_host_kind(program, p, n, want):
    out = subprocess.run([program, f"{p:x}", f"{n:x}"], capture_output=True, text=True, check=True).stdout
    assert out.strip() == want

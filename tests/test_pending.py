"""The batch solve's host flags (mcnla_amd/csrc/pending.hpp) on the CPU: when an error unwinds the
solve while device-to-host copies are queued, the memory they write is not given back before the
wait for them has returned.  In this program the wait looks whether the memory is still there."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdlib>
#include <new>
#include <stdexcept>

#include "pending.hpp"

static void* watched = nullptr;
static bool freed = false;

void* operator new(std::size_t n) {
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept {
  if (p == watched) freed = true;
  std::free(p);
}
void operator delete(void* p, std::size_t) noexcept { operator delete(p); }

int main() {
  int waits = 0;
  bool early = false;
  auto wait = [&] {
    ++waits;
    early = early || freed;
  };
  try {
    mcnla::PendingInts flags(16, wait);
    watched = flags.at(0);
    throw std::runtime_error("a later call fails");
  } catch (const std::runtime_error&) {
  }
  if (waits != 1 || early || !freed) return 1;
  {  // without an error: they have landed, and the destructor does not wait
    mcnla::PendingInts flags(2, wait);
    *flags.at(1) = 7;
    flags.landed();
    if (flags[0] != 0 || flags[1] != 7) return 2;
  }
  return waits == 1 ? 0 : 3;
}
"""


def test_flags_outlive_their_copies(tmp_path):
    src, exe = tmp_path / "pending.cpp", tmp_path / "pending"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I",
                    os.path.join(ROOT, "mcnla_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0

"""The chunks a stack is cut into, against the buffers of their partial sums (host code, compiled
here): a stack of any length writes no more chunks than a full stack has planes for and leaves
out no slot, whatever the workgroups per chunk (frame side, modes and precision), the launch
targets and the stack size."""

import subprocess

from conftest import ROOT

PROGRAM = r"""
#include <cstdio>
#include "host.hpp"

int main() {
  using namespace ptyrs;
  long beyond = 0, tried = 0;
  for (int per = 1; per <= 512; ++per)
    for (int blocks : {1, 12, 96, 384, 768, 1000, 1024, 6144, 8192})
      for (int stack : {1, 7, 16, 32, 64, 100, 128, 256}) {
        const int full = chunk_len(stack, per, blocks);
        const int planes = (stack + full - 1) / full;
        for (int nb = 1; nb <= stack; ++nb) {
          const int own = chunk_len(nb, per, blocks), chunk = chunk_within(own, nb, planes);
          const int count = (nb + chunk - 1) / chunk, free = (nb + own - 1) / own;
          ++tried;
          beyond += free > planes;
          if (count > planes || count * chunk < nb || (count - 1) * chunk >= nb ||
              (free <= planes && chunk != own) || (nb == stack && chunk != full)) {
            std::printf("per %d blocks %d stack %d nb %d: %d chunks of %d in %d planes\n", per,
                        blocks, stack, nb, count, chunk, planes);
            return 1;
          }
        }
      }
  std::printf("%ld %ld\n", tried, beyond);
  return 0;
}
"""


def test_every_stack_fits_the_full_stacks_planes(tmp_path):
    (tmp_path / "chunks.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", str(ROOT / "ptyrs_amd" / "csrc"),
                    str(tmp_path / "chunks.cpp"), "-o", str(tmp_path / "chunks")], check=True)
    run = subprocess.run([str(tmp_path / "chunks")], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
    # The bound is needed: without it some short stacks cut more chunks than a full one.
    tried, beyond = map(int, run.stdout.split())
    assert 0 < beyond < tried

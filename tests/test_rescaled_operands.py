"""The key switch fused with the rescale (hck::ks_rescaled, FP64 words): its last sums stay below 8 p <= 2^53,
i.e. exact, with one kind of addend.  A call with two kinds is refused on the host, before any launch; the
check needs no device, and the program that makes the calls sees none."""

import os
import shutil
import subprocess

import pytest

from holmes_amd import build as hb

MAIN = r"""
#include <cstdio>

#include "holmes_ckks.h"
#include "internal.hpp"

int main() {
  hck_context c{};
  c.log_n = 16, c.L = 4, c.K = 2, c.alpha = 2, c.beta_max = 2, c.np = 6;
  uint64_t word = 0, *p = &word;
  const uint64_t* keys[1] = {p};
  const uint64_t* prod[4] = {p, p, p, p};
  auto call = [&](bool acc, bool tensor) {
    return hck::ks_rescaled(&c, 3, 1, p, 0, 1u, keys, p, 0, acc ? p : nullptr, acc ? p : nullptr, 0, p, p, 0, (char*)p,
                            nullptr, 0, nullptr, nullptr, 0, nullptr, tensor ? prod : nullptr, 0, 0);
  };
  std::printf("%d %d %d %d\n", HCK_ERR_ARG, call(true, false), call(false, true), call(true, true));
}
"""


@pytest.mark.skipif(shutil.which(hb.HIPCC) is None, reason="hipcc is not installed")
def test_two_kinds_of_addend_are_refused(tmp_path):
    src, obj, exe = (tmp_path / n for n in ("main.hip", "main.o", "main"))
    src.write_text(MAIN)
    hb.LIB.exists() or hb.build()
    for cmd in ([*hb.FLAGS, "--cuda-host-only", f"-I{hb.CSRC}", "-c", str(src), "-o", str(obj)],
                [str(obj), f"-L{hb.LIB.parent}", "-lholmes_ckks", f"-Wl,-rpath,{hb.LIB.parent}", "-o", str(exe)]):
        subprocess.run([hb.HIPCC, *cmd], check=True, capture_output=True)
    run = subprocess.run([str(exe)], env={**os.environ, "HIP_VISIBLE_DEVICES": "-1"}, capture_output=True, text=True)
    want, *got = run.stdout.split()
    assert got == [want] * 3, run.stderr

"""What a split and a launch that counts blocks keep in the same words of the forward's arguments (csrc/hbsa_common.h): the second writer is refused,
and a launch finds out when the words are not what its kernel reads."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "hbsa_common.h"
using namespace hbsa;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

FwdParams fresh(int nparts) {
  FwdParams fp;
  std::memset(&fp, 0, sizeof(fp));
  fp.nparts = nparts;
  return fp;
}

int main() {
  float out, lse;
  int32_t counts[4];
  FwdParams plain = fresh(1);
  CHECK(unions_fit(plain, false) && !unions_fit(plain, true));
  FwdParams unset = fresh(3);   // a split without its room
  CHECK(!unions_fit(unset, false) && !unions_fit(unset, true));
  FwdParams cut = fresh(3);
  CHECK(put_parts(cut, &out, &lse) && unions_fit(cut, false) && !unions_fit(cut, true));
  CHECK(!put_counts(cut, counts, 7, 3) && cut.part_out == &out && cut.part_lse == &lse && unions_fit(cut, false));
  FwdParams counted = fresh(1);
  CHECK(put_counts(counted, counts, 7, 3) && unions_fit(counted, true) && !unions_fit(counted, false));
  CHECK(!put_parts(counted, &out, &lse) && counted.counts == counts && counted.count_info[0] == 7 && counted.count_info[1] == 3);
  counted.nparts = 2;
  CHECK(!unions_fit(counted, true) && !unions_fit(counted, false));
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_the_words_have_one_writer(tmp_path):
    source = tmp_path / "args.hip"
    source.write_text(PROGRAM)
    binary = str(tmp_path / "args")
    subprocess.run(["hipcc", "--offload-arch=gfx950", "--offload-host-only", "-O0", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "hbsattn_amd", "csrc"), str(source), "-o", binary], check=True)
    res = subprocess.run([binary], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr

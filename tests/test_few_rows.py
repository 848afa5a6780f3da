"""The pitch of the few-token launches' rows in LDS (no GPU)."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-kunlun_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "few_rows.h"
int main() {
  for (int bytes = 1; bytes <= 2; ++bytes)
    for (int scales = 0; scales <= (bytes == 1); ++scales)
      for (int values = scales ? 128 : 32; values <= 25600; values += scales ? 128 : 32) {
        const int needed = values * bytes + (scales ? values / 128 * 4 : 0), pitch = kmoe::few_row_pitch(values, bytes, scales);
        if (pitch % 16 != 0 || pitch < needed || pitch > needed + 31) return std::printf("%d values of %d bytes: %d", values, bytes, pitch);
      }
  return 0;
}
"""


def test_every_row_starts_on_16_bytes(tmp_path):
    """Lanes read 16 bytes at a time, also in fp8 rows whose scales are no multiple of 16 bytes (lengths that are no multiple of 512)."""
    src, exe = tmp_path / "rows.cc", tmp_path / "rows"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout

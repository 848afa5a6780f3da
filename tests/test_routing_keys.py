"""The sort key of the routing's arg-max (csrc/kmoe_common.h::ordered_bits), compiled for the host: 0 stands for "not a
candidate", so no value may have that key - a NaN of any payload included, which would otherwise leave a token short of
an expert and give the pair the id -1."""
import os
import subprocess

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include <cstdio>
#include <cstring>
#include "kmoe_common.h"
int main() {
  for (unsigned u; scanf("%u", &u) == 1;) {
    float f;
    memcpy(&f, &u, 4);
    printf("%u\\n", kmoe::ordered_bits(f));
  }
}
"""


def _keys(patterns, tmp_path):
    src, exe = tmp_path / "key.hip", tmp_path / "key"
    src.write_text(SOURCE)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-std=c++17",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "vllm-kunlun_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="\n".join(map(str, patterns)), check=True, capture_output=True, text=True)
    return np.array(out.stdout.split(), dtype=np.uint32)


def test_every_candidate_has_a_key_and_numbers_keep_their_order(tmp_path):
    gen = np.random.default_rng(0)
    special = np.array([0xffffffff, 0xfffffffe, 0xffc00000, 0xff800001, 0x7fc00000, 0x7fffffff, 0x7f800001], np.uint32)
    bits = np.concatenate([special, np.array([0, 1 << 31, 0x7f800000, 0xff800000, 1, 0x80000001], np.uint32),
                           gen.integers(0, 1 << 32, 4000, dtype=np.uint64).astype(np.uint32)])
    keys = _keys(bits.tolist(), tmp_path)
    assert keys.shape == bits.shape and (keys != 0).all()
    values = bits.view(np.float32)
    number = ~np.isnan(values)
    v, k = values[number], keys[number].astype(np.int64)
    order = np.argsort(v, kind="stable")
    v, k = v[order].astype(np.float64), k[order]
    assert ((np.diff(v) > 0) == (np.diff(k) > 0)).all() and (np.diff(k) >= 0).all()
    assert keys[0] < k.min()  # below every number

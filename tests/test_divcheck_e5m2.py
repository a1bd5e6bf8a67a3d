"""The e5m2 part of the exhaustive proof (oracle/divcheck.c): the reciprocal + 2-FMA quotient gives the byte of IEEE division
for every bfloat16 pair whose amax has a biased exponent in the range that the kernels use."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_e5m2_quotient_proof_and_kernel_constant():
    subprocess.run(["make", "-C", os.path.join(ROOT, "oracle"), "-s"], check=True)
    out = subprocess.run([os.path.join(ROOT, "oracle", "_build", "divcheck")], check=True, stdout=subprocess.PIPE, text=True).stdout
    lo, hi = map(int, re.search(r"mode 2 clean_amax_exp_range (-?\d+) (-?\d+)", out).groups())
    src = open(os.path.join(ROOT, "mdy_triton_amd", "csrc", "common.h")).read()
    k = int(re.search(r"kFastQuotientMinExpE5m2\s*=\s*(\d+)", src).group(1))
    assert hi == 254 and k == lo, "the kernels' range is the proven one"

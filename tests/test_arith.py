"""The epilogue arithmetic of the matrix-core passes (transformer_amd/csrc/arith.h) against 64 bits, on the
CPU: SwiGLU keeps the accuracy of the library exponential and IEEE divisions, and the division by a
row's rms is the correctly rounded one."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "transformer_amd", "csrc")


def test_swiglu_and_quotient_are_as_accurate_as_f32_allows(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "arith_model")
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe, os.path.join(HERE, "arith_model.cpp")],
                   check=True)
    err, edges = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.splitlines()
    swiglu, quotient, differ = (float(x) for x in err.split()[1::2])
    # one rounding each of 1 + e, its reciprocal and two products, and the exponential's own (2 units)
    assert swiglu <= 4 * 1.0 + 2.0
    assert quotient <= 1.0 and differ == 0
    assert edges.split()[1:] == ["inf", "0", "0", "nan"]


@pytest.mark.parametrize("name", ["prefill.hip", "batched.hip"])
def test_softmax_and_swiglu_take_no_bare_hardware_exponential(name):
    """exp(x) as the hardware's 2^(x log2 e) is off by up to |x| 2^-24: the softmax over scores far apart
    and SwiGLU at large negative gates would lose bits that f32 holds."""
    src = open(os.path.join(CSRC, name)).read()
    for word in ("amdgcn_exp2f", "amdgcn_rcpf", "__expf", "exp2f("):
        assert word not in src, word

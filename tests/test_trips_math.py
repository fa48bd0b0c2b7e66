"""The projection's scalar functions, compiled for the host, over whole ranges of floats: exponential, logarithm, softplus and quotients
have the bits that exp(), log() and the division give."""
import os
import subprocess

import pytest

from trips_amd import build

HOST = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


def _has_fma():
    try:
        with open("/proc/cpuinfo") as f:
            return " fma " in f.read()
    except OSError:
        return False


@pytest.mark.skipif(not _has_fma(), reason="a host without fused multiply-add would take minutes")
def test_scalar_functions_over_all_their_floats(tmp_path):
    prog = tmp_path / "trips_math_host"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-Wno-unknown-pragmas", f"-I{HOST}", f"-I{build.CSRC}",
                           os.path.join(HOST, "trips_math_host.cpp"), "-o", str(prog), "-lpthread"])
    out = subprocess.run([str(prog)], check=True, capture_output=True, text=True).stdout
    got = {w[0]: (int(w[1]), int(w[2]), w[3:]) for w in (line.split() for line in out.splitlines())}
    assert set(got) == {"softplus+", "softplus-", "softplus0", "log", "quotient", "quotient_small", "quotient_middle"}
    # (two floats, neither of them 1 + exp(x) of a float, whose logarithm is next to the middle between two floats)
    assert got.pop("log")[1:] == (2, ["0x4665a9a6", "0x4d604ebe"])
    for name, (values, different, which) in got.items():
        assert values > 10_000_000 and different == 0, (name, different, which)

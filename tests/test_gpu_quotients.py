"""The quotients that share a divisor and the square root of the hydro kernels (physics.hpp ``recip``,
``recip_kb``, ``quot``, ``speed_sqrt``) equal the host's IEEE division and square root bit for bit:
``tests/cpp/quot_check`` runs 2^22 operand pairs of each on the GPU."""

import os
import re
import subprocess

import pytest

pytestmark = pytest.mark.gpu

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "quot_check")


def test_shared_divisor_quotients_are_ieee(cuda):
    assert os.path.exists(BIN), "build it with __graft_entry__.build() (make -C tests/cpp)"
    print("[quotients] running tests/cpp/quot_check", flush=True)
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    for name in ("recip", "recip_kb", "table", "speed_sqrt"):
        m = re.search(rf"^{name}: (\d+) values, (\d+) mismatches", r.stdout, re.M)
        assert m and int(m.group(1)) == 1 << 22 and int(m.group(2)) == 0, r.stdout

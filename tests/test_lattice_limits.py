"""Addresses and sizes on the host: the displacement addresses of lattices past 32
bits, the places of the interface nodes, and the refusal of a lattice that is too
large at creation (before anything is allocated, so no GPU is needed)."""
import ctypes as C
import os
import shutil
import subprocess
import tempfile

import pytest

from hirensi_amd import native

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ absent")
@pytest.mark.parametrize("check", ["index_check", "iface_check", "due_check"])
def test_host_check(check):
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "ic")
        subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(HERE, "native", check + ".cpp"), "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout


def test_lattice_past_the_slots_is_refused():
    L = native.load()
    d = native.MeshDesc()
    d.nex = d.ney = d.nez = 391                    # 783^3 nodes
    for a in range(5):
        d.npml[a] = 4
    for a in range(3):
        d.h[a] = 1.0
    h = C.c_void_p()
    rc = L.hr_ctx_create(C.byref(d), C.byref(h))
    msg = L.hr_last_error(h)
    L.hr_ctx_destroy(h)
    assert rc != 0 and b"too large" in msg, (rc, msg)

"""In the library no launcher is optional: the host code refers to every one of the kernel units with
a strong symbol, so one left out of the link fails it instead of becoming the slow path."""
import os
import shutil
import subprocess

import pytest

from pannde_amd import build


@pytest.mark.skipif(shutil.which("nm") is None or not os.path.exists(build.HIPCC), reason="needs nm and hipcc")
@pytest.mark.timeout(300)
def test_host_code_needs_every_launcher(tmp_path):
    obj = str(tmp_path / "host.o")
    subprocess.run([build.HIPCC] + build.HOST_FLAGS + ["-c", os.path.join(build.CSRC, "rsg_host.cpp"), "-o", obj],
                   check=True, timeout=250)
    names = subprocess.run(["nm", "-C", obj], check=True, stdout=subprocess.PIPE, text=True).stdout.splitlines()
    weak = [n for n in names if " w rsg::" in n]
    strong = {n.split("rsg::")[1].split("(")[0] for n in names if " U rsg::" in n}
    assert not weak
    assert {"resident_limits", "resident_after", "launch_resident_f64", "launch_resident_f32", "launch_state_f64",
            "launch_state_f32", "launch_velocity_f64", "launch_energy_f64"} <= strong
    # a kernel unit left out: the link fails
    r = subprocess.run([build.HIPCC, "-shared", "-fPIC", obj, "-L/opt/rocm/lib", "-lrocprofiler-sdk-roctx",
                        "-Wl,--no-undefined", "-o", str(tmp_path / "lib.so")], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode != 0 and "launch_state_f64" in r.stdout

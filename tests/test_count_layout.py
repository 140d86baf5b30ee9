"""Host code of the counted tables' headers, compiled for the CPU and run:
count_layout_host.cpp checks the column groups of split layouts,
count_keys_host.cpp the keys of agent pairs and their check."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pandemicthrust_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def run_host(source, tmp_path):
    if not (os.path.exists(HIPCC) or shutil.which(HIPCC)):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "host")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-ffp-contract=off", "-Wno-unused-function", "-I", CSRC,
                    os.path.join(HERE, source), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
    return r.stdout


def test_column_groups(tmp_path):
    assert ", 0 wrong" in run_host("count_layout_host.cpp", tmp_path)


def test_pair_keys(tmp_path):
    assert ", 0 wrong" in run_host("count_keys_host.cpp", tmp_path)


def test_contacts_by_workplace_type(tmp_path):
    assert ", 0 wrong" in run_host("workplace_contacts_host.cpp", tmp_path)

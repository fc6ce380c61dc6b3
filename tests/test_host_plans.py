"""Runs the checks of the library's host side (tests/cpp/resident_plan_test.cpp, hex_stage_test.cpp,
chip_share_test.cpp): no GPU."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(name):
    subprocess.check_call(["make", "-s", "-C", os.path.join(ROOT, "oracle")])
    subprocess.check_call(["make", "-s", "-C", os.path.join(ROOT, "tests", "cpp")])
    p = subprocess.run([os.path.join(ROOT, "tests", "cpp", "_build", name)], capture_output=True, text=True, timeout=300)
    sys.stdout.write(p.stdout + p.stderr)
    assert p.returncode == 0, name


def test_resident_plans():
    run("resident_plan_test")


def test_hex_staging_map():
    run("hex_stage_test")


def test_admission_of_solves():
    run("chip_share_test")

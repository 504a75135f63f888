"""Buffer offsets of the wide-row product (honei_amd/csrc/row_slot.hh), checked
on the host by tests/cpp/row_slot_check, built from the header that the device
code includes."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_row_slots():
    r = subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "tests", "cpp")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([os.path.join(ROOT, "tests", "cpp", "_build", "row_slot_check")], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]

"""Every device buffer of the library is allocated by device_alloc, which gives held memory back
and tries again when the device is short of it."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_device_buffers_come_from_device_alloc():
    bare = []
    for path in glob.glob(os.path.join(ROOT, "sparkx_amd", "csrc", "*")):
        with open(path) as fh:
            text = re.sub(r"//[^\n]*", "", fh.read())
        bare += [os.path.basename(path)] * len(re.findall(r"\bhip(?:Ext)?Malloc(?:Async|Managed|WithFlags)?\s*\(", text))
    assert bare == ["hb_exact.hip"] * 2  # the two attempts of device_alloc itself


def test_release_memory_without_a_device():
    import sparkx_amd
    sparkx_amd.release_memory()

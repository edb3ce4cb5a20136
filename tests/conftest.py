import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line(
        "markers", "gpu: needs an MI355X (runs the HIP kernels)")


@pytest.fixture(scope="session")
def gpu():
    """Fails (does not skip) when no device is visible: a GPU test that
    silently skipped would hide a missing native path."""
    from ducc_amd import _lib
    _lib.require_gpu()
    return True


def kernel_rows(ofactor, ndim, single):
    """{W: (index, epsilon)} of the kernel table's rows of an oversampling
    factor"""
    import csv
    path = os.path.join(ROOT, "ducc_amd", "data", "kernel_db.csv")
    rows = [r for r in csv.reader(open(path)) if not r[0].startswith("#")]
    return {int(r[0]): (i, float(r[2])) for i, r in enumerate(rows)
            if float(r[1]) == ofactor and int(r[5]) == ndim
            and int(r[6]) == int(single)}

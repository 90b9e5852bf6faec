import importlib.util
import pathlib
import sys

import numpy as np
import pytest

REPO = pathlib.Path(__file__).resolve().parent.parent
sys.path.insert(0, str(REPO / "op2-common_amd"))
sys.path.insert(0, str(REPO))
GOLDEN = REPO / "tests" / "golden"


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device)")


def golden(name):
    with np.load(GOLDEN / f"{name}.npz", allow_pickle=False) as z:
        return {k: z[k] for k in z.files}


def rel_err(a, b):
    """max |a-b| / max |b| over the arrays (b the reference)."""
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    scale = np.max(np.abs(b))
    return float(np.max(np.abs(a - b)) / scale) if scale > 0 else float(np.max(np.abs(a - b)))


def pointwise_rel_err(a, b):
    """max over entries of |a-b| / |b| (entries with b == 0 use |a-b|)."""
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    d = np.abs(a - b)
    s = np.abs(b)
    return float(np.max(np.where(s > 0, d / np.where(s > 0, s, 1.0), d)))


def _apps():
    spec = importlib.util.spec_from_file_location("apps_build", REPO / "tests" / "apps" / "build.py")
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def reference_program(path):
    """A program that __graft_entry__.build() builds from the reference's own
    sources: the test is skipped only where those are absent too."""
    if not path.exists():
        assert not _apps().reference_present(), f"{path} missing: run __graft_entry__.build()"
        pytest.skip(f"{path} missing, and so are the sources it is built from")
    return path


@pytest.fixture(scope="session")
def gpu_available():
    import ctypes
    try:
        hip = ctypes.CDLL("libamdhip64.so")
        n = ctypes.c_int(0)
        return hip.hipGetDeviceCount(ctypes.byref(n)) == 0 and n.value > 0
    except OSError:
        return False

"""The optimised image formed on the device in pieces, when device memory for
all of it is refused (tests/hip_refuse.c): the same bytes as through the CPU
oracle and the host optimiser.  One child process, since the refusing
hipMalloc has to be loaded before the library."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
KINDS = ["strip8", "grey16", "16to8", "key8", "key16", "pal17", "pal4k"]

pytestmark = pytest.mark.gpu


def test_pieces(tmp_path):
    so = str(tmp_path / "libhip_refuse.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", os.path.join(HERE, "hip_refuse.c"), "-o", so, "-ldl"],
                   check=True)
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), so], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-4000:]


def child(so):
    m = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
    m.refuse.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
    sys.path[:0] = [os.path.dirname(HERE), HERE]
    import cases
    import test_finish_device as dev
    import test_opt_scan as opt
    from conftest import ORACLE_LIB
    from imageworsener_amd import api
    lib = api.Library()
    oracle = ctypes.CDLL(ORACLE_LIB, mode=os.RTLD_LOCAL | os.RTLD_NOW)
    oracle.iwo_run.argtypes = [ctypes.c_void_p, ctypes.c_void_p]

    def executor(plan, img2):
        return bool(oracle.iwo_run(ctypes.addressof(plan), ctypes.addressof(img2)))

    big = api.image_job(np.zeros((1500, 1500, 3), np.uint8), 1500, 1500, cases.RGB, 8, canvas=(1500, 1500),
                        resize=api.resize_both("catrom"))
    for kind in KINDS:
        rng = np.random.default_rng(len(kind))
        a, imgtype, depth, more = dev._image(kind, rng, 301, 307)
        job = opt.job_of(a, imgtype, depth, **more)
        want = lib.run(job, executor=executor)
        for lo in (40000, 4700):
            print(kind, lo, flush=True)
            j = lib.device_job(job)
            j.run()
            # A request that cannot be met gives the library's cached blocks back.
            m.refuse(lo, 1 << 40)
            with pytest.raises(RuntimeError, match="Out of device memory"):
                lib.device_job(big)
            before = m.refusals()
            got = j.finish()
            m.refuse(1, 0)
            cases.assert_same(want, got, kind)
            assert m.refusals() > before, kind


if __name__ == "__main__":
    child(sys.argv[1])

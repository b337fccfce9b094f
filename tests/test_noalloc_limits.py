"""iwamd_process_device_noalloc at the limit of its scratch array: jobs whose
horizontal lists fit it only laid out by output (without room for the most
taps in every output), in the fused kernel and in two passes, give the bytes
of iw_process_image."""
import numpy as np
import pytest

import cases
from imageworsener_amd import api, synth

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")  # before the library, so that both use torch's HIP runtime
import test_zz_no_alloc as zz

JOBS = {  # name: size, output size, horizontal blur, kind
    "fused": (2000, 24, 3700, 30, 500.0, None),
    "fused-late-bkgd": (2000, 24, 3700, 30, 500.0, "bkgd"),
    "twopass": (2900, 24, 1790, 30, 660.0, None),
    "twopass-diffused": (3000, 40, 1003, 800, 500.0, "f"),
}


def make(name):
    w, h, ow, oh, blur, kind = JOBS[name]
    rgba = kind == "bkgd"
    img = synth.c3_image(w, h, 5)
    resize = {0: api.resize_both("triangle", blur)[0], 1: api.resize_both("catrom")[1]}
    job = api.image_job(img if rgba else np.ascontiguousarray(img[..., :3]), w, h, cases.RGBA if rgba else cases.RGB, 8,
                        canvas=(ow, oh), resize=resize, values=[(cases.V_CVT_GRAY, 1)])
    if kind == "f":
        job["dither"] = [(api.CH_ALL, 2, 0)]
    if rgba:
        job["bkgd"] = (0.2, 0.5, 0.9, 1.0)
    return job


@pytest.mark.parametrize("name", sorted(JOBS))
def test_lists_by_output(prod, oracle_exec, name):
    job = make(name)
    zz._check(prod, name, job)
    plain = dict(job, allow_opt=zz.NO_OPT)
    cases.assert_same(prod.run(plain, executor=oracle_exec), prod.run(plain))

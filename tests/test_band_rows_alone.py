"""A job alone in bands of fewer rows (band_rows_alone): heights around the
limits where a band loses rows (512, 1024, 2048), against the same job with
its band height fixed; floats that are not finite keep the bytes of the
tallest band."""
import numpy as np
import pytest

import cases
from imageworsener_amd import api, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("height", [1, 3, 511, 512, 513, 1021, 1024, 1025, 2044, 2045, 2049])
@pytest.mark.parametrize("imgtype", ["GRAY", "RGBA"])
def test_heights(prod, oracle_exec, height, imgtype):
    nch = api.NCH[api.IMGTYPE[imgtype]]
    img = synth.c3_image(31, 700, 3)[..., 4 - nch:].copy()
    job = api.image_job(img, 31, 700, api.IMGTYPE[imgtype], 8, canvas=(17, height), resize=api.resize_both("catrom"))
    got = prod.run(job)
    cases.assert_same(prod.run(job, executor=oracle_exec), got)
    for rows in ("1", "4"):
        cases.assert_same(prod.run(dict(job, options=[("amd:band_rows", rows)])), got)


@pytest.mark.parametrize("height", [5, 100, 601, 1300])
def test_not_finite(prod, height):
    a = np.random.default_rng(2).random((300, 40, 3), dtype=np.float32)
    a[::37, ::11] = np.inf
    a[5::53, 3::13] = np.nan
    job = {"image": {"pixels": a.view(np.uint8).reshape(-1), "width": 40, "height": 300, "imgtype": cases.RGB,
                     "bit_depth": 32, "bpr": 480, "sampletype": 1},
           "canvas": (23, height), "input_cs": (1, 0.0), "output_cs": (1, 0.0), "resize": api.resize_both("catrom"),
           "profile": api.PROFILE_PNG | 0x4000}
    cases.assert_same(prod.run(dict(job, options=[("amd:band_rows", "4")])), prod.run(job))

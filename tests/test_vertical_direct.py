"""The vertical pass with the input read in place (band_vertical): every
sample width and channel count with its own loop and the general one, band
heights of 1, 2 and 4 rows and the two-pass form, tables in LDS and (rows too
wide for them) in memory, transparent edges, an early background, and
downscales and upscales with rows that do not fill a band.  Byte for byte
against the CPU oracle on the same plan."""
import numpy as np
import pytest

import cases
from imageworsener_amd import api, synth

pytestmark = pytest.mark.gpu

LINEAR = {"input_cs": (1, 0.0), "output_cs": (1, 0.0)}
KINDS = {
    "plain": {},
    "linear": LINEAR,
    "edges": {"values": [(17, 3), (18, 1)]},
    "bkgd": {"bkgd": (0.2, 0.5, 0.9, 1.0)},
}
FORMS = {"r1": [("amd:resample", "band"), ("amd:band_rows", "1")], "r2": [("amd:resample", "band"), ("amd:band_rows", "2")],
         "r4": [("amd:resample", "band"), ("amd:band_rows", "4")], "two": [("amd:resample", "twopass")]}


def _job(rng, w, h, imgtype, depth, canvas, opts, **more):
    nch = api.NCH[api.IMGTYPE[imgtype]]
    if depth == 32:
        a = rng.random((h, w, nch), dtype=np.float32)
        job = {"image": {"pixels": a.view(np.uint8).reshape(-1), "width": w, "height": h,
                         "imgtype": api.IMGTYPE[imgtype], "bit_depth": 32, "bpr": w * nch * 4, "sampletype": 1},
               "canvas": canvas, "resize": api.resize_both("catrom"), "profile": api.PROFILE_PNG | 0x4000}
    else:
        a = rng.integers(0, 1 << depth, (h, w, nch)).astype(np.uint16)
        a = synth.be16(a) if depth == 16 else a.astype(np.uint8)
        job = api.image_job(a, w, h, api.IMGTYPE[imgtype], depth, canvas=canvas, resize=api.resize_both("lanczos3"))
    job.update(more, options=opts)
    return job


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("imgtype", ["GRAY", "GRAYA", "RGB", "RGBA"])
@pytest.mark.parametrize("depth", [8, 16, 32])
def test_samples(prod, oracle_exec, depth, imgtype, kind, form):
    rng = np.random.default_rng(depth)
    for w, h, canvas in ((70, 61, (33, 15)), (5, 3, (40, 22)), (300, 1, (7, 1))):
        more = dict(LINEAR if depth == 32 else {}, **KINDS[kind])
        job = _job(rng, w, h, imgtype, depth, canvas, FORMS[form], **more)
        cases.assert_same(prod.run(job, executor=oracle_exec), prod.run(job))


@pytest.mark.parametrize("width", [9850, 9858, 10000, 10112])
def test_tables_past_lds(prod, oracle_exec, width):
    job = _job(np.random.default_rng(1), width, 6, "RGBA", 8, (50, 3), FORMS["r1"])
    cases.assert_same(prod.run(job, executor=oracle_exec), prod.run(job))

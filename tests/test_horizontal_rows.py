"""The horizontal pass with several rows per thread (hrows), in the fused and
the two-pass form: output widths around the splits of a band's columns over
its threads, rows that do not fill the last group, one to four channels, the
generic per-pixel work (ordered dither, checkered background, floating-point
output), transparent edges and lists that differ by channel.  Byte for byte
against the CPU oracle on the same plan."""
import numpy as np
import pytest

import cases
from imageworsener_amd import api, synth

pytestmark = pytest.mark.gpu

KINDS = {
    "plain": {},
    "ordered": {"dither": [(api.CH_ALL,) + api.DITHER["o"]]},
    "edges": {"values": [(17, 3), (18, 1)]},
    "offsets": {"values_dbl": [(42, 2.5), (43, -1.25)]},
}


@pytest.mark.parametrize("path", ["band", "twopass"])
@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("imgtype", ["GRAY", "RGB", "RGBA"])
@pytest.mark.parametrize("size", [(1, 1), (63, 5), (64, 6), (65, 7), (129, 9), (257, 4), (321, 3)])
def test_rows(prod, oracle_exec, size, imgtype, kind, path):
    nch = api.NCH[api.IMGTYPE[imgtype]]
    img = synth.c3_image(97, 23, 7)[..., 4 - nch:].copy()
    job = api.image_job(img, 97, 23, api.IMGTYPE[imgtype], 8, canvas=size, resize=api.resize_both("lanczos3"),
                        options=[("amd:resample", path)], **KINDS[kind])
    cases.assert_same(prod.run(job, executor=oracle_exec), prod.run(job))


@pytest.mark.parametrize("path", ["band", "twopass"])
@pytest.mark.parametrize("nch,imgtype", [(1, "GRAY"), (3, "RGB"), (4, "RGBA")])
@pytest.mark.parametrize("width", [40, 200])
def test_float(prod, oracle_exec, width, nch, imgtype, path):
    a = np.random.default_rng(5).random((31, 77, nch), dtype=np.float32) * 2 - np.float32(0.5)
    job = {"image": {"pixels": np.ascontiguousarray(a).view(np.uint8).reshape(-1), "width": 77, "height": 31,
                     "imgtype": api.IMGTYPE[imgtype], "bit_depth": 32, "bpr": 77 * nch * 4, "sampletype": 1},
           "canvas": (width, 13), "input_cs": (1, 0.0), "output_cs": (1, 0.0), "resize": api.resize_both("catrom"),
           "profile": api.PROFILE_PNG | 0x4000, "options": [("amd:resample", path)]}
    cases.assert_same(prod.run(job, executor=oracle_exec), prod.run(job))

"""Single jobs in the shapes of shape_alone: heights at the ends of its rounds
(1024 bands of 1 row, 768 of 2, 512 and 1024 of 4), widths on both sides of a
batch's kernel (256 and 512 columns), every kind of per-pixel work, against the
CPU oracle."""
import numpy as np
import pytest

import cases
from imageworsener_amd import api, synth

pytestmark = pytest.mark.gpu

KINDS = {
    "plain": (cases.RGB, {}),
    "rgba": (cases.RGBA, {}),
    "bkgd": (cases.RGBA, {"bkgd": (0.2, 0.5, 0.9, 1.0)}),
    "ordered": (cases.RGB, {"dither": [(api.CH_ALL,) + api.DITHER["o"]]}),
    "diffused": (cases.RGB, {"dither": [(api.CH_ALL,) + api.DITHER["f"]]}),
    "deep": (cases.RGBA, {"depth": 16}),
    "edges": (cases.RGB, {"values": [(cases.V_EDGE_X, 3), (cases.V_EDGE_Y, 1)],
                          "values_dbl": [(cases.V_TRANSLATE_X, 2.5), (cases.V_TRANSLATE_Y, -1.25)]}),
    "nearest": (cases.RGB, {"resize": api.resize_both("nearest")}),
}


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("size", [(33, 29, 1024), (33, 29, 1025), (33, 29, 1537), (33, 29, 2051), (20, 257, 1540),
                                  (300, 255, 2049), (255, 300, 2050), (511, 150, 4099)])
def test_sizes(prod, oracle_exec, kind, size):
    w, ow, oh = size
    imgtype, more = KINDS[kind]
    img = synth.c3_image(w, 90, 7)
    if imgtype == cases.RGB:
        img = np.ascontiguousarray(img[..., :3])
    job = dict(api.image_job(img, w, 90, imgtype, 8, canvas=(ow, oh), resize=api.resize_both("catrom")), **more)
    cases.assert_same(prod.run(job, executor=oracle_exec), prod.run(job), "%s %s" % (kind, size))

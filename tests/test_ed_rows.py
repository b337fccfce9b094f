"""Error diffusion with the rows in registers (errdiff_rows_kernel): rows of 1
to 4096 pixels, at the edges of its segments, waves and row shapes, and one
pixel past the widest (errdiff_kernel), byte for byte against the CPU oracle
on the same plan.  Every matrix reach (one pixel and row, x+2, two rows),
level counts from 2 to 256, 8- and 16-bit codes, one to four planes, and
images of exact samples (white, black and mid-grey areas)."""
import numpy as np
import pytest

import cases
from imageworsener_amd import api, synth

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 3, 4, 5, 8, 63, 255, 256, 257, 511, 513, 1024, 1025, 2048, 2049, 4095, 4096, 4097]


def _grey(width, dither, colors, **more):
    img = synth.be16(synth.c2(96)[:24])
    job = api.image_job(img, 96, 24, cases.GRAY, 16, canvas=(width, 13), resize=api.resize_both("catrom"),
                        dither=[(api.CH_ALL,) + api.DITHER[dither]], **more)
    if colors:
        job["color_count"] = [(api.CH_ALL, colors)]
    return job


def _same(prod, oracle_exec, job):
    cases.assert_same(prod.run(job, executor=oracle_exec), prod.run(job))


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("dither,colors", [("f", 0), ("jjn", 4), ("atkinson", 5)])
def test_row_shapes(prod, oracle_exec, width, dither, colors):
    _same(prod, oracle_exec, _grey(width, dither, colors))


@pytest.mark.parametrize("colors", [2, 3, 16, 256])
@pytest.mark.parametrize("dither", ["sierralite", "burkes", "sierra"])
def test_levels(prod, oracle_exec, dither, colors):
    _same(prod, oracle_exec, _grey(777, dither, colors, depth=16 if colors == 16 else 8))


@pytest.mark.parametrize("imgtype", ["GRAYA", "RGB", "RGBA"])
@pytest.mark.parametrize("width", [31, 515, 1500])
def test_planes(prod, oracle_exec, imgtype, width):
    nch = api.NCH[api.IMGTYPE[imgtype]]
    img = synth.c3_image(120, 40, 5)[..., 4 - nch:].copy()
    job = api.image_job(img, 120, 40, api.IMGTYPE[imgtype], 8, canvas=(width, 21), resize=api.resize_both("mitchell"),
                        dither=[(api.CH_ALL, 2, 0)])
    _same(prod, oracle_exec, job)


@pytest.mark.parametrize("width", [40, 600, 1500])
def test_exact_samples(prod, oracle_exec, width):
    img = np.full((64, 80, 3), 255, np.uint8)
    img[20:40, 30:50] = 0
    img[10:15] = 128
    job = api.image_job(img, 80, 64, cases.RGB, 8, canvas=(width, 50), resize=api.resize_both("lanczos3"),
                        dither=[(api.CH_ALL, 2, 0)])
    _same(prod, oracle_exec, job)

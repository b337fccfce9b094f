"""The codes of error-diffused channels into their pixels (edr_interleave4):
images of which only some channels are diffused, 16-bit codes of channels that
differ, and widths that are no multiple of four, as single jobs, in a batch
and as served requests (whose last plane forms the output), all byte for byte
against the CPU oracle."""
import numpy as np
import pytest

import cases
from imageworsener_amd import api, synth

pytestmark = pytest.mark.gpu

RED, GREEN, BLUE, ALPHA = 0, 1, 2, api.CH_ALPHA  # IW_CHANNELTYPE_*
FS, JJN, ORDERED = api.DITHER["f"], api.DITHER["jjn"], api.DITHER["o"]


def _jobs():
    rgba = synth.c3_image(90, 40, 11)
    rgb = np.ascontiguousarray(rgba[..., :3])
    for width in (1, 5, 63, 257, 1026, 2051, 4099):
        for depth in (8, 16):
            for name, img, dither in [
                ("red", rgb, [(RED,) + FS]),
                ("green-blue", rgb, [(GREEN,) + FS, (BLUE,) + JJN]),
                ("all", rgb, [(api.CH_ALL,) + FS]),
                ("mixed", rgba, [(RED,) + FS, (GREEN,) + ORDERED, (ALPHA,) + JJN]),
                ("four", rgba, [(api.CH_ALL,) + JJN]),
            ]:
                job = api.image_job(img, 90, 40, cases.RGB if img is rgb else cases.RGBA, 8, canvas=(width, 19),
                                    resize=api.resize_both("catrom"), dither=dither, depth=depth)
                if depth == 16:
                    # At most 257 levels: rows in registers.
                    job["color_count"] = [(RED, 40), (GREEN, 200), (BLUE, 7), (ALPHA, 100)]
                yield "%s-%d-%d" % (name, width, depth), job


JOBS = list(_jobs())


@pytest.mark.parametrize("name,job", JOBS, ids=[n for n, _ in JOBS])
def test_alone(prod, oracle_exec, name, job):
    cases.assert_same(prod.run(job, executor=oracle_exec), prod.run(job), name)


def test_batch_and_served(prod, oracle_exec):
    want = [prod.run(j, executor=oracle_exec) for _, j in JOBS]
    for (name, _), a, b in zip(JOBS, want, prod.run_batch([j for _, j in JOBS])):
        cases.assert_same(a, b, "batch " + name)
    s = api.Server(prod, streams=2)
    for _, j in JOBS:
        s.submit(j)
    s.drain()
    for (name, _), a, b in zip(JOBS, want, s.results()):
        cases.assert_same(a, b, "served " + name)
    s.close()

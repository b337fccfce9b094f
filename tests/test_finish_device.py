"""The optimised image formed on the device (conv_kernel): every conversion
the optimiser makes, on outputs just below and above the size from which a
single job's image is formed there and at pixel counts that are no multiple
of a thread's four, against the same job through the CPU oracle and the host
optimiser."""
import numpy as np
import pytest

import cases
import test_opt_scan as opt
from imageworsener_amd import api

pytestmark = pytest.mark.gpu

RGB, RGBA, GRAY, GRAYA = cases.RGB, cases.RGBA, cases.GRAY, cases.GRAYA
LINE = 128 << 10  # bytes


def _image(kind, rng, h, w):
    """(samples, image type, depth, settings)"""
    full = lambda hi, n: rng.integers(0, hi, (h, w, n))
    binary = lambda hi: opt.binary_alpha(rng, h, w, hi)[..., None]
    if kind == "strip8":
        return np.concatenate([full(256, 3), np.full((h, w, 1), 255)], 2), RGBA, 8, {}
    if kind == "grey8":
        return np.repeat(full(256, 1), 3, 2), RGB, 8, {"profile": api.PROFILE_PAM}
    if kind == "grey16":
        return np.repeat(full(65536, 1), 3, 2), RGB, 16, {}
    if kind == "greya8":
        return np.concatenate([np.repeat(full(256, 1), 3, 2), full(256, 1)], 2), RGBA, 8, {}
    if kind == "16to8":
        return full(256, 4) * 257, RGBA, 16, {}
    if kind == "keep16":
        return full(65536, 4), RGBA, 16, {}
    if kind == "key8":
        return opt.rgba8_keys(rng, h, w, np.array([192, 193])), RGBA, 8, {}
    if kind == "key16":
        return opt.rgba16_keys(rng, h, w, np.array([192, 7])), RGBA, 16, {}
    if kind == "keygrey16":
        return np.concatenate([full(65536, 1), binary(65535)], 2), GRAYA, 16, {}
    n = int(kind[3:].rstrip("gk"))
    at = rng.integers(0, n, (h, w))
    if kind.endswith("k"):  # grey levels with a colour key
        return np.concatenate([(at * (255 // (n - 1)))[..., None], binary(255)], 2), GRAYA, 8, {}
    if kind.endswith("g"):
        return (at * (255 // (n - 1)))[..., None], GRAY, 8, {}
    return rng.integers(0, 256, (n, 4))[at], RGBA, 8, {}


@pytest.mark.parametrize("kind", ["strip8", "grey8", "grey16", "greya8", "16to8", "keep16", "key8", "key16", "keygrey16",
                                  "pal1", "pal2", "pal17", "pal256", "pal257", "pal2g", "pal4g", "pal4k", "pal16k"])
@pytest.mark.parametrize("extra", [-1, 1, 77])
def test_conversions(prod, oracle_exec, kind, extra):
    rng = np.random.default_rng(len(kind) * 100 + extra + 1)
    probe, _, depth, _ = _image(kind, rng, 8, 8)
    nch = probe.shape[2]
    w = 211
    h = max(1, round(LINE / (w * nch * depth // 8))) + extra
    a, imgtype, depth, more = _image(kind, rng, h, w)
    job = opt.job_of(a, imgtype, depth, **more)
    cases.assert_same(prod.run(job, executor=oracle_exec), prod.run(job))

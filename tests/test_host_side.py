"""The library's host side without a GPU: decisions, work lists, pools and error
paths, on a HIP runtime of host memory whose kernels do nothing
(tests/hip_mock.c).  Each test runs in a process of its own, since the mock
takes the place of the HIP runtime in it."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="session")
def mock_so(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("mock") / "libhip_mock.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", os.path.join(HERE, "hip_mock.c"), "-o", so, "-lpthread"],
                   check=True)
    return so


@pytest.fixture
def scenario(mock_so):
    def run(name, *args):
        r = subprocess.run([sys.executable, os.path.abspath(__file__), mock_so, name] + [str(a) for a in args],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
        assert r.returncode == 0, r.stdout[-4000:]
    return run


# ---- scenarios (run in the child) -----------------------------------------------

class Mock:
    """The mock runtime, loaded for the whole process, and the library on it."""

    def __init__(self, so):
        self.m = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
        self.m.mock_launch.restype = ctypes.c_char_p
        self.m.mock_launch_items.restype = ctypes.c_void_p
        self.m.mock_fail_malloc.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
        sys.path[:0] = [os.path.dirname(HERE), HERE]
        from imageworsener_amd import api
        self.lib = api.Library()

    def launches(self, part=""):
        """(index, name, grid) of the launches so far whose kernel has part in its name."""
        out = []
        g = (ctypes.c_uint * 3)()
        for i in range(self.m.mock_launches()):
            name = self.m.mock_launch(i, g).decode()
            if part in name:
                out.append((i, name, tuple(g)))
        return out


def s_batch_bands(M):
    """A batch of plans with simple and with generic per-pixel work, more of
    each than one band height and LDS class takes: every band kernel gets a
    work list of its own, of rows that its plans have, and every row of every
    fused plan is in one list."""
    import cases
    from imageworsener_amd import api, synth
    jobs = [dict(j, options=[("amd:band_rows", str(r))]) for _, j in cases.sweep_jobs() for r in (1, 2, 4)]
    big = synth.c3_image(900, 60, 3)
    for w in (20, 200, 900):
        for bkgd in (False, True):
            j = api.image_job(np.ascontiguousarray(big[:, :w]), w, 60, cases.RGBA, 8, canvas=(w, 77),
                              resize=api.resize_both("catrom"), options=[("amd:band_rows", "4")])
            jobs.append(dict(j, bkgd=(0.2, 0.5, 0.9, 0.5)) if bkgd else j)
    os.environ["IWAMD_TUNE"] = "0"
    M.m.mock_clear_log()
    b = M.lib.batch(jobs)
    seen, kinds = {}, set()
    for i, name, grid in M.launches("11band_kernel"):
        rows = int(name.split("band_kernelILi")[1][0])
        kinds.add((rows, name.split("BandKindE")[1][0]))
        n, p = M.m.mock_launch_count(i), M.m.mock_launch_items(i)
        assert p and n >= grid[0] > 0, (name, n, p)
        items = np.ctypeslib.as_array((ctypes.c_int * (2 * n)).from_address(p)).reshape(n, 2)
        for plan, row in items:
            assert 0 <= plan < len(jobs) and row % rows == 0, (name, plan, row)
            assert (plan, row) not in seen
            seen[plan, row] = rows
    assert kinds == {(r, k) for r in (1, 2, 4) for k in "12"}, kinds
    for k, j in enumerate(jobs):
        got = sorted(r for p, r in seen if p == k)
        if got:
            assert got == list(range(0, j["canvas"][1], seen[k, 0])), (k, got)
    assert len({p for p, _ in seen}) > len(jobs) // 2
    b.close()


def test_batch_bands(scenario):
    scenario("s_batch_bands")


def s_tune_alone(M):
    """amd:tune = 1 times a single job's own band kernels, one launch each, and
    the job runs the shape that was fastest; later single jobs of its class
    take it too, batches do not."""
    import cases
    from imageworsener_amd import api
    fastest = [4]

    def ms(nlog):
        _, name, _ = M.launches("11band_kernel")[-1]
        return 1.0 if "band_kernelILi%d" % fastest[0] in name else 2.0
    cb = ctypes.CFUNCTYPE(ctypes.c_double, ctypes.c_int)(ms)

    def bands(job):
        M.m.mock_clear_log()
        j = M.lib.device_job(job)
        timed = len(M.launches("11band_kernel"))
        j.run()
        j.sync()
        last = M.launches("11band_kernel")
        assert len(last) == timed + 1 and all("BandKindE0" in n for _, n, _ in last)
        j.close()
        return int(last[-1][1].split("band_kernelILi")[1][0]), last[-1][2][0], timed

    job = cases.c0_job()
    assert bands(job) == (1, 240, 0)  # shape_alone's
    M.m.mock_event_ms(cb)
    tuned = dict(job, options=[("amd:tune", "1")])
    for f in (4, 2):
        fastest[0] = f
        rows, grid, timed = bands(dict(tuned, resize=api.resize_both({4: "lanczos3", 2: "triangle"}[f])))
        assert (rows, grid) == (f, 240 // f) and timed == 3 * 4, (f, rows, grid, timed)
    assert bands(job) == (4, 60, 0)
    M.m.mock_clear_log()
    b = M.lib.batch([job])
    assert len(M.launches("11band_kernel")) > 1 and all("BandKindE1" in n for _, n, _ in M.launches("11band_kernel"))
    b.close()
    e = [t for t in M.lib.tune_entries() if t["form"] == "band"]
    assert len(e) == 3 and all(t["candidates"][t["shape"]] == min(t["candidates"].values()) for t in e)


def test_tune_alone(scenario):
    scenario("s_tune_alone")


def _noalloc(M, job):
    """(accepted, error) of iwamd_process_device_noalloc for a job."""
    d = M.lib.dll
    fn = d.iwamd_process_device_noalloc
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, ctypes.c_size_t,
                   ctypes.c_void_p, ctypes.c_void_p]
    ctx = d.iw_create_context(None)
    M.lib._setup(ctx, job)
    size = job["image"]["bpr"] * job["image"]["height"] + job["canvas"][0] * job["canvas"][1] * 8
    a, b = ctypes.create_string_buffer(size), ctypes.create_string_buffer(size)
    ok = fn(ctx, a, size, b, size, None, None)
    buf = ctypes.create_string_buffer(300)
    err = d.iw_get_errormsg(ctx, buf, 300).decode()
    d.iw_destroy_context(ctx)
    return bool(ok), err


def s_noalloc_lists(M):
    """The fixed scratch array's limit.  Blurs so wide that outputs at the
    image's sides have half the taps of those in its middle: the lists fit only
    without room for the most taps in every output.  And narrow rows by the
    thousand, diffused: they fit without a list of them."""
    import cases
    from imageworsener_amd import api
    for w, h, ow, oh, fits in [(3000, 40, 999, 800, True), (1000, 1000, 2900, 480, True), (3000, 40, 1500, 800, False),
                              (40, 2520, 1, 3686, True), (40, 2520, 1, 3690, False)]:
        job = api.image_job(np.zeros((h, w, 3), np.uint8), w, h, cases.RGB, 8, canvas=(ow, oh),
                            resize=api.resize_both("triangle", 500.0), values=[(cases.V_CVT_GRAY, 1)],
                            dither=[(api.CH_ALL, 2, 0)])
        ok, err = _noalloc(M, job)
        assert ok == fits, (w, h, ow, oh, err)


def test_noalloc_lists(scenario):
    scenario("s_noalloc_lists")


def s_failed_stream(M):
    """A job's stream and events go to the next job, but not those of a job
    whose last wait failed."""
    import cases
    job = cases.c0_job()

    def one(errors):
        j = M.lib.device_job(job)
        j.run()
        M.m.mock_sync_errors(errors)
        j.close()
        M.m.mock_sync_errors(0)
        return M.m.mock_streams_made(), M.m.mock_streams_freed()

    assert one(0) == (1, 0)
    assert one(0) == (1, 0)
    assert one(1) == (1, 1)
    assert one(0) == (2, 1)
    assert one(0) == (2, 1)


def test_failed_stream(scenario):
    scenario("s_failed_stream")


def s_finish_memory(M, limit):
    """An output whose optimised form finds no device memory is formed in
    pieces, down to the size of the scan's block, and comes back whole.  (The
    mock's scan sees no colour: RGB becomes grey, 320 x 240 bytes.)"""
    import cases
    limit = int(limit)
    j = M.lib.device_job(cases.c0_job())
    j.run()
    M.m.mock_fail_malloc(limit, 1 << 40)
    r = j.finish()
    assert r["ok"], r["error"]
    assert (r["width"], r["height"], r["bpr"], r["imgtype"]) == (320, 240, 320, cases.GRAY)
    grids = [g[0] for _, _, g in M.launches("conv_kernel")]  # 1024 pixels a workgroup
    if limit > 76800:
        assert grids == [75]
    else:
        assert len(grids) > 1 and sum(grids) >= 75 and max(grids) * 1024 <= max(limit, 8192) + 1023, grids


@pytest.mark.parametrize("limit", [76801, 76800, 20000, 4700])
def test_finish_memory(scenario, limit):
    scenario("s_finish_memory", limit)


def s_odd_curves(M, gamma, rows):
    """Output curves given by hand (iw_make_gamma_csdescr keeps its gammas to
    0.1..10): rows go to errdiff_rows_kernel only where level 0 is at 0 and the
    levels ascend to 1."""
    import cases
    from imageworsener_amd import api
    job = api.image_job(np.zeros((20, 30, 3), np.uint8), 30, 20, cases.RGB, 8, canvas=(40, 30),
                        resize=api.resize_both("catrom"), dither=[(api.CH_ALL, 2, 0)],
                        output_cs=(api.CS["gamma"], float(gamma)))
    j = M.lib.device_job(job)
    j.run()
    got = {n for _, n, _ in M.launches("errdiff")}
    assert len(got) == 1 and ("errdiff_rows" in got.pop()) == (rows == "1")
    j.close()


@pytest.mark.parametrize("gamma,rows", [(2.2, 1), (0.1, 1), (10.0, 1), (0.01, 1), (0.0, 0), (-1.0, 0), ("inf", 1),
                                        ("nan", 0)])
def test_odd_curves(scenario, gamma, rows):
    scenario("s_odd_curves", gamma, rows)


def s_alone_shapes(M):
    """The bands of single jobs (shape_alone): rounds of what 256 CUs hold at
    once, and a batch's kernel for narrow images with many rows."""
    import cases
    from imageworsener_amd import api
    for w, ow, oh, kind, want in [
            (40, 30, 24, None, (1, "0")), (40, 30, 1024, None, (1, "0")), (40, 30, 1025, None, (2, "0")),
            (40, 30, 1536, None, (2, "0")), (40, 30, 1537, None, (4, "1")), (40, 30, 2048, None, (4, "1")),
            (40, 30, 2049, None, (4, "1")), (40, 30, 2049, "o", (4, "2")), (40, 30, 2049, "float", (2, "0")),
            (300, 400, 1700, None, (4, "0")), (300, 400, 2049, None, (4, "1")), (300, 600, 2049, None, (2, "0")),
            (2000, 1500, 3000, None, (1, "0")), (2000, 1500, 1000, None, (1, "0"))]:
        img = np.zeros(w * 20 * 3 * (4 if kind == "float" else 1), np.uint8)
        job = api.image_job(img, w, 20, cases.RGB, 32 if kind == "float" else 8, canvas=(ow, oh),
                            resize=api.resize_both("catrom"))
        if kind == "float":
            job["image"]["sampletype"] = 1
            job["input_cs"] = (api.CS["linear"], 0.0)
        if kind == "o":
            job["dither"] = [(api.CH_ALL,) + api.DITHER["o"]]
        M.m.mock_clear_log()
        j = M.lib.device_job(job)
        j.run()
        (i, name, grid), = M.launches("11band_kernel")
        got = int(name.split("band_kernelILi")[1][0]), name.split("BandKindE")[1][0]
        assert got == want and grid[0] == -(-oh // got[0]), (w, ow, oh, kind, got, grid)
        n, p = M.m.mock_launch_count(i), M.m.mock_launch_items(i)
        items = np.ctypeslib.as_array((ctypes.c_int * (2 * n)).from_address(p)).reshape(n, 2)
        assert n == grid[0] and items.tolist() == [[0, k * got[0]] for k in range(n)]
        j.close()


def test_alone_shapes(scenario):
    scenario("s_alone_shapes")


def s_hpass_rows(M):
    """The two-pass form's horizontal pass: a row per thread while that gives at
    most six workgroups a CU, then two."""
    import cases
    from imageworsener_amd import api
    for ow, oh, rows in [(256, 1, 1), (256, 1536, 1), (256, 1537, 2), (257, 768, 1), (257, 769, 2), (4000, 100, 2)]:
        job = api.image_job(np.zeros((20, 30, 3), np.uint8), 30, 20, cases.RGB, 8, canvas=(ow, oh),
                            resize=api.resize_both("catrom"), options=[("amd:resample", "twopass")])
        M.m.mock_clear_log()
        j = M.lib.device_job(job)
        j.run()
        (_, name, grid), = M.launches("hpass")
        assert "hpass_rows_kernelILi%dE" % rows in name and grid[:2] == (-(-ow // 256), -(-oh // rows)), (ow, oh, name, grid)
        j.close()


def test_hpass_rows(scenario):
    scenario("s_hpass_rows")


if __name__ == "__main__":
    globals()[sys.argv[2]](Mock(sys.argv[1]), *sys.argv[3:])

"""Which kernels a call runs, as reported without a device: the plan mirror
(backend.gemm_route, required_resources) against the library (vt_gemm_route),
and the routes of sizes on either side of each rule."""
import math
import random

import pytest

from veritac_amd import _lib
from veritac_amd.specializations.hip_gemm import backend as hg

ROW_MAJOR = ("generic", "padded", "mfma_128x128", "mfma_256x128", "mfma_256x256", "skinny")


def native_route(m, n, k, variant="auto", batch=1, shared=False, **kw):
    multi = batch > 1
    return _lib.gemm_route(m, n, k, k, n, n, n, batch, m * k if multi else 0,
                           0 if shared or not multi else k * n, m * n if multi else 0,
                           m * n if multi else 0, variant=variant, **kw)


def drawn(rng, variant):
    def size(hi):
        return int(round(math.exp(rng.uniform(math.log(8), math.log(hi)))))
    while True:
        m, n, k = size(9000), size(17000), size(17000)
        if variant not in ("generic", "padded") or rng.random() < 0.3:
            n, k = max(16, n // 16 * 16), max(16, k // 16 * 16)
        if variant == "skinny":
            m = min(m, 64)
        batch = 1 if rng.random() < 0.6 else rng.randint(2, 40)
        shared = rng.random() < 0.5
        if m * n * batch < 2**30 and k * 16384 < 2**31:
            return m, n, k, batch, shared


@pytest.mark.parametrize("variant", ROW_MAJOR)
def test_the_plan_mirror_names_the_library_s_routes(variant):
    rng = random.Random(3)
    seen = set()
    for _ in range(500):
        m, n, k, batch, shared = drawn(rng, variant)
        plan = hg.make_plan(m, n, k, batch=batch, b_shared=shared, variant=variant)
        assert hg.validate_plan(plan)[0], plan
        for limit in (2**63 - 1, 1 << 22, 0):
            route, ks, scratch = hg.gemm_route(plan, limit)
            want = native_route(m, n, k, variant, batch, shared, scratch_limit=limit)
            seen.add(route)
            if route in ("valu", "copies", "variant"):
                assert want[0] == route, (plan, limit, want)
            else:
                assert want == (route, ks, scratch), (plan, limit)
    want = {"generic": {"valu", "skinny", "tiles_64", "tiles_128", "persistent"},
            "padded": {"copies", "skinny", "tiles_64", "tiles_128", "persistent"},
            "mfma_128x128": {"variant", "tiles_64", "tiles_128", "persistent"},
            "mfma_256x128": {"variant", "persistent"}, "mfma_256x256": {"variant", "persistent"},
            "skinny": {"variant"}}[variant]
    assert seen <= want and (seen >= want - {"copies", "valu"})


@pytest.mark.parametrize("shape,kw,want", [
    # generic and padded: copies only where the vector kernels cannot address or N, K < 16
    ((64, 64, 64), dict(variant="generic"), ("valu", 1)),
    ((64, 60, 64), {}, ("valu", 1)),
    ((100, 203, 333), {}, ("tiles_64", 1)),
    ((70, 80, 4111), {}, ("tiles_128", 8)),
    ((16, 1001, 4095), {}, ("skinny", 32)),
    ((1700, 1001, 700), {}, ("tiles_64", 1)),
    ((2000, 2001, 2003), {}, ("tiles_128", 1)),
    ((3000, 3001, 3003), {}, ("persistent", 1)),
    # short K: by C's bytes, and only where its rows are off 64 bytes
    ((12675, 8829, 87), {}, ("persistent", 1)),
    ((3436, 11135, 178), {}, ("persistent", 1)),
    ((11661, 6839, 26), {}, ("persistent", 1)),
    ((3325, 1267, 66), {}, ("tiles_128", 1)),
    ((8558, 4560, 327), {}, ("tiles_128", 1)),
    ((40000, 8, 200), {}, ("copies", 1)),
    ((4000, 5000, 9), {}, ("copies", 1)),
    ((16, 15, 139264), dict(variant="generic"), ("valu", 1)),
    # aligned, K off 64
    ((3000, 3008, 3024), {}, ("persistent", 1)),
    ((2000, 4096, 2064), {}, ("variant", 1)),
    ((84, 1040, 14832), {}, ("tiles_128", 16)),
    ((1000, 1008, 1008), {}, ("variant", 1)),
    ((8192, 8192, 8192), {}, ("variant", 1)),
])
def test_routes_on_either_side_of_the_rules(shape, kw, want):
    assert native_route(*shape, **kw)[:2] == want


def test_routes_without_a_workspace():
    """A stream captured before it has a workspace: unsplit, in place."""
    for shape, kw, want in (((70, 80, 4111), {}, "tiles_128"), ((16, 1001, 4095), {}, "tiles_64"),
                            ((3000, 3001, 3003), {}, "tiles_128"), ((3000, 3008, 3024), {}, "variant"),
                            ((84, 1040, 14832), {}, "variant")):
        assert native_route(*shape, scratch_limit=0, **kw)[0] == want, shape
    assert native_route(0, 16, 16) == ("none", 0, 0)
    with pytest.raises(_lib.HipGemmError, match="scratch limit"):
        native_route(16, 16, 16, scratch_limit=-1)
    with pytest.raises(_lib.HipGemmError, match="K%16"):
        native_route(100, 160, 100, "mfma_128x128")
    # copies above the optional bound: only the padded variant takes them
    big = (9000, 9001, 16001)
    assert native_route(*big, variant="padded")[0] == "persistent"
    assert native_route(*big, variant="padded")[2] > hg.OPTIONAL_BYTES
    assert native_route(*big, variant="generic")[0] == "tiles_128"


def test_candidates_are_ranked_by_what_runs():
    """Off the 16-byte grid the generic and padded candidates run the same
    kernels and carry the same figures; the winner is the one that keeps its
    workspace under capture. Aligned products never rank in-place tiles first."""
    for shape in ((1000, 1001, 999), (3000, 3001, 3003), (16, 1001, 4095), (100, 203, 333)):
        r = hg.optimize(*shape)
        by = {c["plan"]["variant"]: c for c in r["candidates"]}
        assert by["generic"]["objective"] == by["padded"]["objective"]
        assert by["generic"]["counts"] == by["padded"]["counts"]
        assert by["padded"]["counts"]["lds_bytes"] > 0 and r["winner"]["variant"] == "padded"
    for shape in ((1024, 1024, 1024), (3000, 3008, 3024), (256, 256, 256), (2000, 4096, 2064)):
        assert hg.optimize(*shape)["winner"]["variant"].startswith("mfma"), shape
    assert "64x64 tiles" in hg.native_check(hg.make_plan(100, 203, 333))[1]
    assert "padded copies" in hg.native_check(hg.make_plan(3000, 3008, 3024))[1]

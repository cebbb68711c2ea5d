"""Products whose operands the vector kernels cannot read as they are (sizes,
pitches or addresses that are not multiples of 16), read in place or, large
ones, over padded copies with C stored in place (needs a gfx950 GPU).

Sizes sit at the edges of what the kernels do: one 16-byte load short of and
past a row, K in whole, one-short and one-over slices, tiles and column blocks
with one to fifteen columns, K slices with a short last one. References are
exact float64 products on the GPU, added to D mod 2^32; C starts poisoned, with
a guard after it.
"""
import pytest

torch = pytest.importorskip("torch")

from veritac_amd import _lib
from veritac_amd.specializations.hip_gemm import backend as hg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    assert _lib.load_library().vt_device_count() >= 1, "GPU visible but not gfx950"
    return torch.device("cuda", 0)


def say(*args):
    print(*args, flush=True)


def wrapped(x):
    """Exact float64 integers mod 2^32, as int32."""
    return x.to(torch.int64).to(torch.int32)


def check(dev, variant, m, n, k, batch=1, shared=False, a_off=0, lda=None, b_off=0, ldb=None,
          ldc=None, shared_a=False, gap_a=0, route=None):
    """C = A.B and, in place, C = D + A.B through vt_gemm_i8 on flat buffers at
    the given byte offsets, pitches and gap between A's batches; row padding and
    the guard stay. route: the kernels the call is to run (_lib.ROUTES)."""
    say(variant, m, n, k, batch, shared, a_off, lda, b_off, ldb, ldc, shared_a, gap_a)
    lda, ldb, ldc = lda or k, ldb or n, ldc or n
    strides = (0, 0, 0, 0)
    if batch > 1:
        strides = (0 if shared_a else m * lda + gap_a, 0 if shared else k * ldb, m * ldc, m * ldc)
    if route is not None:
        got = _lib.gemm_route(m, n, k, lda, ldb, ldc, ldc, batch, *strides, has_d=True, variant=variant)
        assert got[0] == route, got
    g = torch.Generator(device=dev)
    g.manual_seed(m * 7 + n * 3 + k)
    bs = 1 if shared else batch
    As = 1 if shared_a else batch
    Af = torch.randint(-128, 128, (a_off + As * (m * lda + gap_a),), generator=g, device=dev, dtype=torch.int8)
    Bf = torch.randint(-128, 128, (b_off + bs * k * ldb,), generator=g, device=dev, dtype=torch.int8)
    A = Af[a_off:].view(As, m * lda + gap_a)[:, :m * lda].reshape(As, m, lda)[:, :, :k]
    B = Bf[b_off:].view(bs, k, ldb)[:, :, :n]
    AB = torch.matmul(A.double(), B.double())
    D = torch.randint(-2**31, 2**31, (batch * m * ldc + 64,), generator=g, device=dev, dtype=torch.int32)
    for d in (None, D):
        C = D.clone() if d is not None else torch.full_like(D, -2**31)
        before = C.clone()
        _lib.gemm_raw(Af.data_ptr() + a_off, Bf.data_ptr() + b_off, C.data_ptr() if d is not None else None,
                      C.data_ptr(), m, n, k, lda, ldb, ldc, ldc, batch, *strides,
                      variant, 0, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got, old = C[:batch * m * ldc].view(batch, m, ldc), before[:batch * m * ldc].view(batch, m, ldc)
        want = AB + old[:, :, :n].double() if d is not None else AB
        assert torch.equal(got[:, :, :n], wrapped(want)), "product"
        assert torch.equal(got[:, :, n:], old[:, :, n:]) and torch.equal(C[-64:], before[-64:]), "outside C"


# tiles: M and N around 64 and 128, K around the 64-deep slices and the pair
TILES = [(17, 16, 128), (65, 17, 129), (64, 63, 191), (100, 31, 143), (129, 65, 192), (70, 80, 193),
         (300, 129, 255), (100, 203, 333), (257, 79, 1000), (130, 1001, 257)]


@pytest.mark.parametrize("m,n,k", TILES)
@pytest.mark.parametrize("variant", ["generic", "padded"])
def test_tiles_in_place(dev, variant, m, n, k):
    check(dev, variant, m, n, k, route="tiles_64")


@pytest.mark.parametrize("m,n,k", [(1500, 1601, 129), (1700, 1301, 700), (1600, 1599, 70)])
def test_tiles_of_128(dev, m, n, k):
    check(dev, "padded", m, n, k, route="tiles_128")


@pytest.mark.parametrize("m,n,k", [(70, 333, 4111), (200, 1001, 15001), (999, 257, 9933), (129, 40, 4609),
                                   (300, 300, 3001)])
def test_k_slices(dev, m, n, k):
    assert _lib.gemm_route(m, n, k, k, n, n, n, variant="padded")[1] > 1
    check(dev, "padded", m, n, k, route="tiles_128" if k >= 4096 else "tiles_64")


# decode: column blocks of 16 and slabs of 256 with a short end, K tails, slices
@pytest.mark.parametrize("m,n,k", [(1, 17, 300), (16, 255, 4095), (3, 5329, 641), (16, 14335, 511),
                                   (33, 259, 1025), (64, 1001, 2047), (2, 100, 20001), (1, 16, 16384 + 1)])
@pytest.mark.parametrize("variant", ["generic", "padded"])
def test_decode_in_place(dev, variant, m, n, k):
    check(dev, variant, m, n, k, route="skinny")


@pytest.mark.parametrize("case", [
    dict(m=96, n=160, k=512, a_off=1), dict(m=96, n=160, k=512, b_off=3, ldb=167),
    dict(m=96, n=150, k=300, a_off=5, lda=311, b_off=9, ldb=151, ldc=157),
    dict(m=8, n=1000, k=900, a_off=7, lda=903, b_off=1, ldb=1003, ldc=1001),
    dict(m=50, n=90, k=200, batch=3), dict(m=50, n=90, k=200, batch=3, shared=True),
    dict(m=9, n=300, k=700, batch=3), dict(m=9, n=300, k=700, batch=2, shared=True, ldc=303)])
def test_addresses_pitches_and_batches(dev, case):
    check(dev, "padded", **case)


# the persistent kernel over padded copies: N and M off the tiles, C rows at
# any alignment, K off and on 256 (A is then read in place when its rows allow)
@pytest.mark.parametrize("case", [
    dict(m=3000, n=3001, k=2050), dict(m=2900, n=3002, k=2304), dict(m=4096, n=2575, k=2303),
    dict(m=3000, n=3003, k=2047, ldc=3010), dict(m=700, n=1999, k=2100, batch=5, shared=True),
    dict(m=700, n=1999, k=2100, batch=6)])
def test_large_products_store_c_in_place(dev, case):
    check(dev, "padded", route="persistent", **case)


# the same with K below the kernel's 256 (zeros from K on): C off 64-byte rows
# and large enough that storing it is what takes the time
@pytest.mark.parametrize("case", [
    dict(m=3400, n=3401, k=17), dict(m=3300, n=3313, k=130), dict(m=257, n=43009, k=48),
    dict(m=40001, n=300, k=64), dict(m=3072, n=3585, k=255), dict(m=700, n=2001, k=90, batch=10),
    dict(m=700, n=2001, k=90, batch=10, shared=True), dict(m=3500, n=3392, k=100, ldc=3401)])
def test_large_products_of_a_short_k(dev, case):
    check(dev, "padded", route="persistent", **case)


# aligned rows with K off 64, where copies for the persistent kernel pay: whole
# and ragged tiles, D, C at its own pitch, batches of both operands, of A or of
# B alone (B shared without the fold: A's batches lie apart); then sizes the
# estimate leaves on the tiles
@pytest.mark.parametrize("case", [
    dict(m=3000, n=3008, k=3024), dict(m=2816, n=3072, k=3088, ldc=3074), dict(m=3328, n=2560, k=2192),
    dict(m=1574, n=2448, k=2768, batch=2), dict(m=421, n=2320, k=2128, batch=7, shared=True, gap_a=16),
    dict(m=1546, n=672, k=2272, batch=7, shared_a=True)])
def test_large_aligned_products_with_k_off_64(dev, case):
    check(dev, "auto", route="persistent", **case)


@pytest.mark.parametrize("case", [
    dict(m=3072, n=3088, k=2832, ldc=3090), dict(m=2048, n=2064, k=4112), dict(m=500, n=528, k=1040),
    dict(m=900, n=2000, k=2320, batch=4), dict(m=900, n=2000, k=2320, batch=4, shared=True)])
def test_aligned_products_with_k_off_64_on_tiles(dev, case):
    check(dev, "auto", route="variant", **case)


# N or K below 16: copies of A and B (one of them where the other is aligned),
# a vector kernel, C copied out where N % 16; auto takes it from 3 * 2^24
# multiply-adds on
@pytest.mark.parametrize("case", [
    dict(m=40000, n=8, k=200), dict(m=9000, n=15, k=500, lda=503, ldb=17, ldc=18, a_off=3, b_off=1),
    dict(m=9000, n=15, k=512), dict(m=6000, n=11, k=300, batch=3), dict(m=6000, n=11, k=300, batch=3, shared=True),
    dict(m=30, n=7, k=16 * 1024 + 5, batch=16), dict(m=2000, n=3000, k=15), dict(m=3000, n=2000, k=12, ldc=2003),
    dict(m=1500, n=2001, k=9, batch=2, shared=True)])
def test_copies_where_n_or_k_is_below_16(dev, case):
    check(dev, "auto", route="copies", **case)


# one thread per output: the same sizes below that, tiny aligned products
@pytest.mark.parametrize("case", [
    dict(m=100, n=15, k=300), dict(m=3, n=9, k=1000, batch=3, ldc=10), dict(m=77, n=130, k=13, a_off=1),
    dict(m=64, n=64, k=64), dict(m=50, n=100, k=127)])
def test_one_thread_per_output(dev, case):
    check(dev, "generic", route="valu", **case)


# few aligned tiles over a K that has no equal slices of whole 128-deep steps
@pytest.mark.parametrize("m,n,k", [(84, 1040, 14832), (128, 512, 4112), (300, 512, 2064),
                                   (256, 2048, 8208), (66, 1600, 3088), (130, 256, 4224)])
def test_aligned_slices_of_unequal_depth(dev, m, n, k):
    route, ks, _ = _lib.gemm_route(m, n, k, k, n, n, n)
    assert route in ("tiles_64", "tiles_128") and ks >= 4
    check(dev, "auto", m, n, k)


def test_a_cold_capture_runs_without_a_workspace(dev):
    """The K slices' and copies' workspaces are not needed: a stream captured
    before it has any runs the same product without them."""
    for m, n, k in ((300, 300, 3001), (16, 1001, 4095), (3000, 3001, 2050), (3000, 3008, 3024), (9, 500, 5001),
                    (84, 1040, 14832), (4000, 15, 1000), (4000, 5000, 9)):
        say("cold capture", m, n, k)
        plan = hg.make_plan(m, n, k)
        A = torch.randint(-128, 128, (m, k), dtype=torch.int8, device=dev)
        B = torch.randint(-128, 128, (k, n), dtype=torch.int8, device=dev)
        want = torch.matmul(A.double(), B.double()).to(torch.int64).to(torch.int32)
        out = torch.zeros((m, n), dtype=torch.int32, device=dev)
        torch.cuda.synchronize()
        graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=stream):
            hg.run(plan, A, B, out=out)
        for _ in range(3):
            out.fill_(-2**31)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)

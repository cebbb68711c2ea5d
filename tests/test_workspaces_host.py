"""The library's per-stream workspaces, on the CPU: vt_gemm_i8's host code runs
against a HIP runtime that only logs (fake_hip.cpp), so what it launches and
allocates, and in which order host threads do, can be checked without a GPU.
Operand addresses are made up and never read."""
import json
import math
import os
import random
import subprocess
import sys

import pytest

from veritac_amd.specializations.hip_gemm import backend as hg

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = "/opt/rocm"

PRELUDE = """
import ctypes, json, sys, threading
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
fake.fake_capture.argtypes = [ctypes.c_void_p, ctypes.c_int]
from veritac_amd import _lib
_lib.load_library()
STREAM = 1 << 20

def gemm(m, n, k, variant="auto", stream=STREAM, batch=1, shared=True, where=0, call=_lib.gemm_raw):
    base = (1 + where) << 43
    multi = batch > 1
    call(base, base + (1 << 40), None, base + (2 << 40), m, n, k, k, n, n, n, batch,
         m * k if multi else 0, k * n if multi and not shared else 0, 0, m * n if multi else 0,
         variant, 0, stream)

def packed(m, n, k, batch=1, where=0, stream=STREAM, k_split=0):
    base = (1 + where) << 43
    multi = batch > 1
    _lib.gemm_packed_raw(base, base + (1 << 40), None, base + (2 << 40), m, n, k, k, n, n, batch,
                         m * k if multi else 0, n * (-(-k // 64) * 64) if multi else 0, 0,
                         m * n if multi else 0, k_split, stream)

def log():
    return [line.split(" ", 3) for line in fake.fake_log().decode().splitlines()]

def launches():
    return [e for e in log() if e[1] == "launch"]

def allocated():
    return [int(e[2]) for e in log() if e[1] == "malloc"]
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    """run(code) -> what the code printed as JSON, in a process of its own."""
    lib = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROCM, "include"),
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", lib, "-pthread"], check=True)

    def run(code):
        proc = subprocess.run([sys.executable, "-c", PRELUDE + code, lib], cwd=ROOT,
                              capture_output=True, text=True, timeout=120)
        assert proc.returncode == 0, proc.stderr
        return json.loads(proc.stdout)
    return run


# One call each that hands data from one launch to the next through a workspace.
TWO_LAUNCHES = [
    "gemm(84, 1040, 14832, where=w)",                      # K slices of unequal depth
    "gemm(3000, 3008, 3024, where=w)",                     # copies for the persistent kernel
    "gemm(3000, 3001, 3003, where=w)",                     # the same off the 16-byte grid
    "gemm(70, 80, 4111, 'generic', where=w)",              # K slices in place
    "gemm(40000, 8, 200, where=w)",                        # copies, a vector kernel, copy-out
    "gemm(48, 4096, 14336, where=w)",                      # row-major decode
    "gemm(128, 4096, 8192, where=w)",                      # equal K slices
    "packed(48, 4096, 14336, where=w)",                    # packed decode, split to read less of A
    "packed(48, 512, 8192, where=w)",                      # packed decode over few columns
    "gemm(128, 4096, 8192, where=w, call=_lib.gemm_noalloc_raw)",   # the static array
]


@pytest.mark.parametrize("call", TWO_LAUNCHES)
def test_a_call_keeps_its_workspace_until_its_last_launch(run, call):
    """Two host threads on one stream: no launch of one comes between the
    launches of the other's call, where it would overwrite what the first
    kernel left for the second."""
    got = run("""
def calls(w):
    for _ in range(6):
        %s
calls(0)                      # the stream's workspace, before the threads start
per_call = len(launches()) // 6
fake.fake_reset()
fake.fake_pause(1500)
ts = [threading.Thread(target=calls, args=(w,)) for w in (0, 1)]
[t.start() for t in ts]; [t.join() for t in ts]
print(json.dumps([per_call, launches()]))
""" % call)
    per_call, seen = got
    assert per_call == (3 if "40000" in call else 2)
    order = [e[0] for e in seen]
    assert sorted(set(order)) == ["0", "1"] and len(order) == 12 * per_call
    for i in range(0, len(order), per_call):
        assert len(set(order[i:i + per_call])) == 1, [e[0] + " " + e[3][:40] for e in seen]


def test_streams_do_not_wait_for_each_other(run):
    """The lock is a stream's own: a thread in the middle of a call on one
    stream does not hold up another stream's."""
    order = run("""
def calls(w):
    for _ in range(4):
        gemm(84, 1040, 14832, where=w, stream=STREAM + w)
calls(0); calls(1)
fake.fake_reset()
fake.fake_pause(3000)
ts = [threading.Thread(target=calls, args=(w,)) for w in (0, 1)]
[t.start() for t in ts]; [t.join() for t in ts]
print(json.dumps([e[0] for e in launches()]))
""")
    assert any(len(set(order[i:i + 2])) == 2 for i in range(0, len(order), 2))


def test_optional_workspaces_stay_within_their_bound(run):
    """Calls that could run without a workspace leave a stream at most 256 MiB
    of one kind, superseded workspaces included; past it they run without."""
    got = run("""
names = lambda: ["pad" if "pad_i8" in e[3] else "ragged" if "ragged" in e[3] else "other" for e in launches()]
out = []
for calls in ([(8192, 8192, 8208, "auto"), (8208, 8192, 8208, "auto"), (8192, 8192, 8208, "auto")],
              [(3000, 3008, 3024, "auto"), (3000, 3008, 3280, "auto"), (8192, 8192, 8208, "auto"),
               (8192, 8192, 9200, "auto")],
              [(3000, 3001, 3003, "generic"), (8001, 8003, 17001, "generic")]):
    fake.fake_reset()
    STREAM += 1
    for m, n, k, v in calls:
        gemm(m, n, k, v, stream=STREAM)
    out.append([allocated(), names()])
print(json.dumps(out))
""")
    mib = 1 << 20
    for sizes, _ in got:
        assert sum(sizes) <= 256 * mib, sizes
    # the second call needs more than is left and runs without copies; the third
    # fits the first one's workspace
    sizes, names = got[0]
    assert len(sizes) == 1 and names.count("ragged") == 2 and names[:2] == ["pad", "ragged"]
    assert names[-2:] == ["pad", "ragged"] and "other" in names[2:-2]
    # growth doubles while there is room, and never past what is left
    sizes, names = got[1]
    assert len(sizes) == 3 and sizes[1] == 2 * sizes[0] and names.count("ragged") == 3
    # the generic variant never needs copies: one of more than 256 MiB reads in place
    sizes, names = got[2]
    assert len(sizes) == 1 and names == ["pad", "ragged", "other"]


def test_a_workspace_is_allocated_while_another_thread_captures(run):
    """A thread capturing its own stream in global mode does not keep other
    threads' calls from their workspaces, nor change how they run; the caller's
    capture mode is as it was afterwards."""
    got = run("""
calls = [(84, 1040, 14832), (3000, 3008, 3024), (48, 4096, 14336), (16, 4096, 8192)]
for other in (0, 1):
    fake.fake_global_capture(other)
    for c in calls:
        STREAM += 1
        gemm(*c, stream=STREAM)
mode = ctypes.c_int(1)
fake.hipThreadExchangeStreamCaptureMode(ctypes.byref(mode))
kinds = [[e[1]] + (e[3:] if e[1] == "launch" else e[2:3]) for e in log()]
print(json.dumps([mode.value, kinds]))
""")
    mode, kinds = got
    assert mode == 0 and not [k for k in kinds if k[0] == "refused"]
    half = len(kinds) // 2
    assert kinds[:half] == kinds[half:] and [k[0] for k in kinds[:half]].count("malloc") == 4


def test_packed_grids_are_the_plan_mirror_s(run):
    """Column groups and K slices the library launches for packed decode are
    those backend.packed_columns and packed_split name, batches included."""
    shapes = []
    rng = random.Random(9)
    while len(shapes) < 150:
        m, n, k = rng.randint(1, 64), 16 * rng.randint(1, 800), 16 * rng.randint(1, 1000)
        batch = 1 if rng.random() < 0.5 else rng.randint(2, 16)
        if n * k * batch < 1 << 30:
            shapes.append((m, n, k, batch))
    got = run("""
out = []
for m, n, k, batch in %r:
    fake.fake_reset()
    packed(m, n, k, batch)
    out.append(launches()[0])
print(json.dumps(out))
""" % (shapes,))
    for (m, n, k, batch), first in zip(shapes, got):
        plan = hg.make_plan(m, n, k, batch=batch, variant=hg.PACKED_VARIANT)
        want = hg.packed_columns(plan)[1] * hg.packed_split(plan)[0] * batch
        assert "packed_skinny" in first[3] and int(first[3].split(" ")[0]) == want, (m, n, k, batch)


def test_captured_copies_do_not_depend_on_what_larger_calls_took(run):
    """A stream warmed up with a larger padded call, which reads its operands
    in place and takes no workspace, captures calls that would copy theirs:
    they run one thread per output."""
    got = run("""
gemm(2000, 2001, 2003)
fake.fake_capture(STREAM, 1)
fake.fake_reset()
gemm(40000, 8, 200)
gemm(4000, 5000, 9, "padded")
fake.fake_capture(STREAM, 0)
gemm(40000, 8, 200)
print(json.dumps([[e[3] for e in launches()], allocated()]))
""")
    names, sizes = got
    assert "generic_kernel" in names[0] and "generic_kernel" in names[1]
    assert ["pad_i8" in names[2], "unpad" in names[-1], len(sizes)] == [True, True, 1]


@pytest.mark.parametrize("variant", ["auto", "generic", "padded", "mfma_128x128", "mfma_256x128",
                                     "mfma_256x256", "skinny", hg.PACKED_VARIANT])
def test_launched_workgroups_are_the_reported_ones(run, variant):
    """required_resources counts the workgroups the library launches (copies
    and sums of K slices aside), for plans on either side of the routes' rules."""
    rng, calls, plans = random.Random(17), [], []
    while len(calls) < 120:
        m, n, k = (int(round(math.exp(rng.uniform(math.log(16), math.log(hi))))) for hi in (9000, 9000, 16000))
        if variant not in ("auto", "generic", "padded") or rng.random() < 0.4:
            n, k = n // 16 * 16, k // 16 * 16
        m = min(m, 64) if variant == "skinny" else m
        batch = 1 if rng.random() < 0.7 else rng.randint(2, 20)
        shared = variant != hg.PACKED_VARIANT and rng.random() < 0.5
        if m * n * batch < 2**29:
            plans.append(hg.make_plan(m, n, k, batch=batch, b_shared=shared, variant=variant))
            v, ks = plans[-1]["variant"], plans[-1]["k_split"]
            calls.append((m, n, k, batch, shared, v, ks))
    got = run("""
out = []
for m, n, k, batch, shared, v, ks in %r:
    fake.fake_reset()
    STREAM += 1        # a stream with all of its workspaces' bounds left
    if v == "skinny_packed":
        packed(m, n, k, batch, stream=STREAM)
    else:
        gemm(m, n, k, v, batch=batch, shared=shared, stream=STREAM)
    out.append([e[3] for e in launches()])
print(json.dumps(out))
""" % (calls,))
    for plan, names in zip(plans, got):
        gemms = [e.split(" ", 1) for e in names if "pad_i8" not in e and "unpad" not in e and "reduce" not in e]
        assert sum(int(g[0]) for g in gemms) == hg.required_resources(plan)[1], (plan, names)

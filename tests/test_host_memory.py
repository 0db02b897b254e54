"""The library's memory management and launch shapes on the CPU: a child process loads
tests/support/host_hip.cpp, which makes the HIP calls on the host alone, before
libtsac_hip.so, and goes through the C ABI as a program does."""
import pathlib
import subprocess
import sys
import textwrap

import pytest

TESTS = pathlib.Path(__file__).resolve().parent

PRELUDE = """
import ctypes, sys
sys.path.insert(0, {package!r})
hip = ctypes.CDLL({hip!r}, mode=ctypes.RTLD_GLOBAL)
hip.host_hip_total.argtypes = [ctypes.c_size_t]
hip.host_hip_largest.argtypes = [ctypes.c_size_t]
hip.host_hip_used.restype = ctypes.c_size_t
hip.host_hip_count.argtypes, hip.host_hip_count.restype = [ctypes.c_char_p], ctypes.c_long
hip.host_hip_launches.restype = ctypes.c_char_p
import numpy as np
from tsac_hip import native, synthetic
lib = native.library()
GiB, MiB = 1 << 30, 1 << 20

def counts():
    return {{name: hip.host_hip_count(name.encode()) for name in ("hipMalloc", "hipFree", "hipMallocAsync", "hipFreeAsync")}}

def launches():
    return [line.split() for line in hip.host_hip_launches().decode().splitlines()]
"""


@pytest.fixture(scope="session")
def host_hip(tmp_path_factory):
    target = tmp_path_factory.mktemp("host_hip") / "libhost_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(TESTS / "support" / "host_hip.cpp"), "-o", str(target)], check=True)
    return target


def run(host_hip, body):
    program = PRELUDE.format(package=str(TESTS.parent / "tsac-metal_amd"), hip=str(host_hip)) + textwrap.dedent(body)
    result = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True, timeout=300)
    assert result.returncode == 0, f"status {result.returncode}\n{result.stdout}{result.stderr[-3000:]}"
    return result.stdout


def test_encode_without_page_locked_memory(host_hip):
    """Where page-locked memory cannot grow, an encode goes through pageable memory, and
    the session's later ones, small or large, are as good as before."""
    run(host_hip, """
    geometry = synthetic.Geometry(width=256, heads=2, head_width=128, ffn=512, temporal_layers=1, codebook_layers=1,
                                  latent=256)
    session = native.HipModel(synthetic.random_model(geometry, seed=1)).session()
    def encode(frames):
        tokens = synthetic.pattern_tokens(frames * 12)
        return session.encode(native.header(frames, 1, 1, 12), tokens)
    small, large = encode(8), native.HipModel(synthetic.random_model(geometry, seed=1)).session()
    want = large.encode(native.header(40, 1, 1, 12), synthetic.pattern_tokens(40 * 12))
    hip.host_hip_pinned_fails(1)
    assert encode(40) == want
    assert encode(8) == small
    hip.host_hip_pinned_fails(0)
    assert encode(40) == want and encode(8) == small
    """)


def test_a_failed_allocation_leaves_no_error_behind(host_hip):
    """A call that failed for want of device memory does not fail the next call's launches."""
    run(host_hip, """
    linear = native.DeviceLinear(np.zeros((256, 256), np.int8), np.ones((1, 256), np.float32), np.zeros(256, np.float32))
    def apply(rows):
        return lib.tsac_hip_linear_apply(linear.handle, 1 << 20, rows, 1 << 40, native.PATH_AUTO, None)
    hip.host_hip_total(hip.host_hip_used())
    assert apply(1 << 20) != 0 and b"out of memory" in lib.tsac_hip_last_error()
    hip.host_hip_total(GiB)
    assert apply(4) == 0, lib.tsac_hip_last_error()
    """)


PROJECTION = """
def projection(k):
    return native.DeviceLinear(np.zeros((256, k), np.int8), np.ones((k // 256, 256), np.float32), np.zeros(256, np.float32))

def apply(linear, bytes_, ok=True):
    # rows in operand tiles, of about that many quantised bytes
    status = lib.tsac_hip_linear_apply(linear.handle, 1 << 44, bytes_ // linear.K, 1 << 45, native.PATH_GEMM, None)
    assert (status == 0) == ok, lib.tsac_hip_last_error()

linear = projection(4096)
base = hip.host_hip_used()
"""


def test_projection_buffers_outlive_larger_calls(host_hip):
    """Calls past the kept bytes take stream-ordered memory, as any other memory
    allocates and frees, and leave the kept buffers alone; sizes that fit are allocated
    once, and their frees (each waits for the device) end with the growing."""
    run(host_hip, PROJECTION + textwrap.dedent("""
    apply(linear, 16 * MiB)
    kept = hip.host_hip_used()
    assert kept - base >= 16 * MiB
    before = counts()
    for _ in range(5):
        apply(linear, 600 * MiB)
        assert hip.host_hip_used() == kept
        apply(linear, 16 * MiB)
    after = counts()
    assert after["hipMalloc"] == before["hipMalloc"] and after["hipFree"] == before["hipFree"]
    assert after["hipMallocAsync"] - before["hipMallocAsync"] == 5
    for size in (127, 400, 300, 16, 480):  # growing past the bound takes the smaller ones' place
        apply(linear, size * MiB)
        assert hip.host_hip_used() - base <= 512 * MiB
    before = counts()
    for size in (16, 480, 127, 300, 600, 400):
        apply(linear, size * MiB)
    after = counts()
    assert after["hipMalloc"] == before["hipMalloc"] and after["hipFree"] == before["hipFree"]
    del linear
    import gc; gc.collect()
    assert hip.host_hip_used() == 0
    """))


def test_projection_buffers_give_way_where_memory_is_short(host_hip):
    """Idle buffers that are too small are freed where a larger one, kept or
    stream-ordered, finds no memory; a call that finds none all the same fails alone."""
    run(host_hip, PROJECTION + textwrap.dedent("""
    apply(linear, 100 * MiB)
    hip.host_hip_total(base + 260 * MiB)
    apply(linear, 200 * MiB)
    hip.host_hip_total(base + 660 * MiB)
    apply(linear, 600 * MiB)
    apply(linear, 100 * MiB)
    hip.host_hip_total(base + 300 * MiB)
    apply(linear, 400 * MiB, ok=False)
    apply(linear, 600 * MiB, ok=False)
    apply(linear, 100 * MiB)
    """))


def test_projection_buffers_of_overlapping_calls(host_hip):
    run(host_hip, PROJECTION + textwrap.dedent("""
    import random, threading
    failures = []
    def work(seed):
        rng = random.Random(seed)
        for _ in range(200):
            size = rng.choice((1, 20, 130, 300, 510, 700)) * MiB
            if lib.tsac_hip_linear_apply(linear.handle, 1 << 44, size // 4096, 1 << 45, native.PATH_GEMM, None):
                failures.append(lib.tsac_hip_last_error())
    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads: t.start()
    for t in threads: t.join()
    assert not failures, failures
    assert hip.host_hip_used() - base <= 512 * MiB
    del linear
    import gc; gc.collect()
    assert hip.host_hip_used() == 0
    """))


DAC = """
geometry = synthetic.Geometry(width=256, heads=2, head_width=128, ffn=512, temporal_layers=1, codebook_layers=1,
                              latent=256, books=9, channels=1)
session = native.HipModel(synthetic.random_model(geometry, seed=1)).session()
model = synthetic.random_dac(channels=1, books=9, seed=1)
dac = native.HipDac(model)
launches()
"""


@pytest.mark.parametrize("frames,groups", [(2700, 400), (400, 2700), (20, 60000)])
def test_analysis_of_very_many_channels(host_hip, frames, groups):
    """Interleaved PCM whose channels' rows span more than 2 GiB is analysed, chunks long
    and short: offsets are relative to a workgroup's first frame."""
    run(host_hip, DAC + f"frames, groups = {frames}, {groups}" + textwrap.dedent("""
    pcm = np.zeros((frames * 512, groups), np.float32)  # never touched
    tokens = np.zeros(frames * groups, np.uint16)
    status = lib.tsac_hip_dac_analyze(session.handle, dac.handle, native._ptr(pcm, ctypes.c_float), frames, groups, 1,
                                      native._ptr(tokens, ctypes.c_uint16))
    assert status == 0, lib.tsac_hip_last_error()
    assert len(launches()) >= groups * 31
    """))


CHUNKS = DAC + """
def analyze(frames, groups=1):
    launches()
    dac.analyze(session, np.zeros((frames * 512, groups), np.float32), frames, groups)
    return sum("rvq_encode" in line[0] for line in launches()) // groups  # chunks

def synthesize(frames):
    launches()
    dac.synthesize(session, np.zeros(frames * 9, np.uint16), frames)
    return sum("rvq_decode" in line[0] for line in launches())

base = hip.host_hip_used()
SLOTS = {False: 3 * 64 * 512 * 4, True: 3 * 96 * 512 * 4}  # bytes a frame
"""


def test_dac_chunks_follow_the_memory(host_hip):
    """Long recordings run in equal chunks of up to 2,708 latent frames (the default
    element limit; at most 3,072 by any), in the reference's 400 where an eighth of the
    device's free memory holds no more."""
    run(host_hip, CHUNKS + textwrap.dedent("""
    assert [analyze(n) for n in (1, 400, 401, 2584, 2708, 2709, 8000)] == [1, 1, 1, 1, 1, 2, 3]
    assert [synthesize(n) for n in (1, 400, 401, 2584, 2708, 2709, 8000)] == [1, 1, 1, 1, 1, 2, 3]
    wide = native.HipDac(model, native.Limits(0, 0, 0, 0, 1 << 30))
    launches()
    wide.analyze(session, np.zeros((3073 * 512, 1), np.float32), 3073)
    assert sum("rvq_encode" in line[0] for line in launches()) == 2
    session.clear()
    hip.host_hip_total(base + GiB)
    assert analyze(2584) == 7 and synthesize(2584) == 7
    """))


def test_dac_graphs_share_their_scratch(host_hip):
    """Analysis and synthesis keep one set of slots between them, as large as the larger
    needs, next to their inputs and outputs."""
    run(host_hip, CHUNKS + textwrap.dedent("""
    analyze(2584), synthesize(2584)
    assert hip.host_hip_used() - base < 2584 * SLOTS[True] + 64 * MiB
    """))


def test_dac_scratch_is_given_back_where_memory_is_short(host_hip):
    """Slots kept from a call with more memory are freed once they exceed an eighth of what
    is left, and at once where another of the session's buffers finds no memory; where
    the memory for a large chunk cannot be had, chunks of 400 frames run."""
    run(host_hip, CHUNKS + textwrap.dedent("""
    for frames, chunks in ((2584, 7), (100, 1)):  # by a long call and by a short one
        hip.host_hip_total(288 * GiB)
        assert synthesize(2584) == 1
        hip.host_hip_total(hip.host_hip_used() + 300 * MiB)
        assert synthesize(frames) == chunks
        assert hip.host_hip_used() - base < 422 * SLOTS[True] + 64 * MiB
    session.clear()

    hip.host_hip_total(288 * GiB)
    assert synthesize(2584) == 1
    hip.host_hip_total(hip.host_hip_used() + 12 * GiB)
    assert analyze(2584, groups=2450) == 1  # 12.1 GiB of samples
    session.clear()

    hip.host_hip_total(288 * GiB)
    hip.host_hip_largest(200 * MiB)
    assert synthesize(2584) == 7 and analyze(2584) == 7
    """))


@pytest.mark.parametrize("sequences,heads,longest", [(1, 1, 2_200_000), (1, 1, 4_194_240), (3, 2, 1_100_000), (2, 1, 65536 * 8),
                                                     (4_300_000, 16, 1), (16_000_000, 16, 12), (5_500_000, 16, 20),
                                                     (4_300_000, 16, 65), (1, 65535, 300), (2_000_000, 1, 17)])
@pytest.mark.parametrize("width", [64, 128])
def test_causal_attention_launches_any_size(host_hip, sequences, heads, longest, width):
    """Every (sequence, head, query) has a workgroup, in launches within the limits of a grid."""
    run(host_hip, f"sequences, heads, longest, width = {sequences}, {heads}, {longest}, {width}" + textwrap.dedent("""
    status = lib.tsac_hip_attention_causal(1 << 44, heads, width, 1 << 45, 1 << 46, 1 << 47, sequences, longest, None,
                                           1.0, 1 << 48, None)
    assert status == 0, lib.tsac_hip_last_error()
    pairs = 0
    for name, x, y, z, threads in launches():
        if "short_kernel" in name:
            pairs += int(x) * int(threads) // 64  # a wave each, up to 3 to spare
        else:
            pairs += int(x)
            queries = int(name.split("Li")[3].split("E")[0])
            assert int(y) * int(z) * queries >= longest
    assert sequences * heads <= pairs <= sequences * heads + 3 * len(launches() or [0]) + 3 * 64
    """))


def test_causal_attention_refuses_no_heads(host_hip):
    run(host_hip, """
    for longest in (1, 100):
        assert lib.tsac_hip_attention_causal(1 << 44, 0, 64, 1 << 45, 1 << 46, 1 << 47, 1, longest, None, 1.0, 1 << 48,
                                             None) != 0
    """)


def test_operators_without_page_locked_memory(host_hip):
    """The calls that report a nonfinite input run without page-locked memory too."""
    run(host_hip, """
    hip.host_hip_pinned_fails(1)
    linear = native.DeviceLinear(np.zeros((256, 256), np.int8), np.ones((1, 256), np.float32), np.zeros(256, np.float32))
    used = hip.host_hip_used()
    a, b, c = 1 << 44, 1 << 45, 1 << 46
    for rows in (3, 100, 5000):
        assert lib.tsac_hip_linear_apply(linear.handle, a, rows, b, native.PATH_AUTO, None) == 0, lib.tsac_hip_last_error()
        assert lib.tsac_hip_bf8l(a, rows, 256, b, c, None) == 0, lib.tsac_hip_last_error()
        assert lib.tsac_hip_bf8l_tiles(a, rows, 256, b, c, None) == 0, lib.tsac_hip_last_error()
        assert lib.tsac_hip_softmax(a, rows, 256, b, None) == 0, lib.tsac_hip_last_error()
    after = counts()
    assert after["hipMallocAsync"] == after["hipFreeAsync"] == 12
    hip.host_hip_pinned_fails(0)
    assert lib.tsac_hip_softmax(a, 3, 256, b, None) == 0
    assert counts() == after
    """)

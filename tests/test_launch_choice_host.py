"""What the library launches, on the CPU: its own choice of kernels through tests/host_launch_recorder.cpp, which stands in
for the HIP runtime (256 CUs) and writes down the launches of a call."""

import os
import random
import re
import subprocess

import pytest

from wave_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
QUERY = -1  # scratch: what the library's query names


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rec") / "host_launch_recorder")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-rdynamic", "-o", exe,
                           os.path.join(ROOT, "tests", "host_launch_recorder.cpp"), "-ldl"])

    def run(calls):
        """(kind, m, n, k, out_dtype, x, y, b_layout, split_k or groups, variant, scratch) -> status and launches"""
        text = "".join(" ".join(str(v) for v in c) + "\n" for c in calls)
        out = subprocess.run([exe, _lib.LIB_PATH], input=text, capture_output=True, text=True)
        assert out.returncode == 0, out.stderr[-2000:]
        lines = out.stdout.split("\n")[:-1]
        assert len(lines) == len(calls)
        return lines

    return run


def log_size(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def random_gemms(count, seed):
    rng = random.Random(seed)
    calls = []
    while len(calls) < count:
        m, n, k = round(log_size(rng, 1, 8192)), 8 * round(log_size(rng, 128, 32768) / 8), 32 * round(log_size(rng, 512, 16384) / 32)
        if rng.random() < 0.5:
            n = 256 * -(-n // 256)
        if rng.random() < 0.7:
            k = 256 * -(-k // 256)
        b = rng.choice([_lib.B_ROW_MAJOR, _lib.B_PRESHUFFLE])
        if b == _lib.B_PRESHUFFLE:
            n, k = 16 * -(-n // 16), 64 * -(-k // 64)
        a_scale, b_scale = rng.choice([(0, 0), (0, 0), (1, 1), (2, 2), (2, 2), (0, 2), (2, 0), (1, 2), (3, 0), (3, 2)])
        calls.append(("gemm", m, n, k, rng.randint(0, 1), a_scale, b_scale, b, 0, 0))
    return calls


def same_with_more_scratch(launches, calls):
    want = launches([c + (QUERY,) for c in calls])
    assert all(w.startswith("0 |") for w in want)
    for scratch in (1 << 28, 1 << 32):
        for call, a, b in zip(calls, want, launches([c + (scratch,) for c in calls])):
            assert a == b, (call, scratch)


def test_scratch_beyond_the_query_changes_nothing(launches):
    """A call takes the same kernels, and so gives the same bits, with exactly the scratch that the query names and with any
    larger buffer (the Python wrapper keeps one that grows)."""
    calls = random_gemms(6000, 0)
    # more 256x256 tiles than CUs, N inside a tile, a last round of tiles that a cut along K would fill
    calls += [("gemm", m, n, k, o, 2, 2, 0, 0, 0) for m, n, k in [(5882, 17024, 5824), (5818, 28512, 3584), (539, 24648, 8960)]
              for o in (0, 1)]
    same_with_more_scratch(launches, calls)


def test_mxfp8_scratch_beyond_the_query_changes_nothing(launches):
    """The same for MXFP8, K in whole and in half scale blocks (K % 256 = 128)."""
    rng = random.Random(1)
    calls = [("mxfp8", 32, 9472, 8832, 0, 0, 0, 0, 0, 0), ("mxfp8", 15, 1024, 5504, 1, 1, 2, 0, 0, 0)]
    while len(calls) < 3000:
        m, n, k = round(log_size(rng, 1, 8192)), 8 * round(log_size(rng, 64, 32768) / 8), 128 * round(log_size(rng, 512, 16384) / 128)
        a_fmt, b_fmt = rng.choice([(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 1)])
        calls.append(("mxfp8", m, n, k, rng.randint(0, 1), a_fmt, b_fmt, 0, 0, 0))
    same_with_more_scratch(launches, calls)


@pytest.mark.parametrize("n,out,whole", [(13480, _lib.OUT_F32, False), (13472, _lib.OUT_F32, True), (13488, _lib.OUT_F32, False),
                                         (13416, _lib.OUT_BF16, False), (13440, _lib.OUT_BF16, True), (13472, _lib.OUT_BF16, False)])
def test_mxfp8_persistent_kernel_stores_part_lines_with_the_default_policy(launches, n, out, whole):
    """Rows of C that are not whole 128-byte lines must not go out non-temporal (4363 x 13480 x 768: 143 us against 73)."""
    line, = launches([("mxfp8", 4363, n, 768, out, 0, 1, 0, 0, 0, QUERY)])
    flag = "true" if whole else "false"
    assert "persist_gemm_fp8_kernel" in line and f", 0, 1, {flag}> <256,1,1>" in line, line


@pytest.mark.parametrize("scratch", [QUERY, 1 << 30])
@pytest.mark.parametrize("k,relaid", [(288, False), (480, False), (736, False), (512, True), (800, True), (2880, True)])
def test_grouped_short_k_with_a_partial_tile_reads_its_scales_as_they_come(launches, k, relaid, scratch):
    """22 rows of 16 experts x 352 x 320: 8.2 us without the re-layout launch, 11.2 with it."""
    for a_scale, b_scale in ((_lib.SCALE_ROW_MAJOR, _lib.SCALE_ROW_MAJOR), (_lib.SCALE_MFMA32, _lib.SCALE_E8M0_SHUFFLE)):
        line, = launches([("grouped", 3000, 352, k, 1, a_scale, b_scale, 0, 16, 0, scratch)])
        assert line.startswith("0 |") and ("scale_" in line) == relaid, line


def test_deep_ring_splits_stay_within_one_round_on_every_xcd(launches):
    """Tiles are dealt to eight XCDs of 32 CUs in runs of equal length, each part along K anew: the longest run times the
    parts must fit (84 tiles in three parts were 33 workgroups on seven XCDs, and took two rounds)."""
    calls = [c for c in random_gemms(20000, 2) if c[5] == c[6]]
    calls += [("gemm", 2, 5376, 10240, 0, 2, 2, 0, 0, 0), ("gemm", 4, 2304, 21504, 1, 0, 0, 1, 0, 0)]
    calls += [("mxfp8", m, n, k, 0, 0, 0, 0, 0, 0) for _, m, n, k, *_ in random_gemms(3000, 3) if k % 128 == 0]
    split = 0
    for call, line in zip(calls, launches([c + (QUERY,) for c in calls])):
        found = re.search(r"deep_gemm_kernel<.*?> <(\d+),(\d+),1>", line)
        if found:
            x, parts = int(found[1]), int(found[2])   # x is padded to a multiple of eight
            split += parts > 1
            assert x % 8 == 0 and x // 8 * parts <= 32, (call, line)
    assert split > 200
    # ... unless there is no other way: half scale blocks, staged up to 31 K tiles a part (111 us on the tile kernel, 37 here)
    line, = launches([("mxfp8", 675, 1760, 11136, 1, 0, 0, 0, 0, 0, QUERY)])
    assert "deep_gemm_kernel" in line and "<88,3,1>" in line, line


ROW, E8M0, MFMA32 = _lib.SCALE_ROW_MAJOR, _lib.SCALE_E8M0_SHUFFLE, _lib.SCALE_MFMA32


@pytest.mark.parametrize("m,n,k,scales,preshuffled,deep", [
    # the streaming kernel keeps (us there, on the deep ring):
    (3, 2048, 2560, MFMA32, 1, False),   # 5.2, 6.8
    (1, 3584, 2816, MFMA32, 1, False),   # 5.2, 7.1
    (5, 1280, 2560, E8M0, 1, False),     # 5.3, 6.7
    (7, 1536, 2816, E8M0, 0, False),     # 1.14 of the time
    (18, 4096, 4096, MFMA32, 0, False),  # 1.14
    (24, 3072, 4096, MFMA32, 1, False),  # 1.23
    (4, 1440, 1536, ROW, 1, False),      # 5.1, 6.6
    (1, 5376, 12544, ROW, 0, False),     # 12.4, 14.8
    (4, 2304, 21504, ROW, 1, False),     # 11.4, 15.3
    # the mid-M kernel keeps:
    (188, 16952, 2176, MFMA32, 0, False),  # 12.3, 15.5
    (165, 30208, 1280, MFMA32, 0, False),  # 10.3, 12.6
    (120, 14592, 6272, MFMA32, 0, False),  # 22.0, 25.2
    (57, 4936, 3072, ROW, 0, False),       # 8.5; the ring, whose staged rows have become faster, 7.8
    # the deep ring keeps, on the near side of the same borders:
    (3, 2048, 2048, MFMA32, 0, True), (12, 12288, 2816, MFMA32, 0, True), (2, 8192, 2560, E8M0, 1, True),
    (18, 4096, 3072, MFMA32, 0, True), (24, 3072, 6144, MFMA32, 1, True), (40, 2048, 4096, E8M0, 1, True),
    (4, 1440, 1280, ROW, 1, True), (2, 3840, 12544, ROW, 0, True), (2, 3200, 13568, MFMA32, 0, True),
    (188, 16384, 2048, MFMA32, 0, True), (120, 8192, 6144, MFMA32, 0, True), (120, 12288, 4096, MFMA32, 0, True),
    (96, 4936, 4096, ROW, 0, True), (256, 28672, 6144, MFMA32, 0, True), (1000, 7168, 4096, MFMA32, 0, True),
])
def test_borders_of_the_deep_ring(launches, m, n, k, scales, preshuffled, deep):
    """Shapes on both sides of the borders between the deep-ring kernel and the two that read B straight."""
    n -= n % 16 if preshuffled else 0
    for out in (_lib.OUT_F32, _lib.OUT_BF16):
        line, = launches([("gemm", m, n, k, out, scales, scales, preshuffled, 0, 0, QUERY)])
        assert ("deep_gemm_kernel" in line) == deep, line


@pytest.mark.parametrize("m,n,k", [(128, 2256, 6496), (190, 2904, 12736), (309, 1536, 9504)])
def test_deep_ring_prices_rows_that_are_not_whole_lines(launches, m, n, k):
    """K % 256 != 0 with a row-major B: K tiles take longer, and these are faster in parts (190 x 2904 x 12736: 26.2 us
    whole on 64x64 tiles, 19.6 in parts, the kernel before 19.4)."""
    line, = launches([("gemm", m, n, k, 1, MFMA32, MFMA32, 0, 0, 0, QUERY)])
    assert "deep_gemm_kernel" in line and "splitk_reduce" in line, line


def parametrized(test, names):
    return next(mark.args[1] for mark in test.pytestmark if mark.name == "parametrize" and mark.args[0] == names)


def test_the_deep_ring_tests_through_the_library_choice_reach_it(launches):
    """What tests/test_gpu_deep_ring*.py run without naming a kernel must run on the one that they are about (up to 16 rows
    and against a wide B they stand on both sides of its borders)."""
    import test_gpu_deep_ring as four
    import test_gpu_deep_ring_mxfp8 as eight

    code = {"row": ROW, "e8m0": E8M0, "mfma32": MFMA32}
    calls = []
    small = [(m, n, k) for m in parametrized(four.test_small_tiles, "m") for n, k in parametrized(four.test_small_tiles, "n,k")]
    for shapes, test in ((small, four.test_small_tiles), (parametrized(four.test_large_tiles, "m,n,k"), four.test_large_tiles),
                         (parametrized(four.test_splits, "m,n,k"), four.test_splits)):
        calls += [("gemm", m, n, k, _lib.OUT_F32, code[s], code[s], 0, 0, 0) for m, n, k in shapes
                  for s in parametrized(test, "scales")]
    for m, n, k in parametrized(four.test_partial_last_k_tile, "m,n,k"):
        calls += [("gemm", m, n, k + t, _lib.OUT_F32, MFMA32, MFMA32, 0, 0, 0) for t in parametrized(four.test_partial_last_k_tile, "tail")]
    for test in (eight.test_formats, eight.test_splits_and_long_k):
        calls += [("mxfp8", m, n, k, _lib.OUT_F32, a, b, 0, 0, 0) for m, n, k in parametrized(test, "m,n,k")
                  for a, b in parametrized(test, "fmt")]
    calls = [c for c in calls if c[0] == "mxfp8" or (c[1] > 16 and c[2] <= 16384) or c[3] > 8192]
    assert len(calls) > 150
    off = [(c, line) for c, line in zip(calls, launches([c + (QUERY,) for c in calls])) if "deep_gemm_kernel" not in line]
    assert not off, off


@pytest.mark.parametrize("m,n,k,preshuffled,tile,parts", [
    (1062, 5088, 15360, 1, "256, 128", 1),   # 55.9 us; 73.3 on the 128x256 tiles that a row-major B takes
    (137, 15504, 7424, 1, "128, 128", 1),    # 25.7; 36.7 on 256x128
    (201, 16128, 17472, 0, "256, 128", 2),   # rows of B that are not whole lines: 59.4 in two parts, 84.2 whole
    (496, 2560, 9472, 1, "128, 128", 3),
    (2048, 4096, 14336, 0, "128, 256", 1),   # 59.6
    (1000, 7168, 4096, 0, "256, 128", 1),    # 21.3
])
def test_deep_ring_estimates(launches, m, n, k, preshuffled, tile, parts):
    """The choice of tile and parts sees the layout of B and its lines, and has no term that makes a larger B cheaper."""
    line, = launches([("gemm", m, n, k, 1, MFMA32, MFMA32, preshuffled, 0, 0, QUERY)])
    found = re.search(r"DeepCfg<(\d+, \d+), .*?> <\d+,(\d+),1>", line)
    assert found and found[1] == tile and int(found[2]) == parts, line

"""What the library's host code launches and how it keeps its scratch, on a
HIP runtime that only records (fake_hip.cpp): no GPU, nothing computed."""
import pytest

import fakehip


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fakehip.build(tmp_path_factory.mktemp("fake_hip"))


def new_allocs(before, after):
    """Indices of the allocations that a step made."""
    return range(len(before["allocs"]), len(after["allocs"]))


# A graph captured after an eager call holds the scratch's addresses: a later
# call that needs more must not free it.  The argmax's pairs share their buffer
# with the tile GEMM's partial sums, so a prompt whose K is split grows it.
@pytest.mark.parametrize("grow", [["gemm", "q4_k", 5120, 17408, 64], ["gemm", "iq4_xs", 5120, 17408, 333],
                                  ["argmax", 248320, 64]], ids=lambda g: g[0] + "_" + str(g[1]))
def test_captured_argmax_keeps_its_scratch(fake, grow):
    r = fakehip.run(fake, [["norm", 64, 1, 0], ["argmax", 248320, 1], ["capture", 1], ["argmax", 248320, 1],
                           ["capture", 0], grow])
    assert [s["status"] for s in r] == [0] * len(r)
    held = new_allocs(r[0], r[1])
    assert len(held) == 2 and len(r[3]["allocs"]) == len(r[1]["allocs"])  # pairs, counters; nothing in the capture
    assert len(r[-1]["allocs"]) > len(r[1]["allocs"])                     # (it did grow)
    assert [r[-1]["allocs"][i][1] for i in held] == [0, 0]


# What is kept is bounded: a buffer that no graph holds is freed when it is
# replaced, and one that a graph holds by a successor of at least twice its size.
def test_kept_scratch_is_bounded(fake):
    steps = [["norm", 64, 1, 0], ["argmax", 248320, 1], ["capture", 1], ["argmax", 248320, 1], ["capture", 0]]
    for rows in range(2, 70):
        steps.append(["argmax", 248320, rows])
        if rows < 20:  # (a graph after each growth, then growth without graphs)
            steps += [["capture", 1], ["argmax", 248320, rows], ["capture", 0]]
    r = fakehip.run(fake, steps)
    base = len(r[0]["allocs"])
    for s in r:
        live = [n for n, freed in s["allocs"][base:] if not freed]
        pairs = sorted(n for n in live if n >= 122 * 8)
        assert sum(pairs[:-1]) <= (pairs[-1] if pairs else 0)
    assert sum(f for n, f in r[-1]["allocs"][base:]) > 0


# The buffers that a capture did not hand to a launch are not held by it.
def test_capture_holds_what_it_uses(fake):
    r = fakehip.run(fake, [["gemm", "q4_k", 5120, 17408, 64], ["argmax", 1000, 1], ["capture", 1], ["argmax", 1000, 1],
                           ["capture", 0], ["gemm", "q4_k", 5120, 17408, 128]])
    xh = 64 * 17408 * 2
    assert [f for n, f in r[-1]["allocs"] if n == xh] == [1]


# ------------------------------------------------------------------ tile GEMM plans
def tile_launch(step):
    """The tile kernel of a GEMM step: (name, template arguments, workgroups, K ranges)."""
    (k,) = [v for v in step["launches"] if v["name"] in ("gemm_few_kernel", "gemm_many_kernel", "gemm_mfma_kernel")]
    return k["name"], k["args"], k["grid"][0] * k["grid"][1], k["grid"][2]


# A context whose partial-sum buffer may not grow (reserved: it holds the argmax
# pairs only; or its stream is being captured; or no memory) plans for one K
# range: the tile that fills the CUs without a split, not the split plan's tile
# on the fraction of the CUs that it was cut for.
@pytest.mark.parametrize("fmt,M,K,N", [("q4_k", 5120, 17408, 64), ("q4_k", 5120, 17408, 333), ("q4_k", 2048, 6144, 101),
                                       ("iq4_xs", 5120, 17408, 333), ("q8_0", 2048, 6144, 512), ("q2_k", 2048, 6144, 20)])
@pytest.mark.parametrize("how", ["reserved", "captured", "memory"])
def test_one_range_is_planned_as_one(fake, fmt, M, K, N, how):
    call, warm = ["gemm", fmt, M, K, N], ["tile", fmt, 1 << 18, K, N]  # (warm: many rows, no split; grows X's buffer, not the partials)
    limit = {"reserved": [["reserve", N * K, 248320, 1]], "captured": [warm, ["capture", 1]],
             "memory": [warm, ["fail_above", 1]]}[how]
    free = fakehip.run(fake, [call])[-1]
    one = fakehip.run(fake, [call], OKF_GEMM_SPLIT="0")[-1]
    got = fakehip.run(fake, limit + [call])[-1]
    assert [s["status"] for s in (free, one, got)] == [0, 0, 0]
    assert tile_launch(free)[3] > 1 and "gemm_ksum_kernel" in [v["name"] for v in free["launches"]]
    assert tile_launch(got)[3] == 1 and "gemm_ksum_kernel" not in [v["name"] for v in got["launches"]]
    assert tile_launch(got)[2] > tile_launch(free)[2]
    assert tile_launch(got) == tile_launch(one)  # (OKF_GEMM_SPLIT=0 plans one range of both kernels)


# With room for some of the ranges, as many as fit.
def test_ranges_that_fit(fake):
    M, K, N = 5120, 17408, 64
    r = fakehip.run(fake, [["tile", "q4_k", M, K // 17, N], ["reserve", N * K, 248320, 2 * M * N * 4 // 976 + 1],
                           ["gemm", "q4_k", M, K, N]])
    assert tile_launch(r[-1])[3] == 2


# Millions of tokens on a few rows: within the grid's limits (65535 in y and z).
@pytest.mark.parametrize("M,K,N", [(1, 512, 4200001), (16, 512, 4200001), (64, 256, 2000000)])
def test_many_tokens_fit_the_grid(fake, M, K, N):
    (r,) = fakehip.run(fake, [["gemm", "q4_k", M, K, N]])
    assert r["status"] == 0
    for v in r["launches"]:
        assert max(v["grid"][1:]) <= 65535 and v["grid"][0] * v["block"] < 1 << 32


# Tall matrices of short rows: a few-token workgroup there is mostly the sum of its
# wavefronts' tiles (Q4_K 65536 x 512, N = 33 36 us, on gemm_many_kernel 21).
@pytest.mark.parametrize("fmt,M,K,N,few", [("q4_k", 65536, 512, 33, False), ("q4_0", 151936, 1024, 64, False),
                                           ("iq4_nl", 151936, 1024, 33, False), ("q4_k", 65536, 512, 17, True),
                                           ("q4_k", 6144, 2048, 19, True), ("q4_k", 1000, 512, 64, True)])
def test_tall_short_rows(fake, fmt, M, K, N, few):
    (r,) = fakehip.run(fake, [["gemm", fmt, M, K, N]])
    assert tile_launch(r)[0] == ("gemm_few_kernel" if few else "gemm_many_kernel")


# ------------------------------------------------------------------ superblock matvec
# gemv_sb_kernel keeps a lane's staged activations in registers: up to five
# rounds (K = 20480); longer rows stay with the other matvecs, alone and paired.
@pytest.mark.parametrize("fmt", ["q8_0", "q5_k", "q4_0", "iq4_nl", "iq4_xs", "q4_k"])
def test_superblock_matvec_rows(fake, fmt):
    ks = (17408, 20480, 20736, 24576, 28672, 36864)
    r = fakehip.run(fake, [["gemv", fmt, 8192, K] for K in ks] + [["gate_up", fmt, 8192, K] for K in ks])
    assert [s["status"] for s in r] == [0] * len(r)
    sb = [s["launches"][0]["name"] == "gemv_sb_kernel" for s in r]
    assert sb == 2 * [K <= 20480 for K in ks]


# Gate and up paired: an even number of rows whose items fill one round of the
# 256 lanes.
@pytest.mark.parametrize("fmt,K", [("q4_k", 3072), ("q5_k", 3072), ("q5_k", 7168), ("iq4_xs", 3072), ("q5_k", 6912)])
def test_paired_superblock_rows(fake, fmt, K):
    M = 40320
    (r,) = fakehip.run(fake, [["gate_up", fmt, M, K]])
    (k,) = [v for v in r["launches"] if v["name"] == "gemv_sb_kernel"]
    rows = 2 * -(-M // k["grid"][0])
    assert k["block"] == 256 and 200 < rows * (K // 256) <= 256


# Where gemv_sb_kernel is the slower one: some short rows of whole 1024s, and one to
# one and a half 32-row workgroups a CU of long rows (Q8_0; IQ4_XS paired).
@pytest.mark.parametrize("call,fmt,M,K,sb", [
    ("gemv", "q8_0", 9803, 14336, False), ("gemv", "q8_0", 8192, 14336, True), ("gemv", "q8_0", 12289, 14336, True),
    ("gemv", "q4_k", 9803, 14336, True), ("gemv", "iq4_xs", 4096, 6144, False), ("gemv", "iq4_xs", 4096, 6400, True),
    ("gemv", "iq4_xs", 17408, 5120, True), ("gemv", "q8_0", 4096, 6144, False), ("gemv", "q8_0", 12250, 2048, True),
    ("gate_up", "iq4_xs", 17408, 5120, True), ("gate_up", "iq4_xs", 12500, 7168, False),
    ("gate_up", "iq4_xs", 5120, 17408, False), ("gate_up", "iq4_xs", 8192, 17408, True),
    ("gate_up", "q4_k", 8704, 7168, False), ("gate_up", "q4_k", 8704, 6912, True), ("gate_up", "q4_k", 17408, 5120, True),
    ("gate_up", "iq4_nl", 8704, 7168, False), ("gate_up", "iq4_nl", 17408, 5120, True), ("gate_up", "q5_k", 8704, 7168, True)])
def test_superblock_matvec_lines(fake, call, fmt, M, K, sb):
    (r,) = fakehip.run(fake, [[call, fmt, M, K]])
    assert [v["name"] for v in r["launches"]] == ["gemv_sb_kernel" if sb else "gemv_kernel"]


# IQ2_XXS: tall matrices of short rows too (248320 x 1024 33.0 us on gemv_kernel, 26.6).
@pytest.mark.parametrize("M,K,sb", [(248320, 1024, True), (120000, 2048, True), (60000, 512, True), (60000, 2048, False),
                                    (6144, 2048, False), (17408, 5120, True), (30000, 256, False)])
def test_superblock_matvec_iq2_xxs(fake, M, K, sb):
    (r,) = fakehip.run(fake, [["gemv", "iq2_xxs", M, K]])
    assert [v["name"] for v in r["launches"]] == ["gemv_sb_kernel" if sb else "gemv_kernel"]


# ------------------------------------------------------------------ several columns
# Many short rows: four wavefronts without a split, in the instance whose
# registers are those of four (a larger workgroup's cost F32, N = 2, a fifth).
@pytest.mark.parametrize("fmt,M,K,N", [("f32", 151936, 2048, 2), ("q8_0", 248320, 1024, 2), ("q8_0", 6144, 2048, 2),
                                       ("q2_0", 4096, 2048, 2), ("q6_k", 10240, 2048, 5), ("q4_0", 4096, 1024, 3),
                                       ("f16", 12288, 2048, 3), ("q2_0", 6144, 2048, 5)])
def test_columns_of_many_short_rows(fake, fmt, M, K, N):
    (r,) = fakehip.run(fake, [["gemm", fmt, M, K, N]])
    (v,) = r["launches"]
    f, nc, rows, depth, split, silu, most = v["args"]
    assert (v["name"], nc, v["block"], split, most) == ("gemv_kernel", N, 256, 1, 4)


# ------------------------------------------------------------------ RMSNorm
# Threads a row: short rows past one a CU keep 256 (a head's norm over 128
# values took 25.1 us for 16384 rows on 512 threads, 14.7 on 256).
@pytest.mark.parametrize("n,rows,add,threads", [(128, 16384, 0, 256), (1024, 300, 0, 256), (1536, 300, 0, 512),
                                                (2048, 1023, 0, 512), (2048, 1024, 0, 256), (2052, 2000, 0, 512),
                                                (5120, 512, 1, 256), (5120, 255, 0, 1024), (128, 1, 1, 1024)])
def test_norm_threads(fake, n, rows, add, threads):
    (r,) = fakehip.run(fake, [["norm", n, rows, add]])
    (v,) = r["launches"]
    assert (v["block"], v["grid"]) == (threads, [rows, 1, 1]) and v["args"][:2] == [add, threads]

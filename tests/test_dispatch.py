"""Which kernels the calls run and with which K splits, on the CPU (tests/launches.py)."""
import pytest

from csed499ii_amd import marlin
from tests.launches import build_fake, launches

COUNTERS = 64 * 1024 // 4  # arrival counters of a stream's split-K scratch


@pytest.fixture(scope="module")
def fake(built_lib, tmp_path_factory):
    return build_fake(tmp_path_factory.mktemp("fake_hip"))


@pytest.mark.parametrize("op,M,K,N", [("2_4", 192, 1024, 524288), ("w3", 17, 1 << 17, 576 << 10), ("2_4", 33, 16384, 4096),
                                      ("dense", 2048, 1024, 16384), ("dense", 1, 16384, 1040 << 10)])
@pytest.mark.parametrize("sms", [256, 1 << 15, 1 << 20, (1 << 31) - 1])
def test_splits_within_counters(fake, op, M, K, N, sms):
    """Any number of compute units a caller names: a call whose K is split has an arrival
    counter for every tile."""
    for x in launches(fake, [[[op, M, K, N, 128, sms]]]):
        assert x["splits"] <= 1 or x["grid"] // x["splits"] <= COUNTERS, x


@pytest.mark.parametrize("rows", ["64", "96", "128"])
def test_forced_splits_within_counters(fake, rows):
    """Forced K splits of the large-M kernel, on every tile height."""
    env = {"MARLIN_HIP_PREFILL_SPLITS": "2", "MARLIN_HIP_PREFILL_ROWS": rows}
    (x,) = launches(fake, [[["2_4", 4096, 2048, 131072, 128, 256]]], env)
    assert x["kernel"] == "sm24_prefill_kernel"
    assert x["splits"] <= 1 or x["grid"] // x["splits"] <= COUNTERS, x


@pytest.mark.parametrize("op,env,kernel", [
    ("2_4", {"MARLIN_HIP_PREFILL_MIN_M": "48"}, "sm24_prefill_kernel"),
    ("w3", {"MARLIN_HIP_PREFILL_MIN_M": "48"}, "sm24_prefill_kernel"),
    ("dense", {"MARLIN_HIP_DENSE_PREFILL_MIN_M": "48"}, "marlin_dense_prefill_kernel"),
])
def test_prefill_min_m_switch(fake, op, env, kernel):
    """The smallest batch of the large-M kernels, where it is set: every call they can take
    from it on, none below it."""
    for M, K, N in ((48, 4096, 4096), (64, 2048, 1024), (160, 4096, 12288), (1000, 1024, 2048)):
        assert launches(fake, [[[op, M, K, N, 128, 256]]], env)[-1]["kernel"] == kernel, (M, K, N)
        assert launches(fake, [[[op, 47, K, N, 128, 256]]], env)[-1]["kernel"] != kernel, (47, K, N)


@pytest.mark.parametrize("chunks,block", [("4", 256), ("8", 512)])
def test_prefill_chunks_switch(fake, chunks, block):
    """4: every large-M call on the narrow tile of four waves; 8: on 512-column tiles of
    eight, also at the batches of the two-group tiles."""
    for M, K, N in ((80, 4096, 22016), (131, 4096, 22016), (192, 8192, 16384), (1000, 4096, 8192)):
        (x,) = launches(fake, [[["2_4", M, K, N, 128, 256]]], {"MARLIN_HIP_PREFILL_CHUNKS": chunks})
        assert x["kernel"] == "sm24_prefill_kernel" and x["block"] == block, (M, K, N, x)
        assert f"ELi{chunks}ELi1EE" in x["symbol"], x  # chunks, one k-group


@pytest.mark.parametrize("K", [128, 256, 384])
def test_dense_short_k(fake, K):
    """Dense calls of fewer than eight k-steps run the faster of the two kernels, as longer
    K do: the large-M kernel on much work, the mid-batch one on little."""
    for M, N, kernel in ((2048, 57344, "marlin_dense_prefill_kernel"), (512, 22016, "marlin_dense_prefill_kernel"),
                         (131, 57344, "marlin_dense_prefill_kernel"), (2048, 4096, "marlin_dense_prefill_kernel"),
                         (512, 4096, "marlin_dense_mid_kernel"), (131, 11008, "marlin_dense_mid_kernel"),
                         (2048, 1024, "marlin_dense_mid_kernel"), (64, 57344, "marlin_dense_mid_kernel")):
        assert [x["kernel"] for x in launches(fake, [[["dense", M, K, N, 128, 256]]])] == [kernel], (M, K, N)


def test_dense_prefill_splits_switch(fake):
    """The switch forces the large-M kernel's K splits (at most one per eight k-steps, one
    arrival counter per tile) and leaves the choice of kernel alone."""
    calls = [["dense", M, K, N, 128, 256] for M in (65, 131, 512, 2048, 4096)
             for K, N in ((4096, 4096), (11008, 4096), (4096, 22016), (256, 11008), (1024, 1 << 20))]
    free = launches(fake, [calls])
    forced = launches(fake, [calls], {"MARLIN_HIP_DENSE_PREFILL_SPLITS": "3"})
    assert [x["kernel"] for x in free] == [x["kernel"] for x in forced]
    for (_, M, K, N, *_), x in zip(calls, forced):
        if x["kernel"] == "marlin_dense_prefill_kernel":
            tiles = -(-N // 512) * -(-M // 128)
            s = min(3, max(1, K // 512)) if tiles <= COUNTERS else 1
            assert x["grid"] == tiles * s, (M, K, N, x)


@pytest.mark.parametrize("splits", [1, 3, 16])
def test_dense_splits_switch(fake, splits):
    """The switch forces the K splits of the dense decode- and mid-batch kernel (at most
    one per 256 of K, one arrival counter per tile) and leaves the choice of kernel alone."""
    calls = [["dense", M, K, N, 128, 256] for M in (1, 16, 64, 131, 2048)
             for K, N in ((4096, 4096), (11008, 4096), (1152, 22016), (256, 11008), (8192, 1 << 21))]
    free = launches(fake, [calls])
    forced = launches(fake, [calls], {"MARLIN_HIP_DENSE_SPLITS": str(splits)})
    assert [x["kernel"] for x in free] == [x["kernel"] for x in forced]
    for (_, M, K, N, *_), x in zip(calls, forced):
        if x["kernel"] == "marlin_dense_mid_kernel":
            assert x["splits"] in (min(splits, K // 256), 1)
            assert x["splits"] == 1 or x["grid"] // x["splits"] <= COUNTERS, (M, K, N, x)
            assert x["splits"] > 1 or splits == 1 or K == 256 or N > 1 << 20, (M, K, N, x)


#: kernels of the plan query, by the name of the kernel that runs
KERNELS = {"sm24_decode_kernel": "decode", "sm24_decode_dma_kernel": "decode_dma", "sm24_mid_kernel": "mid",
           "sm24_prefill_kernel": "large_m", "sm24_gemm_kernel": "general"}


@pytest.mark.parametrize("op", ["2_4", "noalloc"])
@pytest.mark.parametrize("K,N", [(4096, 4096), (4096, 22016), (8192, 57344), (28672, 8192), (4096, 768), (192, 4096),
                                 (8192, 1024), (28672, 1024), (1024, 12288)])
def test_plan_names_what_runs(fake, op, K, N):
    """The plan query against the launches themselves: kernel, workgroups, threads and
    launches of calls of 1 to 4096 rows."""
    g = -1 if K % 128 else 128
    calls = [[op, M, K, N, g, 256] for M in (1, 4, 8, 16, 17, 24, 32, 33, 64, 65, 96, 97, 131, 192, 193, 300, 640,
                                             1024, 1025, 4096) if M > 16 or K % 128 == 0]
    ls = launches(fake, [calls])
    for _, M, *_ in calls:
        p = marlin.plan_2_4(M, K, N, g, sms=256, noalloc=op == "noalloc")
        mine, ls = ls[:p["launches"]], ls[p["launches"]:]
        assert KERNELS[mine[0]["kernel"]] == p["kernel"], (M, p, mine)
        assert len(mine) == 1 or {KERNELS[x["kernel"]] for x in mine} <= {"decode", "decode_dma"}, (M, mine)
        assert (mine[0]["grid"], mine[0]["block"]) == (p["workgroups"], p["threads"]), (M, p, mine)
    assert not ls

"""Launches of host threads that share a stream, on the CPU (tests/launches.py).  Calls of
one stream share its split-K scratch and its staging buffer; ctypes releases the GIL, so
another thread's launches may reach the stream between two launches of one call."""
import pytest

from tests.launches import build_fake, launches


@pytest.fixture(scope="module")
def fake(built_lib, tmp_path_factory):
    return build_fake(tmp_path_factory.mktemp("fake_hip"))


def assert_calls_whole(fake, call, per_call):
    """Two threads, four times the same call each: the launches of a call that hand data
    over in the stream's buffers follow each other."""
    ls = launches(fake, [[call] * 4] * 2)
    assert len(ls) == 8 * per_call
    for i in range(0, len(ls), per_call):
        assert len({x["thread"] for x in ls[i:i + per_call]}) == 1, [(x["kernel"], x["thread"]) for x in ls]


@pytest.mark.parametrize("op", ["2_4", "w3", "meta3"])
@pytest.mark.parametrize("M,K,N", [(33, 4096, 4096), (64, 4096, 4096), (64, 11008, 4096), (48, 28672, 7936)])
def test_split_k_hand_off_in_one_launch(fake, op, M, K, N):
    """Mid-batch calls whose column tiles cover under half of the compute units: the sums
    of their K splits are handed over inside the launch."""
    call = [op, M, K, N, 128, 256]
    assert [x["kernel"] for x in launches(fake, [[call]])] == ["sm24_mid_kernel"]
    assert_calls_whole(fake, call, 1)


@pytest.mark.parametrize("op,M,K,N,kernels", [
    ("w3", 512, 4096, 4096, ["w3_to_w4_kernel", "sm24_prefill_kernel"]),
    ("meta3", 131, 4096, 22016, ["meta3_unpack_kernel", "sm24_prefill_kernel"]),
    ("native", 24, 4096, 4096, ["native_unpack_values_kernel", "native_unpack_meta_kernel", "sm24_mid_kernel"]),
    ("native", 600, 4096, 4096, ["native_unpack_values_kernel", "native_unpack_meta_kernel", "sm24_prefill_kernel"]),
])
def test_staged_operands(fake, op, M, K, N, kernels):
    """Operands expanded into the stream's staging buffer: the expansion and the kernel that
    reads it follow each other."""
    call = [op, M, K, N, 128, 256]
    assert [x["kernel"] for x in launches(fake, [[call]])] == kernels
    assert_calls_whole(fake, call, len(kernels))

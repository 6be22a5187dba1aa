"""CPU: the quantiser's fast division path (FMA-based, shared header aiter_amd/csrc/fp8bs_math.h)
compiled for the host and compared exhaustively with IEEE division; also the header's software
e4m3fn conversion against the oracle's.  Host logic only, no GPU."""

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "host_math", "fastpath_check.cpp")
ORACLE_C = os.path.join(os.path.dirname(HERE), "oracle", "fp8bs_oracle.c")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("fastpath") / "fastpath_check")
    subprocess.check_call(
        ["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-o", exe, SRC, "-x", "c", ORACLE_C, "-lm"]
    )
    return exe


@pytest.mark.parametrize("mode", ["bf16", "fp16", "scale", "mean", "cvt"])
def test_fast_division_is_ieee_exact(checker, mode):
    out = subprocess.run([checker, mode], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("OK")


def test_capture_lane_bookkeeping(tmp_path):
    """Streams of one capture sequence get scratch lanes of their own (two streams, two pointers),
    a stream keeps its lane, a new sequence starts at lane 0: aiter_amd/csrc/capture_lanes.h on the host."""
    exe = str(tmp_path / "capture_lanes_check")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "host_math", "capture_lanes_check.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.stdout + out.stderr


def test_k_ranges_of_a_plan_do_not_depend_on_the_kernel_that_carries_them_out():
    # two ranges of K are two sums: the choice is the same on both sides of any number of rows, and 256 x 128 tiles, which
    # take the ranges one after the other, do not turn them into one
    from aiter_amd import _ffi

    for n, k in ((4096, 7168), (3504, 7040)):
        assert {_ffi.gemm_choice(m, n, k) for m in range(1793, 2049, 15)} == {"prefill_256x256:s=2"}
    for m, n, k in ((256, 24576, 7168), (300, 16384, 7168), (700, 7168, 7168), (1500, 4096, 7168), (2048, 2304, 7168)):
        assert _ffi.gemm_choice(m, n, k).endswith(":s=2")


def test_expert_layer_rule_counts_rows_per_routed_expert(tmp_path):
    """An expert-parallel rank holds a part of the experts its tokens are routed to: aiter_amd/csrc/moe_rules.h on the host."""
    exe = str(tmp_path / "moe_rules_check")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "host_math", "moe_rules_check.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.stdout + out.stderr


def test_kernel_choice_query_on_the_headline_shapes():
    """The shape rule that stands in for the reference's tuned-table lookup (get_CKGEMM_config,
    aiter/ops/gemm_op_a8w8.py:448-490) can be asked without a GPU."""
    import aiter_amd

    names = set(aiter_amd.gemm_kernel_names())
    for m in (1, 16, 64):
        for n, k in ((7168, 2048), (24576, 1536), (2112, 7168)):
            # the weight-streaming kernel up to 16 rows, and everywhere on the shape whose N / 16 row tiles
            # with one K step per wave cover the chip; the mid_* tilings where they are modelled (and
            # measured) faster: at 64 rows on the other two shapes
            want = "decode_stream" if m <= 16 or (n, k) == (7168, 2048) else "mid_"
            assert aiter_amd.get_CKGEMM_config(m, n, k)["kernelName"].startswith(want)
    assert aiter_amd.get_CKGEMM_config(8192, 36864, 7168)["kernelName"] == "prefill_256x256"
    cfg5 = aiter_amd.get_CKGEMM_config(2048, 4096, 7168)  # 128 tiles: two K ranges per tile
    assert cfg5["kernelName"] == "prefill_256x256:s=2" and cfg5["kRanges"] == 2
    cfg = aiter_amd.get_CKGEMM_config(128, 4096, 7168)  # few tiles, long K: K is split
    assert cfg["kernelName"].startswith("mid_") and cfg["kRanges"] > 1 and cfg["libtype"] == "hip"
    for m, n, k in ((65, 512, 128), (300, 1000, 384), (4096, 2112, 7168), (100000, 128, 128)):
        cfg = aiter_amd.get_CKGEMM_config(m, n, k, isBpreshuffled=(n % 16 == 0))
        assert cfg["kernelName"].split(":")[0] in names
    import pytest

    with pytest.raises(RuntimeError, match="multiple of 128"):
        aiter_amd.get_CKGEMM_config(4, 512, 100)

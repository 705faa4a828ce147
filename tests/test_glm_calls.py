"""The evaluation calls' host side on a stand-in HIP runtime (no GPU): what
they return when stores reach the host late and out of order, what they leave
queued, and what they do when memory is refused (tests/cpp/glm_calls_check.cpp
says how)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("cpp") / "glm_calls_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROCM, "include"), "-o", exe,
                    os.path.join(HERE, "cpp", "glm_calls_check.cpp")], check=True)

    def run(scenario):
        out = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=100)
        assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr

    return run


@pytest.mark.parametrize("scenario", ["single_fresh", "single_slow"])
def test_single_evaluations(check, scenario):
    """Every value is this call's own: also those that arrive after the log
    density and the status, and those of a launch that takes longer than the
    host watches the output; a launch that stores nothing is an error."""
    check(scenario)


def test_failed_calls_leave_nothing_queued(check):
    """A call whose launch is refused waits for the copies it has queued: they
    read the caller's points or buffers that the next call fills."""
    check("failed_calls_drain")


def test_batches_where_memory_is_refused(check):
    """FP64 batches run in smaller slabs, down to chain by chain in the
    context's own buffers, and every batch runs without a pinned buffer; the
    refused allocation's error is not reported by a later launch."""
    check("refused_memory")


def test_middle_batches_keep_no_host_memory(check):
    """Batches whose results go through pageable memory (64 KB to 1 MB) give
    it back with the call."""
    check("nothing_kept")


def test_small_batches_pin_no_memory(check):
    """Batches below 64 KB go through pinned memory that the context has from
    its creation."""
    check("small_batches_pin_nothing")


def test_batches_report_domain_errors(check):
    """-inf for every chain with a domain error, the last one's message, the
    gradient of a chain at a non-finite point left alone; on one thread and on
    several."""
    check("batch_errors")


def test_which_batches_share_tiles(check):
    """The several-chains FP64 pass is taken where it is the faster one."""
    check("chains_rule")


def test_row_splits_that_are_timed(check):
    check("split_targets")

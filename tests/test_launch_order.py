"""How the library's launches follow each other, on a CPU: its host code bound to a stand-in for the HIP
runtime (launch_order_check.cpp) that notes what every operation waits for."""

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
LIB = os.path.join(REPO, "qwen0.6b_amd", "libqwen_megakernel.so")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not os.path.exists(LIB):
        pytest.skip("library not built (run __graft_entry__.build())")
    exe = str(tmp_path_factory.mktemp("launch_order") / "launch_order_check")
    # (the rocm headers the library is built with; no HIP runtime is linked)
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", "-w", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{os.path.join(REPO, 'include')}", os.path.join(HERE, "launch_order_check.cpp"), "-o", exe,
                    "-ldl", "-lpthread"], check=True)

    def run(scenario):
        r = subprocess.run([exe, LIB, scenario], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]

    return run


@pytest.mark.parametrize("scenario", ["eager", "threads"])
def test_calls_follow_each_other(check, scenario):
    """Every entry point and every build of the kernels, on several streams and from two threads: each
    kernel follows the one before it, and every grid was checked to be resident at once."""
    check(scenario)


def test_captured_calls_are_ordered(check):
    """A replay of captured calls waits for the eager launch before it and is waited for by the next, on
    whatever streams, the first time and later."""
    check("captured")


def test_streams_with_a_cu_mask(check):
    """Calls on a stream that is restricted to some CUs: their grids, which need the whole chip, do not go
    to its queue, and they keep their place in the order."""
    check("masked")


def test_stream_whose_capture_state_is_unknown(check):
    """Where the runtime cannot say whether a stream is captured, nothing is sent to it."""
    check("unknown")


@pytest.mark.parametrize("build", ["4fast", "6traced", "7sampled", "8dsampled", "8tsampled", "8isolated", "qwen_sample_kernel",
                                   "mid_kernelILi16E", "mid_kernelILi64E", "mid_kernelILi128E", "mid_kernelILi256E",
                                   "mid_kernelILi512E", "mid_kernelILi1024E", "19qwen_prefill_kernel"])
def test_a_build_that_does_not_fit_is_refused(check, build):
    """A grid of workgroups that wait for each other must be resident at once: where any build would not
    be, every call is refused and nothing is launched."""
    check("fits:" + build)

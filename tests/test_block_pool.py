"""The pool of device blocks, on the CPU over a counted memory of a fixed size: what it keeps,
its bounds, and that everything kept goes back before an allocation is refused."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_block_pool(tmp_path):
    exe = str(tmp_path / "block_pool_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-I", os.path.join(ROOT, "gpujoin_amd", "csrc"),
                    os.path.join(ROOT, "tests", "block_pool_check.cpp"), "-o", exe], check=True)
    assert subprocess.run([exe], timeout=60).returncode == 0  # the failing line otherwise


def test_every_allocation_goes_through_the_pool():
    # hipMalloc on its own would refuse memory that the pool holds idle
    src = os.path.join(ROOT, "gpujoin_amd", "csrc")
    calls = [(f, line.strip()) for f in sorted(os.listdir(src)) for line in open(os.path.join(src, f))
             if "hipMalloc(" in line and not line.lstrip().startswith("//")]
    assert [f for f, _ in calls] == ["runtime.hip"] * 2, calls  # the pool's own, and the wait's token


def test_release_cached_is_exported(gj):
    assert hasattr(gj._lib.load(), "gj_release_cached") and callable(gj.release_cached)

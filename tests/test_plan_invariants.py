"""Small-batch planner invariants over 60000 random shapes (host code only,
no GPU): built from tests/plan_invariants.hip with hipcc into a temporary
directory and run."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def _hipcc():
    path = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
    return path if os.path.exists(path) else shutil.which("hipcc")


@pytest.mark.skipif(_hipcc() is None, reason="hipcc not available")
def test_small_batch_plan_invariants(tmp_path):
    exe = str(tmp_path / "plan_invariants")
    build = subprocess.run([_hipcc(), "-O1", "-std=c++17", "--offload-arch=gfx950",
                            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                            os.path.join(HERE, "plan_invariants.hip"), "-o", exe],
                           capture_output=True, text=True, timeout=600)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout[-2000:]


@pytest.mark.skipif(_hipcc() is None, reason="hipcc not available")
def test_pair_split(tmp_path):
    """The row-pair kernels' pair ranges (host-computed split, multiply-shift
    division on the device) against exact 64-bit division."""
    exe = str(tmp_path / "pair_split_check")
    build = subprocess.run([_hipcc(), "-O1", "-std=c++17", "--offload-arch=gfx950",
                            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                            os.path.join(HERE, "pair_split_check.hip"), "-o", exe],
                           capture_output=True, text=True, timeout=900)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout[-2000:]


@pytest.mark.skipif(_hipcc() is None, reason="hipcc not available")
def test_prefill_gemm_split(tmp_path):
    """The prefill GEMM's work split: runs, pieces and the second launch that
    adds them, over 20000 random calls; and the calls that the GPU tests make
    for the sake of their pieces are cut."""
    from tests.test_gpu_gemm_sk import CUT_FUSED, CUT_GRAPH, CUT_STREAMS, CUT_SWIGLU
    calls = [(mt, M, K, 0, *Ns) for mt, M, Ns, K in CUT_FUSED]
    calls += [(mt, M, K, 1, N) for mt, M, N, K in CUT_SWIGLU + CUT_GRAPH[:1]]
    calls += [(mt, M, K, 0, N) for mt, M, N, K in CUT_GRAPH[1:] + CUT_STREAMS]
    exe = str(tmp_path / "sk_plan_check")
    build = subprocess.run([_hipcc(), "-O1", "-std=c++17", "--offload-arch=gfx950",
                            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                            os.path.join(HERE, "sk_plan_check.hip"), "-o", exe],
                           capture_output=True, text=True, timeout=900)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([exe, *(",".join(map(str, c)) for c in calls)], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout[-2000:]


@pytest.mark.skipif(_hipcc() is None, reason="hipcc not available")
def test_scratch_owners(tmp_path):
    """Who owns the split-K slots and the prefill GEMM's areas."""
    exe = str(tmp_path / "scratch_check")
    build = subprocess.run([_hipcc(), "-O1", "-std=c++17", "--offload-arch=gfx950",
                            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                            os.path.join(HERE, "scratch_check.hip"), "-o", exe],
                           capture_output=True, text=True, timeout=900)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout[-2000:]


@pytest.mark.skipif(_hipcc() is None, reason="hipcc not available")
def test_prefill_gemm_launch_pairs(tmp_path):
    """The two launches of a cut prefill call, with several host threads on a
    stream."""
    exe = str(tmp_path / "sk_enqueue_check")
    build = subprocess.run([_hipcc(), "-O1", "-std=c++17", "--offload-arch=gfx950",
                            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                            os.path.join(HERE, "sk_enqueue_check.hip"), "-o", exe, "-pthread"],
                           capture_output=True, text=True, timeout=900)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout[-2000:]

"""Host code and single device functions of the library built with g++ against
tests/hip_model (threads for lanes, a thread per stream)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def _run(tmp_path, source, *flags):
    exe = str(tmp_path / "model")
    subprocess.run(["g++", "-std=c++20", "-O1", "-w", "-pthread", "-I", os.path.join(HERE, "hip_model"), *flags,
                    os.path.join(HERE, source), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_residual_fold_is_the_same_for_a_whole_block(tmp_path):
    """The kernel after the residual's update (rr_fold): one answer per block,
    whenever its waves start beside the block that ends the solve, and nothing
    counted once the solve has ended."""
    _run(tmp_path, "rr_fold_model.cpp")


def test_host_transfers(tmp_path):
    """Host arrays through the ring of pinned chunks (t3x_stage.hip)."""
    _run(tmp_path, "stage_model.cpp")

"""The streamer's SVD workspace where memory runs out, on the CPU."""
import os
import subprocess

from conftest import ROOT


def test_workspace_without_page_locked_memory(tmp_path):
    exe = tmp_path / "svd_workspace"
    # the file's other device calls stay unresolved: nothing here reaches them
    subprocess.run(["gcc", "-std=c11", "-O1", "-g", "-w", os.path.join(ROOT, "tests", "c_caller", "svd_workspace.c"),
                    "-o", str(exe), "-Wl,--unresolved-symbols=ignore-all", "-lm", "-lpthread"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr

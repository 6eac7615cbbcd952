"""csrc/build.sh with stand-ins for the compilers (each writes the file behind its -o): what is built where torch is not there."""
import os
import shutil
import stat
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("torch", [False, True])
@pytest.mark.parametrize("torch_ops_compile", [True, False])
def test_the_c_library_builds_without_torch(tmp_path, torch, torch_ops_compile):
    """The C library, its tests and the example program come out without Python or torch; where torch is there, a _torch_ops.so that does
    not compile fails the build."""
    csrc = tmp_path / "async-gpu_amd" / "csrc"
    csrc.mkdir(parents=True)
    (tmp_path / "tests" / "cpp").mkdir(parents=True)
    (tmp_path / "async-gpu_amd" / "examples").mkdir()
    shutil.copy(os.path.join(ROOT, "async-gpu_amd", "csrc", "build.sh"), csrc)
    for name in ("decode_xcd.hip", "gpt2_model.hip", "quantize_host.cpp", "torch_ops.cpp"):
        (csrc / name).write_text("")
    tools = tmp_path / "tools"
    tools.mkdir()

    def tool(name, text):
        (tools / name).write_text("#!/bin/bash\n" + text)
        (tools / name).chmod(0o755 | stat.S_IXUSR)

    fails = "" if torch_ops_compile else 'case "$*" in *torch_ops.cpp*) exit 1;; esac\n'
    compiler = fails + 'while [ $# -gt 0 ]; do if [ "$1" = -o ]; then echo built > "$2"; fi; shift; done\n'
    tool("hipcc", compiler)
    tool("g++", compiler)
    tool("python3", "echo /nowhere/torch /nowhere/include 1\n" if torch else "echo no torch here >&2; exit 1\n")
    env = dict(os.environ, PATH=f"{tools}:{os.environ['PATH']}", HIPCC=str(tools / "hipcc"))
    r = subprocess.run(["bash", str(csrc / "build.sh")], env=env, capture_output=True, text=True, timeout=60)
    package = tmp_path / "async-gpu_amd"
    assert (r.returncode == 0) == (torch_ops_compile or not torch), r.stdout + r.stderr
    for built in (package / "libagpu_hip.so", package / "libagpu_hip_trace.so", package / "examples" / "gpt2_inference",
                  tmp_path / "tests" / "cpp" / "test_nn", tmp_path / "tests" / "cpp" / "test_gpu_array_host"):
        assert built.exists(), built
    assert (package / "_torch_ops.so").exists() == (torch and torch_ops_compile)
    assert torch or "_torch_ops.so" in r.stdout

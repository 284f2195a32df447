"""kernels/compile.sh with stand-ins for the compilers: what it builds where PyTorch is missing, and what a failed compile leaves."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

COMPILER = """#!/usr/bin/env bash
# writes the file named behind -o after $DELAY seconds, or fails for the source named in $FAIL
echo start >> "$LOG"
out=; prev=
for a in "$@"; do [ "$prev" = -o ] && out="$a"; prev="$a"; done
case " $* " in *"/${FAIL:-nothing} "*) echo failed >> "$LOG"; exit 1;; esac
sleep "${DELAY:-0}"
: > "$out"
echo end >> "$LOG"
"""
PYTHON = {"torch": "#!/usr/bin/env bash\necho /nowhere\n", "no torch": "#!/usr/bin/env bash\necho \"No module named 'torch'\" >&2\nexit 1\n", "none": None}


def _build(tmp_path, python, **env):
    tree, tools = tmp_path / "tree", tmp_path / "tools"
    for d in (tree / "kernels", tree / "ternainfer_amd" / "csrc", tools):
        d.mkdir(parents=True)
    shutil.copy(os.path.join(ROOT, "kernels", "compile.sh"), tree / "kernels")
    scripts = {"hipcc": COMPILER, "g++": COMPILER, "python3": PYTHON[python]}
    for name, text in scripts.items():
        if text is not None:
            (tools / name).write_text(text)
            (tools / name).chmod(0o755)
    for name in ("bash", "dirname", "mkdir", "grep", "sleep"):
        (tools / name).symlink_to(shutil.which(name))
    log = tmp_path / "log"
    log.write_text("")
    said = tmp_path / "said"                      # (a file: a pipe would wait for whatever the script leaves running)
    with open(said, "w") as f:
        code = subprocess.run(["bash", str(tree / "kernels" / "compile.sh")], env={"PATH": str(tools), "LOG": str(log), **env}, stdout=f, stderr=f, timeout=60).returncode
    return code, said.read_text(), tree, log.read_text().split()


@pytest.mark.parametrize("python", sorted(PYTHON))
def test_library_is_built_without_pytorch(tmp_path, python):
    code, said, tree, log = _build(tmp_path, python)
    assert code == 0, said
    assert (tree / "kernels" / "libternaspmm.so").exists()
    assert (tree / "ternainfer_amd" / "_native.so").exists() == (python == "torch")
    assert ("no PyTorch" in said) == (python != "torch")
    assert log.count("start") == log.count("end")


@pytest.mark.parametrize("source,library", [("ternaspmm.hip", False), ("py_native.cpp", True)])
def test_a_failed_compile_fails_the_build_and_leaves_none_running(tmp_path, source, library):
    code, _, tree, log = _build(tmp_path, "torch", FAIL=source, DELAY="0.3")
    assert code != 0
    assert log.count("failed") == 1 and log.count("start") == log.count("end") + 1
    assert (tree / "kernels" / "libternaspmm.so").exists() == library

"""When make builds the native part of the Python binding again: it is tied to the PyTorch that it was built against."""
import os
import shutil
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_another_pytorch_builds_the_native_part_again(tmp_path):
    root, tools, counted = tmp_path / "pkg", tmp_path / "tools", tmp_path / "builds"
    for d in (root / "csrc", tmp_path / "include", tools):
        d.mkdir(parents=True)
    shutil.copy(os.path.join(REPO, "flash-attn-rtx5060_amd", "Makefile"), root)
    for f in (root / "csrc" / "fa_torch.cpp", tmp_path / "include" / "fa_fwd.h", tmp_path / "include" / "fa_bwd.h", counted):
        f.write_text("")
    # stand-ins: an interpreter that says which PyTorch it has, a compiler that leaves its output and counts
    (tools / "python").write_text("#!/bin/sh\ncat %s\n" % (tools / "version"))
    (tools / "c++").write_text('#!/bin/sh\necho x >> %s\nwhile [ "$1" != -o ]; do shift; done\ntouch "$2"\n' % counted)
    for f in ("python", "c++"):
        (tools / f).chmod(0o755)

    def builds(version):
        (tools / "version").write_text(version)
        target = os.path.realpath(root / "lib" / "_fa_torch.so")
        subprocess.run(["make", "-s", "-C", str(root), "PYTHON=%s" % (tools / "python"), "CXX=%s" % (tools / "c++"), target], check=True)
        return len(counted.read_text().split())
    assert [builds("1"), builds("1"), builds("2"), builds("2"), builds("1")] == [1, 1, 2, 2, 3]

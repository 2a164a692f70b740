"""The build needs nothing of tests/: both libraries come from the package's
own sources, so they build beside any state of the tests."""
import shutil
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_hostcheck_builds_without_the_tests(tmp_path):
    shutil.copytree(ROOT / "lattice_amd", tmp_path / "lattice_amd",
                    ignore=shutil.ignore_patterns("_build", "__pycache__", "*.so"))
    shutil.copytree(ROOT / "include", tmp_path / "include")
    subprocess.run([sys.executable, "-c",
                    "from lattice_amd import build as b; assert b.build_hostcheck().exists()"],
                   cwd=tmp_path, check=True)


def test_the_product_is_built_before_the_check_library(monkeypatch):
    from lattice_amd import build as b
    order = []
    monkeypatch.setattr(b, "build_kcmm", lambda jobs=8: order.append("kcmm"))
    monkeypatch.setattr(b, "build_hostcheck", lambda: order.append("hostcheck"))
    b.build_all()
    assert order == ["kcmm", "hostcheck"]

"""bench.py reports a committed profile's figures only for the kernels that it was taken
from: their sources' digest, which comments and spaces do not change."""
import json
import os
import shutil

import pytest

import bench

CSRC = os.path.join("jaxrenderer_amd", "csrc")


@pytest.fixture
def tree(tmp_path, monkeypatch):
    shutil.copytree(os.path.join(bench.ROOT, CSRC), tmp_path / CSRC,
                    ignore=shutil.ignore_patterns("*.o"))
    (tmp_path / "profiles").mkdir()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    return tmp_path


def profile(tree, **kw):
    (tree / "profiles" / "config3_traffic.json").write_text(
        json.dumps({"kernels": {"main.raster": {"hbm_bytes": 1}}, **kw}))


def test_a_profile_of_other_kernels_is_not_reported(tree):
    assert bench.profiled() == {}  # none there
    profile(tree)
    assert bench.profiled() == {}  # of kernels that it does not name
    profile(tree, source=bench.forward_source())
    assert bench.profiled()["kernels"]["main.raster"]["hbm_bytes"] == 1
    path = tree / CSRC / "jr_forward.hip"
    text = path.read_text()
    path.write_text("// another comment\n/* and\n one more */" + text.replace("\n", "\n\n"))
    assert bench.profiled() != {}
    path.write_text(text.replace("kTaggedPixels = 1 << 20", "kTaggedPixels = 1 << 21"))
    assert bench.profiled() == {}

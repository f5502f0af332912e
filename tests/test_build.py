"""What the incremental build compiles again."""
import os
import shutil

from daceml_amd.csrc import build


def test_objects_are_stale_behind_whatever_their_source_includes(tmp_path, monkeypatch):
    here, include = tmp_path / "daceml_amd" / "csrc", tmp_path / "include"
    objects = here / "build"
    objects.mkdir(parents=True)
    include.mkdir()
    for name in os.listdir(build.HERE):
        if name.endswith((".hip", ".h", ".cpp")):
            shutil.copy(os.path.join(build.HERE, name), here / name)
    shutil.copy(os.path.join(build.HERE, "..", "..", "include", "daceml_hip.h"), include)
    monkeypatch.setattr(build, "HERE", str(here))
    monkeypatch.setattr(build, "OBJ_DIR", str(objects))
    sources = {os.path.splitext(s)[0] + ".o": s for s in build.SOURCES}
    assert all(build._stale(s) for s in sources.values())

    def stale_after(changed):
        for d in (here, include):
            for name in os.listdir(d):
                os.utime(d / name, (1e9, 1e9))
        for name in sources:
            (objects / name).touch()
            os.utime(objects / name, (2e9, 2e9))
        os.utime(changed, (3e9, 3e9))
        return {s for s in sources.values() if build._stale(s)}

    # a source included by another one, a header of a few, one behind other headers, a source
    assert stale_after(here / "conv_dense3_weight.hip") == {"conv_dense3_weight_split.hip"}
    assert stale_after(here / "bf16_split.h") == {"conv_dense3_split.hip", "conv_dense3_weight_split.hip", "gemm_f32_split.hip"}
    assert stale_after(include / "daceml_hip.h") == set(sources.values())
    assert stale_after(here / "attention.hip") == {"attention.hip"}

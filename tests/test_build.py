"""The link commands of the Fortran host layer. Its sources hold subroutines
only, so linked as a program they end in an undefined main."""
import os

import pytest

from opentelemac_amd import build as B


@pytest.mark.parametrize("recipe,name", [("build_shim", "libbiefshim.so"),
                                         ("build_dropin", "libbief_dropin.so")])
def test_fortran_recipes_link_shared_objects(monkeypatch, tmp_path, recipe, name):
    ref = tmp_path / "oracle" / "_ref"
    ref.mkdir(parents=True)
    (ref / "libbief_ref.a").touch()
    commands = []
    monkeypatch.setattr(B, "ROOT", str(tmp_path))
    monkeypatch.setattr(B, "HERE", str(tmp_path))
    monkeypatch.setattr(B, "have_flang", lambda: True)
    monkeypatch.setattr(B, "_run", lambda cmd, cwd=None: commands.append(cmd))
    out = getattr(B, recipe)()
    assert os.path.basename(out) == name
    assert len(commands) == 1
    assert "-shared" in commands[0] and "-fPIC" in commands[0]
    assert commands[0][commands[0].index("-o") + 1] == out

"""Options that only some versions of the compiler know: a unit is built without them, and every other error is an error."""
import os

import pytest

from metaattention_amd import build


def _compiler(tmp_path, monkeypatch, message):
    """A stand-in for hipcc that refuses -amdgpu-mfma-vgpr-form with `message` and writes what it was asked for into the object."""
    path = tmp_path / "hipcc"
    path.write_text(f"""#!/bin/sh
out=
for x in "$@"; do
  [ "$x" = -amdgpu-mfma-vgpr-form ] && {{ echo "{message}" >&2; exit 1; }}
  [ "$last" = -o ] && out="$x"
  last="$x"
done
echo "$@" > "$out"
""")
    path.chmod(0o755)
    monkeypatch.setenv("HIPCC", str(path))
    monkeypatch.setattr(build, "OBJ_DIR", str(tmp_path))


def test_unknown_option(tmp_path, monkeypatch):
    _compiler(tmp_path, monkeypatch, "clang (LLVM option parsing): Unknown command line argument '-amdgpu-mfma-vgpr-form'.")
    unit = next(iter(build.UNIT_FLAGS))
    with pytest.warns(UserWarning, match=unit):
        obj = build._compile(os.path.join(build.CSRC, unit), False)
    assert "-ffast-math" in open(obj).read()


def test_other_errors(tmp_path, monkeypatch):
    _compiler(tmp_path, monkeypatch, "error: no such register")
    with pytest.raises(RuntimeError, match="no such register"):
        build._compile(os.path.join(build.CSRC, next(iter(build.UNIT_FLAGS))), False)

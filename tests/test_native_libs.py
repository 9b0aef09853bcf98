"""The mixer-kernel libraries' staleness check: entry points are called without
types, so a library built from other sources must not be loaded."""

import subprocess

import pytest

from production_stack_amd.ops import native


@pytest.fixture
def tree(tmp_path, monkeypatch):
    """A source folder of one unit and one header, and a builder that makes a
    plain library with whatever key the sources have."""
    src = tmp_path / "csrc"
    src.mkdir()
    (src / "a.hip").write_text("int a;\n")
    (src / "common.h").write_text("// one\n")
    lib = tmp_path / "lib.so"
    builds = []

    def build(group):
        key = native.source_key(group)
        builds.append(key)
        c = tmp_path / "k.c"
        c.write_text('const char mx_build_key[] = "mx_build_key=%s";\n'
                     "int mx_answer(void) { return %d; }\n"
                     % (key, len(builds)))
        subprocess.run(["gcc", "-shared", "-fPIC", str(c), "-o",
                        str(tmp_path / "new.so")], check=True)
        (tmp_path / "new.so").replace(lib)

    monkeypatch.setattr(native, "SRC_DIR", str(src))
    monkeypatch.setattr(native, "GROUPS", {"core": [("a.hip", ["-DX=1"])]})
    monkeypatch.setattr(native, "LIB_PATHS", {"core": str(lib)})
    monkeypatch.setattr(native, "SYMBOL_GROUP", {})
    monkeypatch.setattr(native, "INT_RESULT", {"mx_answer"})
    monkeypatch.setattr(native, "_build_group", build)
    native.source_key.cache_clear()
    yield src, lib, builds
    native.source_key.cache_clear()


def changed():
    native.source_key.cache_clear()  # as a new process


def test_library_of_other_sources_is_built_anew(tree):
    src, lib, builds = tree
    # one from before libraries had a key
    old = lib.with_suffix(".c")
    old.write_text("int mx_answer(void) { return -1; }\n")
    subprocess.run(["gcc", "-shared", "-fPIC", str(old), "-o", str(lib)],
                   check=True)
    assert not native.current("core")
    assert native._Libs().mx_answer() == 1
    assert native.current("core") and len(builds) == 1
    # nothing changed: loaded as it is
    changed()
    native.build()
    assert len(builds) == 1
    # a shared header, a source, a define
    (src / "common.h").write_text("// two\n")
    changed()
    assert not native.current("core")
    native._Libs()._handle("core")
    assert native.current("core") and len(builds) == 2
    (src / "a.hip").write_text("int a, b;\n")
    changed()
    native.build()
    native.GROUPS["core"][0][1].append("-DY")
    changed()
    native.build()
    assert len(builds) == 4 == len(set(builds))


def test_library_without_sources_is_taken_as_it_is(tree):
    src, lib, builds = tree
    native.build()
    (src / "a.hip").unlink()
    changed()
    assert native.current("core")
    assert native._Libs().mx_answer() == 1 and len(builds) == 1

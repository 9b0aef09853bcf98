"""The mixer-kernel libraries' staleness check: entry points are called without
types, so a library built from other sources must not be loaded."""

import subprocess
import sys

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


ENTRY_C = """
#include <stdint.h>
#define W(i, v) r = r * 31 + (int64_t)(v) * (i)
long mx_mixed(const float* p, int a, float x, const void* q, long b, float y,
              int c0, int c1, int c2, int c3, int c4, int c5, int c6, int c7,
              float z, int d0, int d1, int d2, int d3, int d4, int d5, int d6,
              int d7, int e0, int e1, int e2, int e3, int e4, int e5, int e6,
              int e7, float f0, float f1, float f2, float f3, float f4,
              int last, void* stream) {
  int64_t r = 0;
  W(1, p[1]); W(2, a); W(3, x * 4); W(4, q == 0); W(5, b); W(6, y * 4);
  W(7, c0); W(8, c1); W(9, c2); W(10, c3); W(11, c4); W(12, c5); W(13, c6);
  W(14, c7); W(15, z * 4); W(16, d0); W(17, d1); W(18, d2); W(19, d3);
  W(20, d4); W(21, d5); W(22, d6); W(23, d7); W(24, e0); W(25, e1);
  W(26, e2); W(27, e3); W(28, e4); W(29, e5); W(30, e6); W(31, e7);
  W(32, f0 * 4); W(33, f1 * 4); W(34, f2 * 4); W(35, f3 * 4); W(36, f4 * 4);
  W(37, last); W(38, (intptr_t)stream >> 33);
  return r % 1000003;
}
int mx_minus(int a) { return -a; }
void mx_set(float* p, float v) { *p = v; }
"""


@pytest.mark.parametrize("extension", [True, False])
def test_entry_points_get_their_arguments(tmp_path, monkeypatch, extension):
    """Pointers, integers and floats in any order, more than registers hold,
    through the extension and through ctypes."""
    import ctypes

    import torch

    import production_stack_amd

    if extension:
        pytest.importorskip("production_stack_amd._C")
    else:
        monkeypatch.setitem(sys.modules, "production_stack_amd._C", None)
        monkeypatch.delattr(production_stack_amd, "_C", raising=False)
    src, lib = tmp_path / "e.c", tmp_path / "e.so"
    src.write_text(ENTRY_C)
    subprocess.run(["gcc", "-shared", "-fPIC", "-fwrapv", str(src), "-o",
                    str(lib)], check=True)
    h = ctypes.CDLL(str(lib))
    monkeypatch.setattr(native, "LONG_RESULT", {"mx_mixed"})
    monkeypatch.setattr(native, "INT_RESULT", {"mx_minus"})
    mixed, minus, put = (native._entry(getattr(h, n), n)
                         for n in ("mx_mixed", "mx_minus", "mx_set"))
    t = torch.tensor([1.0, 77.0, 3.0])
    args = [t, -5, 0.25, None, 1 << 40, -1.5, 1, 2, 3, 4, 5, 6, 7, 8, 2.25, 9,
            10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20, 21, 22, 23, True, 0.5,
            0.75, 1.0, 1.25, 7.5, -3, 0x7f1234567000]
    terms = [77, -5, 1, 1, 1 << 40, -6, 1, 2, 3, 4, 5, 6, 7, 8, 9, 9, 10, 11,
             12, 13, 14, 15, 16, 17, 18, 19, 20, 21, 22, 23, 1, 2, 3, 4, 5, 30,
             -3, 0x7f1234567000 >> 33]
    r = 0
    for i, v in enumerate(terms):
        r = r * 31 + v * (i + 1)
    r = (r + (1 << 63)) % (1 << 64) - (1 << 63)       # as 64 bits have it
    assert mixed(*args) == (abs(r) % 1000003) * (1 if r >= 0 else -1)
    assert minus(7) == -7 and minus(-7) == 7
    assert put(t[2:], 5.5) is None and t[2] == 5.5
    if extension:
        with pytest.raises(TypeError):
            minus("7")
        with pytest.raises(TypeError):
            minus(*range(60))
        with pytest.raises(TypeError):
            put(t, *[0.5] * 9)
        from production_stack_amd import _C

        view = torch.zeros(4, 6)[:, 1:3]
        assert _C.row_stride(view, "x") == 6
        for bad in (view.t(), t):
            with pytest.raises(ValueError, match="x: need a 2-D view"):
                _C.row_stride(bad, "x")

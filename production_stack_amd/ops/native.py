"""Builder and loader of the mixer-kernel libraries (`_mixops*.so`).

The fp32-residual / delta-rule / linear-scan / attention kernels expose a
plain C ABI, so the libraries need hipcc only: no torch headers,
seconds-to-minutes to build, and a fresh checkout compiles on first use just
the group of files a model's ops live in, without building the large `_C`
extension (which, where it is built, makes the calls: entry_call.cpp). Launchers
receive raw device pointers and the current HIP stream; shape checks live in the
Python wrappers
(production_stack_amd/ops/__init__.py).

Groups (one shared library each):
  core    resid32, norm_conv, mixer_prep, talk_attention, talk_mfma,
          talk_token, window_attention, attn_f32, mfma_attention,
          expand_attention, latent_decode, keyval_attention, moe_route, moe_group, mingru_scan -> _mixops.so
  delta   delta_rule                        -> _mixops_delta.so
  gdelta  gated_delta                       -> _mixops_gdelta.so
  scan    linear_scan                       -> _mixops_scan.so
  chunk   chunk_scan, token_scan            -> _mixops_chunk.so
"""

from __future__ import annotations

import ctypes
import functools
import glob
import hashlib
import mmap
import os
import shutil
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROOT = os.path.dirname(PKG)
LIB_PATH = os.path.join(PKG, "_mixops.so")

HIPCC_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950",
    # packed-fp32 instruction forms stay off
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]

# group -> [(source, extra defines)]: the recurrence files are compiled once
# per element type (or decay law) so their many head-size instantiations
# build in parallel
GROUPS = {
    "core": [
        ("resid32.hip", []),
        ("norm_conv.hip", []),
        ("talk_attention.hip", []),
        ("talk_mfma.hip", []),
        ("window_attention.hip", []),
        ("attn_f32.hip", []),
        ("talk_token.hip", []),
        ("mixer_prep.hip", []),
        ("mfma_attention.hip", []),
        ("expand_attention.hip", []),
        ("latent_decode.hip", []),
        ("keyval_attention.hip", []),
        ("moe_route.hip", []),
        ("moe_group.hip", []),
        ("mingru_scan.hip", []),
    ],
    "delta": [
        ("delta_rule.hip", ["-DMX_ONLY_DTYPE=0"]),
        ("delta_rule.hip", ["-DMX_ONLY_DTYPE=1"]),
    ],
    "gdelta": [
        ("gated_delta.hip", ["-DMX_ONLY_DTYPE=0"]),
        ("gated_delta.hip", ["-DMX_ONLY_DTYPE=1"]),
    ],
    # one unit per (decay law, element type)
    "scan": [("linear_scan.hip", [f"-DLS_ONLY={i}"]) for i in range(6)],
    # one unit per recurrence
    "chunk": ([("chunk_scan.hip", [f"-DCK_ONLY={i}"]) for i in range(5)]
              + [("token_scan.hip", [])]),
}

LIB_PATHS = {
    "core": LIB_PATH,
    "delta": os.path.join(PKG, "_mixops_delta.so"),
    "gdelta": os.path.join(PKG, "_mixops_gdelta.so"),
    "scan": os.path.join(PKG, "_mixops_scan.so"),
    "chunk": os.path.join(PKG, "_mixops_chunk.so"),
}

# entry points outside the core group
SYMBOL_GROUP = {
    "mx_delta_rule": "delta",
    "mx_gated_delta": "gdelta",
    "mx_linear_scan": "scan",
    "mx_linear_scan_splits": "scan",
    "mx_chunk_scratch": "chunk",
    "mx_chunk_delta": "chunk",
    "mx_chunk_gated": "chunk",
    "mx_chunk_scan": "chunk",
    "mx_token_scan": "chunk",
}

# entry points that return a status (the others return nothing)
INT_RESULT = {
    "mx_delta_rule", "mx_talk_attention", "mx_gated_delta",
    "mx_short_conv_silu", "mx_mfma_attention", "mx_linear_scan",
    "mx_linear_scan_splits", "mx_norm_conv32", "mx_moe_route",
    "mx_add_layer_norm32", "mx_expert_plan", "mx_expand_attention",
    "mx_latent_decode", "mx_keyval_attention", "mx_chunk_delta",
    "mx_chunk_gated", "mx_chunk_scan", "mx_token_scan", "mx_talk_mfma",
    "mx_window_attention", "mx_attn_f32", "mx_talk_token",
    "mx_talk_rows_f32",
}

# entry points that return a 64-bit count
LONG_RESULT = {"mx_mingru_scratch", "mx_chunk_scratch"}


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: cannot build the mixer kernels")
    return exe


SRC_DIR = os.path.join(ROOT, "csrc")
_KEY = b"mx_build_key="


@functools.lru_cache(maxsize=None)
def source_key(group: str) -> str:
    """Names what a group's library is built from: its units and defines, the
    shared headers, the flags. Empty where the sources are not there."""
    units = GROUPS[group]
    names = sorted({src for src, _ in units})
    names += sorted(os.path.basename(h)
                    for h in glob.glob(os.path.join(SRC_DIR, "*.h")))
    digest = hashlib.sha256(repr((HIPCC_FLAGS, units, names)).encode())
    for name in names:
        try:
            with open(os.path.join(SRC_DIR, name), "rb") as f:
                digest.update(hashlib.sha256(f.read()).digest())
        except OSError:
            return ""
    return digest.hexdigest()[:16]


def built_key(path: str) -> str:
    """The key in a built library, empty where it has none."""
    with open(path, "rb") as f, mmap.mmap(
            f.fileno(), 0, access=mmap.ACCESS_READ) as m:
        at = m.find(_KEY)
        return m[at + len(_KEY):at + len(_KEY) + 16].decode() if at >= 0 else ""


def current(group: str) -> bool:
    """A library is there and built from the sources that are. The entry
    points are called without types: one of other sources may take other
    arguments and would read them as its own."""
    path = LIB_PATHS[group]
    return os.path.exists(path) and source_key(group) in (
        "", built_key(path))


def _build_group(group: str) -> str:
    hipcc = _hipcc()
    src_dir = SRC_DIR
    key = source_key(group)
    units = GROUPS[group]
    tmp = tempfile.mkdtemp(prefix=f"mixops-{group}-", dir=PKG)
    try:
        def compile_one(i_unit):
            i, (src, defs) = i_unit
            obj = os.path.join(tmp, f"u{i}.o")
            cmd = [hipcc, *HIPCC_FLAGS, *defs, "-I", src_dir, "-c",
                   os.path.join(src_dir, src), "-o", obj]
            r = subprocess.run(cmd, stdout=subprocess.PIPE,
                               stderr=subprocess.STDOUT, text=True)
            if r.returncode != 0:
                raise RuntimeError(
                    f"hipcc failed on {src}:\n{r.stdout[-4000:]}")
            return obj

        with ThreadPoolExecutor(max_workers=len(units)) as ex:
            objs = list(ex.map(compile_one, enumerate(units)))
        mark = os.path.join(tmp, "key.c")
        with open(mark, "w") as f:
            f.write('__attribute__((used)) const char mx_build_key[] = "%s";\n'
                    % (_KEY.decode() + key))
        out = os.path.join(tmp, "lib.so")
        r = subprocess.run(
            [hipcc, "-shared", "-fPIC", "--offload-arch=gfx950", *objs,
             "-x", "c", mark, "-o", out],
            stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stdout[-4000:]}")
        os.replace(out, LIB_PATHS[group])
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    return LIB_PATHS[group]


def build(force: bool = False, groups=None) -> str:
    """Compile the libraries in-tree (atomic replace), all groups unless
    `groups` names some; those that are current only with `force`. Returns
    the core library's path."""
    if force:
        source_key.cache_clear()
    todo = [g for g in (groups or GROUPS) if force or not current(g)]
    with ThreadPoolExecutor(max_workers=max(len(todo), 1)) as ex:
        list(ex.map(_build_group, todo))
    return LIB_PATH


def _entry(fn, name: str):
    """A callable for an entry point, whose arguments are tensors or None (a
    pointer), integers and floats. The `_C` extension marshals them; without it
    ctypes does, which takes longer than a launch."""
    try:
        from production_stack_amd import _C
    except ImportError:
        _C = None
    if hasattr(_C, "entry"):
        kind = 1 if name in INT_RESULT else 2 if name in LONG_RESULT else 0
        return _C.entry(ctypes.cast(fn, ctypes.c_void_p).value, kind, name)
    fn.restype = (ctypes.c_int if name in INT_RESULT else
                  ctypes.c_long if name in LONG_RESULT else None)

    def argument(a):
        if isinstance(a, float):
            return ctypes.c_float(a)
        if a is None or isinstance(a, int):
            return ctypes.c_void_p(a) if not a or a >> 31 else a
        return ctypes.c_void_p(a.data_ptr())

    return lambda *args: fn(*map(argument, args))


class _Libs:
    """Attribute access resolves an entry point in its group's library,
    which is loaded (and built, when it is not there or was built from other
    sources) on first use."""

    def __init__(self) -> None:
        self._handles = {}

    def _handle(self, group: str):
        h = self._handles.get(group)
        if h is None:
            if not current(group):
                _build_group(group)
            h = ctypes.CDLL(LIB_PATHS[group])
            self._handles[group] = h
        return h

    def __getattr__(self, name: str):
        if not name.startswith("mx_"):
            raise AttributeError(name)
        fn = _entry(getattr(self._handle(SYMBOL_GROUP.get(name, "core")),
                            name), name)
        setattr(self, name, fn)
        return fn


_lib = None


def load():
    """Handle of the libraries (see _Libs)."""
    global _lib
    if _lib is None:
        _lib = _Libs()
    return _lib


def available() -> bool:
    return all(os.path.exists(p) for p in LIB_PATHS.values())

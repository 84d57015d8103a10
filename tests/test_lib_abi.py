"""C ABI surface of libvbhip.so (CPU tier: no kernel is launched).

* every function declared in include/vbhip.h is exported by the library and
  bound by dslperfgap_amd._lib with the same arity;
* argument errors are rejected before any HIP call, with a negative status and
  a message in vbh_last_error(), surfaced in Python as VbhError.
"""
import ctypes
import re
from pathlib import Path

import pytest
import torch

from dslperfgap_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "vbhip.h"


def _declared():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    decls = {}
    for m in re.finditer(r"\b(?:int|int64_t|const char\*)\s+(vbh_\w+)\s*\(([^)]*)\)\s*;", text):
        args = [a.strip() for a in m.group(2).split(",") if a.strip() and a.strip() != "void"]
        decls[m.group(1)] = len(args)
    return decls


def test_library_present():
    assert _lib.LIB_PATH.exists(), "run `python -m dslperfgap_amd.build` first"


def test_header_symbols_exported_and_bound():
    decls = _declared()
    assert len(decls) >= 10
    lib = _lib.lib()
    for name, arity in decls.items():
        assert hasattr(lib, name), f"{name} declared in vbhip.h but not exported"
        assert name in _lib.SIGNATURES, f"{name} not bound in _lib.SIGNATURES"
        assert len(_lib.SIGNATURES[name][1]) == arity, f"{name}: arity differs from the header"
    assert set(_lib.SIGNATURES) == set(decls)


def test_abi_version():
    assert _lib.lib().vbh_abi_version() == _lib.ABI_VERSION


def _expect(code, name, *args, match=None):
    with pytest.raises(_lib.VbhError) as ei:
        _lib.call(name, *args)
    assert ei.value.code == code
    if match:
        assert re.search(match, str(ei.value)), str(ei.value)


def test_argument_errors_before_launch():
    # dtype errors
    _expect(_lib.E_DTYPE, "vbh_layer_norm_fwd", 16, 16, 16, 16, 4, 4, 1e-5, 7, 7, None,
            match="unsupported dtype")
    _expect(_lib.E_DTYPE, "vbh_layer_norm_fwd", 16, 16, 16, 16, 4, 4, 1e-5, _lib.BF16, _lib.F16,
            None, match="weight dtype")
    _expect(_lib.E_DTYPE, "vbh_softmax_fwd", 16, 16, 4, 4, _lib.F32, _lib.BF16, 0, None)
    _expect(_lib.E_DTYPE, "vbh_cross_entropy_fwd", 16, 16, _lib.F32, _lib.F32, 16, 16, 16, 4, 4,
            4, 0.0, 1.0, 0.0, -100, 4, 0, 4, 0, 0, None, match="int32 or int64")
    # size / flag errors
    _expect(_lib.E_INVALID, "vbh_rms_norm_fwd", 16, 16, 16, -1, 4, 1e-5, _lib.F32, _lib.F32,
            None, match="negative")
    _expect(_lib.E_INVALID, "vbh_softmax_fwd", 16, 16, 4, 4, _lib.F32, _lib.F32, 2, None,
            match="log_mode")
    _expect(_lib.E_INVALID, "vbh_cross_entropy_fwd", 16, 16, _lib.F32, _lib.I64, 16, 16, 16, 4,
            4, 4, 0.0, 1.0, 0.0, -100, 4, 0, 0, 0, 0, None, match="BLOCK_SIZE")
    _expect(_lib.E_INVALID, "vbh_cross_entropy_fwd", 16, 16, _lib.F32, _lib.I64, 16, 16, 16, 4,
            8, 4, 0.0, 1.0, 0.0, -100, 8, 0, 8, 0, 0, None, match="row_stride")
    _expect(_lib.E_INVALID, "vbh_layer_norm_fwd", None, 16, 16, 16, 4, 4, 1e-5, _lib.F32,
            _lib.F32, None, match="null")
    _expect(_lib.E_INVALID, "vbh_stream_copy", 16, 16, 15, None, match="multiple of 16")
    _expect(_lib.E_RANGE, "vbh_softmax_fwd", 16, 16, 4, 1 << 31, _lib.F32, _lib.F32, 0, None)
    _expect(_lib.E_INVALID, "vbh_tune_override", 0, 3, 0, 0, match="power of two")
    _expect(_lib.E_INVALID, "vbh_tune_override", 0, 96, 0, 0, match="multiple of 64")
    _expect(_lib.E_INVALID, "vbh_tune_override", 0, 128, 192, 0, match="multiple of tpr")
    _expect(_lib.E_INVALID, "vbh_tune_override", 9, 0, 0, 0, match="bad op")
    _expect(_lib.E_INVALID, "vbh_tune_override", 0, 0, 0, 64, match="flag")
    assert _lib.last_error()


def test_huge_sizes_are_range_errors_before_launch():
    """Row counts whose products overflow 64 bits (or exceed 2^32 work-items)
    are rejected with VBH_E_RANGE before anything is launched."""
    huge = 1 << 62
    _expect(_lib.E_RANGE, "vbh_layer_norm_fwd", 16, 16, 16, 16, huge, 1024, 1e-5, _lib.F32,
            _lib.F32, None, match="exceeds 2\\^32")
    _expect(_lib.E_RANGE, "vbh_rms_norm_fwd", 16, 16, 16, huge, 4096, 1e-5, _lib.BF16,
            _lib.BF16, None)
    _expect(_lib.E_RANGE, "vbh_softmax_fwd", 16, 16, huge, 8, _lib.F16, _lib.F16, 1, None)
    _expect(_lib.E_RANGE, "vbh_logsumexp_fwd", 16, 16, huge, 8, _lib.F32, _lib.F32, None)
    _expect(_lib.E_RANGE, "vbh_softmax_dim_fwd", 16, 16, huge, 4, huge, _lib.F32, _lib.F32, 0,
            None, match="too large")
    _expect(_lib.E_RANGE, "vbh_reduce_fwd", 16, 16, 16, huge, 64, 1, _lib.F32, _lib.F32, 1, None)
    _expect(_lib.E_RANGE, "vbh_reduce_fwd", 16, 16, 16, huge, 64, huge, _lib.F32, _lib.F32, 1,
            None, match="too large")
    _expect(_lib.E_RANGE, "vbh_cross_entropy_fwd", 16, 16, _lib.F32, _lib.I64, 16, 16, 16, huge,
            1 << 20, 1 << 20, 0.0, 1.0, 0.0, -100, 1 << 20, 0, 16, 0, 0, None)
    _expect(_lib.E_RANGE, "vbh_cross_entropy_bwd", 16, 16, 16, 16, 16, _lib.F32, _lib.I64, huge,
            1 << 20, 1 << 20, 1 << 20, 1, 0.0, 1.0, 0.0, -100, 1 << 20, 0, 0, None)


def test_empty_sizes_are_noops():
    # zero rows: nothing to launch, status 0 (no device touched)
    _lib.call("vbh_layer_norm_fwd", None, None, None, None, 0, 128, 1e-5, _lib.F32, _lib.F32,
              None)
    _lib.call("vbh_softmax_fwd", None, None, 0, 7, _lib.F16, _lib.F32, 1, None)
    _lib.call("vbh_stream_copy", None, None, 0, None)
    _lib.call("vbh_tune_override", 2, 0, 0, 0)


def test_missing_library_is_loud(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "absent.so")
    monkeypatch.setattr(_lib, "_lib", None)
    with pytest.raises(ImportError, match="no non-HIP fallback"):
        _lib.lib()


# ---------------------------------------------------------------------------
# the CPython binding (_vbhfast) of the launching entry points
# ---------------------------------------------------------------------------
def _fast():
    _lib.lib()
    from dslperfgap_amd import _vbhfast
    return _vbhfast


def test_fast_binding_covers_every_launching_entry_point():
    """Every entry point that takes a stream is bound by _vbhfast, with the
    header's arity, and launches go through it."""
    fast = _fast()
    decls = _declared()
    launching = {n for n, (_, args) in _lib.SIGNATURES.items()
                 if args and args[-1] is ctypes.c_void_p and n != "vbh_tune_override"}
    assert launching == set(_lib.FAST_ENTRY_POINTS)
    assert fast.ABI_VERSION == _lib.ABI_VERSION
    for name in _lib.FAST_ENTRY_POINTS:
        fn = getattr(fast, name)
        assert _lib._fns[name] is fn
        with pytest.raises(TypeError, match=f"expected {decls[name]} arguments"):
            fn(*([0] * (decls[name] - 1)))


def test_fast_and_ctypes_bindings_agree_on_argument_errors():
    """The same call through both bindings gives the same status and message."""
    fast = _fast()
    handle = _lib.lib()
    cases = [
        ("vbh_softmax_fwd", (16, 16, -1, 4, 0, 0, 0, None)),
        ("vbh_softmax_fwd", (16, 16, 4, 4, 0, 0, 2, None)),
        ("vbh_layer_norm_fwd", (16, 16, 16, 16, 4, 4, 1e-5, 7, 7, None)),
        ("vbh_reduce_fwd", (16, 16, 16, 1, 8, 1, 0, 0, 3, None)),
        ("vbh_stream_copy", (16, 16, 15, None)),
        ("vbh_cross_entropy_bwd", (16, 16, 16, 16, 16, 0, 9, 2, 4, 4, 4, 1, 0.0, 1.0, 0.0,
                                   -100, 4, 0, 0, None)),
    ]
    for name, args in cases:
        rc_fast = getattr(fast, name)(*args)
        msg_fast = _lib.last_error()
        rc_ct = getattr(handle, name)(*args)
        assert rc_fast == rc_ct < 0, (name, rc_fast, rc_ct)
        assert msg_fast == _lib.last_error(), name


def test_fast_binding_rejects_bad_argument_types():
    fast = _fast()
    with pytest.raises(TypeError):
        fast.vbh_stream_copy(16, 16, 1.5, None)       # size must be an int
    with pytest.raises(TypeError):
        fast.vbh_stream_copy("16", 16, 16, None)      # pointer must be an int or None


def test_fast_binding_formats_match_the_ctypes_signatures():
    """Each _vbhfast entry point converts its arguments as the ctypes
    declaration of the same header entry does (pointer, int64, int, float)."""
    fast = _fast()
    code = {ctypes.c_void_p: "p", ctypes.c_int64: "q", ctypes.c_int: "i", ctypes.c_float: "f"}
    assert set(fast.FORMATS) == set(_lib.FAST_ENTRY_POINTS)
    for name in _lib.FAST_ENTRY_POINTS:
        want = "".join(code[a] for a in _lib.SIGNATURES[name][1])
        assert fast.FORMATS[name] == want, name


def test_fast_binding_rejects_ints_outside_c_int():
    """An int parameter (a dtype code here) out of C int range raises instead of
    wrapping round to another value; nothing is called (and the other
    arguments would be rejected by the library if anything were)."""
    fast = _fast()
    with pytest.raises(OverflowError, match="does not fit a C int"):
        fast.vbh_softmax_fwd(16, 16, -1, 4, 1 << 32, 0, 0, None)
    with pytest.raises(OverflowError):
        fast.vbh_reduce_fwd(16, 16, 16, 1, 8, 1, 0, 0, -(1 << 31) - 1, None)


def test_fast_binding_calls_the_instance_ctypes_loaded(tmp_path):
    """With VBHIP_LIB naming another copy of the library, launches through
    _vbhfast reach that copy: an argument error raised through the fast path
    leaves its message in that copy's vbh_last_error (read through ctypes)."""
    import os
    import shutil
    import subprocess
    import sys

    copy = tmp_path / "libvbhip.so"
    shutil.copy(_lib.LIB_PATH, copy)
    shutil.copy(_lib.LIB_PATH.with_suffix(".srchash"), copy.with_suffix(".srchash"))
    code = (
        "from pathlib import Path\n"
        "from dslperfgap_amd import _lib\n"
        "_lib.lib()\n"
        f"assert _lib.LIB_PATH == Path({str(copy)!r}), _lib.LIB_PATH\n"
        "rc = _lib.entry('vbh_softmax_fwd')(16, 16, -1, 4, 0, 0, 0, None)\n"
        "assert rc == _lib.E_INVALID, rc\n"
        "assert 'negative size' in _lib.last_error(), repr(_lib.last_error())\n"
    )
    env = dict(os.environ, VBHIP_LIB=str(copy),
               PYTHONPATH=str(HEADER.parents[1]) + os.pathsep + os.environ.get("PYTHONPATH", ""))
    res = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True,
                         timeout=120)
    assert res.returncode == 0, res.stderr[-2000:]


def test_fast_binding_refuses_calls_before_bind():
    """The module only calls entry points it was bound to (by _lib.lib())."""
    fast = _fast()
    with pytest.raises(KeyError, match="no address"):
        fast.bind({})
    with pytest.raises(TypeError):
        fast.bind([])


def test_split_workspace_sizes():
    """The row split is a pure function of the launch shape: few rows of at
    least 256 KiB split (segments of >= 512 16-byte vectors, a power of two per
    row, about 1024 segments per launch), many rows or shorter rows do not, and
    an overridden geometry turns it off.  A logsumexp or softmax segment keeps
    its max and its sum of exp (two fp32 values), a cross-entropy segment its
    loss, max and sum (three)."""
    h = _lib.lib()
    lse, red = h.vbh_logsumexp_workspace_bytes, h.vbh_reduce_workspace_bytes
    assert lse(8192, 4096, _lib.F32) == 0                 # many rows
    assert lse(128, 131072, _lib.F32) == 128 * 8 * 8      # 8 segments of 4096 vectors
    assert lse(1, 65536, _lib.F32) == 1 * 32 * 8          # capped by the segment size
    assert lse(300, 131072, _lib.F32) == 300 * 4 * 8      # long rows: up to 511 rows
    assert lse(384, 32768, _lib.F32) == 0                 # not long enough for that
    assert lse(64, 50304, _lib.F32) == 0                  # 200 KB rows: not worth a split
    assert lse(1, 65536, _lib.F16) == 0                   # 128 KB row
    assert lse(4, 1000, _lib.F32) == 0                    # too short to split
    assert lse(4, 65537, _lib.F32) == 4 * 32 * 8          # not whole vectors: 31 x 2052 + 1925
    assert lse(333, 50257, _lib.F32) == 333 * 4 * 8       # long rows, 4 segments of 12568
    assert lse(4, 65536, 9) == 0 and lse(0, 65536, _lib.F32) == 0
    assert red(128, 131072, 1, _lib.F32, _lib.REDUCE_MEAN) == 128 * 8 * 4
    assert red(128, 131072, 1, _lib.F32, _lib.REDUCE_MAX) == 128 * 8 * (8 + 4)
    assert red(128, 131072, 1, _lib.F16, _lib.REDUCE_ARGMAX) == 128 * 8 * (8 + 2)
    assert red(300, 131072, 1, _lib.F32, _lib.REDUCE_MEAN) == 0  # long rows: logsumexp only
    assert red(128, 131072, 4, _lib.F32, _lib.REDUCE_MEAN) == 0  # middle axis: enough slabs
    assert red(1, 4100, 264, _lib.F32, _lib.REDUCE_MEAN) > 0      # one slab of few columns
    sm = h.vbh_softmax_workspace_bytes
    assert sm(128, 131072, _lib.F32) == 128 * 8 * 8       # as logsumexp's few-rows split
    assert sm(8192, 4096, _lib.F32) == 0 and sm(300, 131072, _lib.F32) == 0
    assert sm(200, 65536, _lib.F32) == 0                  # 129 rows or more: not split
    assert sm(64, 65536, _lib.F32) == 0                   # fp32 33-64 rows: 32768 vectors
    assert sm(64, 65536, _lib.BF16) == 64 * 16 * 8        # 16-bit 33-64 rows: 6144 vectors
    assert sm(8, 32000, _lib.F32) == 8 * 8 * 8            # a decode step over a 32000 vocabulary
    assert sm(8, 16384, _lib.F32) == 0                    # 4096 vectors: not worth a split
    assert sm(4, 65537, _lib.F32) == 4 * 32 * 8           # rows not whole vectors: 2052-column segments
    assert sm(8, 50257, _lib.F32) == 8 * 16 * 8           # GPT-2's vocabulary, 16 x 3144 columns
    assert sm(1, 131072, _lib.BF16) == 1 * 32 * 8
    ce = h.vbh_cross_entropy_workspace_bytes
    assert ce(64, 128256, 1 << 17, _lib.F32) == 3 * 64 * 16 * 4  # one block per row
    assert ce(64, 128256, 32768, _lib.F32) == 0           # several column blocks: not split
    assert ce(64, 50304, 65536, _lib.F32) == 0
    assert ce(333, 50257, 65536, _lib.F32) == 3 * 333 * 4 * 4  # long rows, not whole vectors
    assert ce(667, 50257, 65536, _lib.BF16) == 0          # 667 rows: not split
    try:
        _lib.tune_override(_lib.OP_LOGSUMEXP, 64, 0, 0)
        assert _lib.logsumexp_workspace_bytes(128, 131072, _lib.F32) == 0
        _lib.tune_override(_lib.OP_SOFTMAX, 64, 0, 0)
        assert _lib.softmax_workspace_bytes(128, 131072, _lib.F32) == 0
    finally:
        _lib.tune_override(_lib.OP_LOGSUMEXP, 0, 0, 0)
        _lib.tune_override(_lib.OP_SOFTMAX, 0, 0, 0)
    assert _lib.softmax_workspace_bytes(128, 131072, _lib.F32) == 128 * 8 * 8
    assert _lib.logsumexp_workspace_bytes(128, 131072, _lib.F32) == 128 * 8 * 8


def test_split_entry_points_check_arguments():
    _expect(_lib.E_INVALID, "vbh_logsumexp_fwd_ws", 16, 16, 4, 4, _lib.F32, _lib.F32, 16, -1,
            None, match="workspace")
    _expect(_lib.E_INVALID, "vbh_reduce_fwd_ws", 16, 16, 16, 4, 8, 1, _lib.F32, _lib.F32, 1, 16,
            -1, None, match="workspace")
    _expect(_lib.E_DTYPE, "vbh_logsumexp_fwd_ws", 16, 16, 4, 4, _lib.F32, _lib.F16, 16, 64, None)
    _expect(_lib.E_RANGE, "vbh_reduce_fwd_ws", 16, 16, 16, 1 << 62, 64, 1, _lib.F32, _lib.F32, 1,
            16, 64, None)


def test_positive_hip_status_raises_vbh_error_with_the_runtime_message():
    """A call that passes argument validation reaches the HIP runtime; with no
    device the runtime reports hipErrorNoDevice (100).  The entry point returns
    that positive status, vbh_last_error() names the launch and the runtime's
    error, and _lib.call raises VbhError carrying both -- the failure the
    reference's harness records as an ERROR (ViperBench/test_utils.py:115-119)."""
    if torch.cuda.device_count() > 0:
        pytest.skip("a GPU is visible; this test passes host pointers and needs none")
    import ctypes

    buf = (ctypes.c_float * 4096)()
    p = (ctypes.addressof(buf) + 15) // 16 * 16
    cases = [("vbh_layer_norm_fwd", (p, p, p, p, 4, 256, 1e-5, 0, 0, None), "layer_norm launch"),
             ("vbh_softmax_fwd", (p, p, 4, 256, 0, 0, 1, None), "softmax launch"),
             ("vbh_stream_copy", (p, p, 256, None), "stream_copy launch")]
    for name, args, what in cases:
        rc = _lib.entry(name)(*args)
        assert rc > 0, (name, rc)
        msg = _lib.last_error()
        assert msg.startswith(what) and "hipError" in msg, (name, msg)
        with pytest.raises(_lib.VbhError) as ei:
            _lib.call(name, *args)
        assert ei.value.code == rc and msg in str(ei.value), name


def _tree_copy(tmp_path):
    """The package (sources, built library and binding, hash) and include/ in tmp."""
    import shutil

    root = Path(__file__).resolve().parents[1]
    dst = tmp_path / "repo"
    shutil.copytree(root / "dslperfgap_amd", dst / "dslperfgap_amd",
                    ignore=shutil.ignore_patterns("_build", "__pycache__", "results"))
    shutil.copytree(root / "include", dst / "include")
    return dst


def _load_in(tree) -> "subprocess.CompletedProcess":
    import subprocess
    import sys

    code = ("import dslperfgap_amd._lib as l\n"
            "try:\n    l.lib()\nexcept ImportError as e:\n    print('IMPORTERROR', e)\n"
            "else:\n    print('LOADED', l.LIB_PATH)\n")
    env = {k: v for k, v in __import__("os").environ.items() if k != "VBHIP_LIB"}
    return subprocess.run([sys.executable, "-c", code], cwd=tree, env=env, capture_output=True,
                          text=True, timeout=120)


def test_library_built_from_other_sources_is_refused(tmp_path):
    """The library loads from an untouched copy of the tree; after one source
    file changes (a comment is enough) the loader raises ImportError naming the
    rebuild, and a missing hash file is refused the same way."""
    tree = _tree_copy(tmp_path)
    ok = _load_in(tree)
    assert "LOADED" in ok.stdout and str(tree) in ok.stdout, ok.stdout + ok.stderr
    src = tree / "dslperfgap_amd" / "csrc" / "softmax.hip"
    src.write_text(src.read_text() + "\n// touched\n")
    bad = _load_in(tree)
    assert "IMPORTERROR" in bad.stdout and "built from other sources" in bad.stdout, bad.stdout
    assert "dslperfgap_amd.build" in bad.stdout
    (tree / "dslperfgap_amd" / "libvbhip.srchash").unlink()
    gone = _load_in(tree)
    assert "IMPORTERROR" in gone.stdout and "srchash is missing" in gone.stdout, gone.stdout


def test_header_change_is_a_source_change(tmp_path):
    tree = _tree_copy(tmp_path)
    hdr = tree / "include" / "vbhip.h"
    hdr.write_text(hdr.read_text() + "\n/* touched */\n")
    bad = _load_in(tree)
    assert "IMPORTERROR" in bad.stdout and "built from other sources" in bad.stdout, bad.stdout


def test_release_library_has_no_bounds_checks():
    """The debug-bounds entry points exist in the release library and say it
    is not the checked build (before any HIP call)."""
    n = ctypes.c_int64(-1)
    _expect(_lib.E_UNSUPPORTED, "vbh_debug_bounds", ctypes.byref(n), None, 0, 1,
            match="VBH_DEBUG_BOUNDS")
    _expect(_lib.E_UNSUPPORTED, "vbh_debug_bounds_slack", 16, match="VBH_DEBUG_BOUNDS")


def test_debug_library_exports_the_abi():
    """libvbhip_debug.so, the bounds-checked build, exports the header's ABI
    and rejects bad arguments of its debug entry points before any HIP call
    (loaded in a child process, next to no other copy of the library)."""
    import subprocess
    import sys

    from dslperfgap_amd.build import DEBUG_LIB_PATH

    assert DEBUG_LIB_PATH.exists(), "run `python -m dslperfgap_amd.build` first"
    code = f"""
import ctypes, sys
lib = ctypes.CDLL({str(DEBUG_LIB_PATH)!r})
names = {sorted(_declared())!r}
missing = [n for n in names if not hasattr(lib, n)]
assert not missing, missing
assert lib.vbh_abi_version() == {_lib.ABI_VERSION}
lib.vbh_debug_bounds.argtypes = [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_int64, ctypes.c_int]
assert lib.vbh_debug_bounds(None, None, 0, 0) == {_lib.E_INVALID}
lib.vbh_debug_bounds_slack.argtypes = [ctypes.c_int64]
assert lib.vbh_debug_bounds_slack(-16) == {_lib.E_INVALID}
lib.vbh_last_error.restype = ctypes.c_char_p
print(lib.vbh_last_error().decode())
"""
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                         timeout=120)
    assert res.returncode == 0, res.stderr[-3000:]
    assert "negative byte count" in res.stdout

"""ctypes binding of libhira_hip.so (include/hira_hip.h).

The library is the product: when it is missing or an entry point is absent this module
raises, it never falls back to a host implementation.
"""
from __future__ import annotations

import ctypes as C
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
LIB_PATH = CSRC / "libhira_hip.so"

HIRA_MAX_LEVELS = 8
HIRA_STATS_COLS = HIRA_MAX_LEVELS + 3  # counters per tree a search can fill in
HIRA_F32, HIRA_BF16 = 0, 1
HIRA_ROW_MAJOR, HIRA_TILE16, HIRA_TILE16_Q8 = 0, 1, 2
HIRA_ABI_VERSION = 12
HIRA_UNIT_SCALE_HEADS = 4096

_vp = C.c_void_p


class HiraTree(C.Structure):
    _fields_ = [
        ("num_trees", C.c_int32),
        ("num_levels", C.c_int32),
        ("bf", C.c_int32),
        ("dim", C.c_int32),
        ("vdim", C.c_int32),
        ("dtype", C.c_int32),
        ("layout", C.c_int32),
        ("reserved_", C.c_int32),
        ("size", C.c_int32 * HIRA_MAX_LEVELS),
        ("cap", C.c_int32 * HIRA_MAX_LEVELS),
        ("keys", _vp),
        ("values", _vp),
        ("perm", _vp),
        ("centers", _vp * HIRA_MAX_LEVELS),
        ("radii", _vp * HIRA_MAX_LEVELS),
        ("counts", _vp * HIRA_MAX_LEVELS),
        ("keys8", _vp),
        ("kscale", _vp),
        ("keps", _vp),
    ]


class HiraQuery(C.Structure):
    """`out_dtype` (HIRA_F32 or HIRA_BF16: the type hira_search writes attn_out in) lies in what was
    padding once, and comes last by position: structs filled in by position keep their meaning."""

    _fields_ = [
        ("num_q_heads", C.c_int32),
        ("out_dtype", C.c_int32),
        ("q", _vp),
        ("tau", _vp),
        ("scaling", _vp),
        ("tree_q_off", _vp),
        ("tree_q_heads", _vp),
        ("max_group", C.c_int32),
        ("group_size", C.c_int32),
    ]

    def __init__(self, num_q_heads=0, q=None, tau=None, scaling=None, tree_q_off=None, tree_q_heads=None,
                 max_group=0, group_size=0, out_dtype=HIRA_F32):
        super().__init__(num_q_heads, out_dtype, q, tau, scaling, tree_q_off, tree_q_heads, max_group,
                         group_size)


class HiraQueue(C.Structure):
    _fields_ = [("keys", _vp), ("values", _vp), ("len", C.c_int32), ("cap", C.c_int32)]


class HiraSample(C.Structure):
    _fields_ = [("rows", _vp), ("num_rows", C.c_int32), ("method", C.c_int32), ("k", C.c_int32),
                ("wait", C.c_int32), ("tau", _vp), ("scratch", _vp)]


class HiraSearchOut(C.Structure):
    _fields_ = [
        ("dense", _vp),
        ("dense_stride", C.c_int64),
        ("dense_by_position", C.c_int32),
        ("dense_fill", C.c_int32),
        ("sel_index", _vp),
        ("sel_score", _vp),
        ("sel_count", _vp),
        ("sel_cap", C.c_int32),
        ("dense_fill_value", C.c_float),
        ("attn_out", _vp),
        ("stats", _vp),
    ]


class HiraLaunch(C.Structure):
    _fields_ = [
        ("block_threads", C.c_int32),
        ("nodes_per_wave", C.c_int32),
        ("kernel", C.c_int32),
        ("separate_merge", C.c_int32),
    ]


class HiraArray(C.Structure):
    _fields_ = [("dst", _vp), ("src", _vp), ("dst_stride", C.c_int64), ("src_stride", C.c_int64),
                ("copy_bytes", C.c_int64), ("fill_from", C.c_int64), ("fill", C.c_uint32),
                ("reserved_", C.c_int32)]


# every symbol include/hira_hip.h declares: (restype, argtypes)
SYMBOLS = {
    "hira_abi_version": (C.c_int, []),
    "hira_last_error": (C.c_char_p, []),
    "hira_unit_scale": (_vp, []),
    "hira_search_workspace_bytes": (
        C.c_size_t,
        [C.POINTER(HiraTree), C.POINTER(HiraQuery), C.POINTER(HiraQueue), C.POINTER(HiraLaunch)],
    ),
    "hira_search_counter_bytes": (
        C.c_size_t, [C.POINTER(HiraTree), C.POINTER(HiraQuery), C.POINTER(HiraLaunch)],
    ),
    "hira_search": (
        C.c_int,
        [C.POINTER(HiraTree), C.POINTER(HiraQuery), C.POINTER(HiraQueue),
         C.POINTER(HiraSearchOut), C.POINTER(HiraLaunch), _vp, C.c_size_t, _vp],
    ),
    "hira_search_sampled": (
        C.c_int,
        [C.POINTER(HiraTree), C.POINTER(HiraQuery), C.POINTER(HiraSample), C.POINTER(HiraQueue),
         C.POINTER(HiraSearchOut), C.POINTER(HiraLaunch), _vp, C.c_size_t, _vp],
    ),
    "hira_search_noalloc": (
        C.c_int,
        [C.POINTER(HiraTree), C.POINTER(HiraQuery), C.POINTER(HiraQueue),
         C.POINTER(HiraSearchOut), C.POINTER(HiraLaunch), _vp],
    ),
    "hira_build_workspace_bytes": (C.c_size_t, [C.POINTER(HiraTree), C.c_int32]),
    "hira_build": (
        C.c_int,
        [C.POINTER(HiraTree), _vp, _vp, C.c_int32, C.c_int32, C.c_int32, C.c_uint64, _vp,
         C.c_size_t, _vp],
    ),
    "hira_build_ragged": (
        C.c_int,
        [C.POINTER(HiraTree), _vp, _vp, C.c_int32, _vp, C.c_int32, C.c_int32, C.c_uint64, _vp,
         C.c_size_t, _vp],
    ),
    "hira_rebuild_workspace_bytes": (C.c_size_t, [C.POINTER(HiraTree)]),
    "hira_rebuild_subtree": (
        C.c_int,
        [C.POINTER(HiraTree), C.c_int32, C.c_int32, C.c_int32, C.c_uint64, _vp, _vp, C.c_size_t, _vp],
    ),
    "hira_nearest_workspace_bytes": (C.c_size_t, [C.c_int32, C.c_int32, C.c_int32, C.c_int32]),
    "hira_nearest": (
        C.c_int,
        [_vp, C.c_int32, C.c_int32, C.c_int32, _vp, C.c_int32, C.c_int32, _vp, _vp, _vp, _vp,
         C.c_size_t, _vp],
    ),
    "hira_quantize": (C.c_int, [C.POINTER(HiraTree), C.c_int32, C.c_int32, C.c_int32, _vp]),
    "hira_update": (C.c_int, [C.POINTER(HiraTree), _vp, _vp, C.c_int32, _vp, _vp]),
    "hira_update_sample": (
        C.c_int,
        [C.POINTER(HiraTree), _vp, _vp, C.c_int32, _vp, _vp, C.c_int32, C.POINTER(C.c_int32),
         C.POINTER(C.c_int32), C.c_int32, _vp],
    ),
    "hira_read_state": (
        C.c_int, [C.POINTER(HiraTree), _vp, _vp, C.c_uint32, C.POINTER(C.c_int32), _vp],
    ),
    "hira_update_state": (C.c_int, [C.POINTER(HiraTree), C.c_int32, _vp, _vp]),
    "hira_sparse_attention": (
        C.c_int,
        [C.POINTER(HiraTree), C.POINTER(HiraQuery), _vp, _vp, _vp, C.c_int32, _vp, _vp],
    ),
    "hira_update_threshold": (
        C.c_int,
        [C.POINTER(HiraTree), _vp, _vp, C.c_int32, _vp, _vp, C.c_int32, C.POINTER(HiraQuery),
         C.c_int32, C.c_int32, _vp, _vp],
    ),
    "hira_enqueue": (
        C.c_int,
        [_vp, _vp, C.c_int32, C.c_int32, C.c_int32, C.c_int32, C.c_int32, C.c_int32, C.c_int32, _vp,
         _vp, _vp],
    ),
    "hira_replace_rows": (
        C.c_int,
        [_vp, C.c_int32, C.c_int32, C.c_int32, C.c_int32, _vp, C.c_int32, C.c_int32,
         C.POINTER(C.c_int32), C.POINTER(C.c_int32), C.c_int32, _vp],
    ),
    "hira_fill_arrays": (C.c_int, [C.POINTER(HiraArray), C.c_int32, C.c_int32, _vp]),
    "hira_threshold": (
        C.c_int,
        [_vp, C.c_int32, C.c_int32, C.c_int32, C.c_int32, C.POINTER(HiraQuery), C.c_int32,
         C.c_int32, _vp, _vp],
    ),
}

_lib = None


def build_library(verbose: bool = False) -> None:
    """Compile libhira_hip.so for gfx950 (hipcc cross-compiles without a GPU) and the native host side, for this interpreter."""
    r = subprocess.run(["make", "-C", str(CSRC), "-B", "-j8", f"PYTHON={sys.executable}"], capture_output=True, text=True)
    if verbose or r.returncode != 0:
        print(r.stdout[-4000:], r.stderr[-4000:])
    if r.returncode != 0:
        raise RuntimeError("building libhira_hip.so failed")


def use_library(path) -> None:
    """Load another build of the library than the default one (the build with time stamps that
    `make -C hira_amd/csrc timeline` makes, for looking at a decode step): call before anything
    else has used the library."""
    global LIB_PATH
    if _lib is not None:
        raise RuntimeError("the library is already loaded")
    LIB_PATH = Path(path).resolve()


def lib() -> C.CDLL:
    """The loaded library; raises when it has not been built."""
    global _lib
    if _lib is None:
        if not LIB_PATH.exists():
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with `make -C {CSRC}` "
                "(or __graft_entry__.build()); there is no host fallback")
        l = C.CDLL(str(LIB_PATH))
        for name, (res, args) in SYMBOLS.items():
            fn = getattr(l, name)  # AttributeError if the export is absent
            fn.restype = res
            fn.argtypes = args
        got = l.hira_abi_version()
        if got != HIRA_ABI_VERSION:
            raise RuntimeError(f"libhira_hip.so ABI {got}, expected {HIRA_ABI_VERSION}")
        _lib = l
    return _lib


_host_module = None


def host():
    """The native host side of the calls a decode step makes (csrc/host.cpp), on the loaded library's functions; raises when
    it has not been built, or was built for another torch, interpreter or library."""
    global _host_module
    if _host_module is None:
        l = lib()
        build = f"build it with `make -C {CSRC} PYTHON={sys.executable}` (or __graft_entry__.build())"
        try:
            import torch  # (its libraries, which the module needs)

            from hira_amd import _host
        except ImportError as ex:
            raise RuntimeError(f"the native host side, hira_amd/_host, is missing or was built for another torch ({ex}): {build}") from ex
        here = (f"{torch.__version__} {torch.version.git_version}", sys.version_info[0] << 8 | sys.version_info[1], l.hira_abi_version())
        built = getattr(_host, "BUILT_FOR", None)
        if built != here:
            raise RuntimeError(f"the native host side, {_host.__file__}, was built for {built} (torch, Python, ABI of the library), "
                               f"here are {here}: {build}")
        _host.bind({name: C.cast(getattr(l, name), _vp).value for name in SYMBOLS})
        _host_module = _host
    return _host_module


def in_chunks(x):
    """x, or its copy where it does not start at a multiple of 16 bytes: the kernels read rows in chunks of that, and
    ``contiguous`` hands a view that starts between two of them back as it is."""
    return x if x.data_ptr() % 16 == 0 else x.clone()


def check(rc: int) -> None:
    """Map a return code to the exception the reference's wrappers raise
    (kernels/triton_search_wrappers.py:9-110: ValueError for bad shapes)."""
    if rc == 0:
        return
    msg = lib().hira_last_error().decode(errors="replace")
    if rc == -1:
        raise ValueError(msg)
    raise RuntimeError(f"hira error {rc}: {msg}")


def stream_of(index: int) -> int:
    """Handle of torch's current HIP stream on device number `index`, as a tensor's ``get_device()``
    gives it: -1 is host memory, which torch would take for "the current device"."""
    if index < 0:
        raise ValueError("the arrays are in host memory: this call runs on the GPU")
    global _raw_stream
    if _raw_stream is None:
        import torch

        _raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or \
            (lambda i: torch.cuda.current_stream(i).cuda_stream)
    return _raw_stream(index)


_raw_stream = None


def current_stream(device) -> int:
    """Handle of torch's current HIP stream on `device`, for the `stream` argument of the
    library's calls.  The raw getter costs a fraction of a microsecond where
    ``torch.cuda.current_stream(device).cuda_stream`` builds two Python objects (some 15 us, once
    per layer and decode step)."""
    import torch

    device = torch.device(device)
    if device.type == "cpu":
        raise ValueError("the arrays are in host memory: this call runs on the GPU")
    idx = device.index
    if idx is None:
        idx = torch.cuda.current_device()
    raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)
    if raw is not None:
        return int(raw(idx))
    return torch.cuda.current_stream(idx).cuda_stream

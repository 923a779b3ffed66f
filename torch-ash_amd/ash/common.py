"""Loader and thin Python face of libash_hip.so.

The reference binds its native code with pybind11 (`import __ash`,
ash/common.py:4-15 and ash/src/pybind.cpp:8-38).  Here the native side is a
plain C-ABI shared library (include/ash_hip.h) loaded with ctypes; this module
rebuilds the exact surface the rest of the package expects from the extension
module: a `HashMap` class and the three `query_*` functions.  The calls that
programs make often go through `_ash_host` (csrc/ash_host.cpp), which checks
operands, allocates outputs and calls the same C ABI from C++.

There is no CPU or PyTorch fallback: if the library is missing, or a tensor is
not on a HIP device, the calls raise.
"""
import ctypes
import importlib.util
import itertools
import os
import warnings
from typing import Dict, Optional, Tuple

import torch
from torch.autograd import forward_ad

_LIB_NAME = "libash_hip.so"
_HOST_NAME = "_ash_host.so"
_LIB_DIR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib")

_I64 = ctypes.c_int64
_PTR = ctypes.c_void_p


class DotDict(dict):
    """dict whose items are also attributes (ash/common.py:19-22)."""

    __getattr__ = dict.__getitem__
    __setattr__ = dict.__setitem__
    __delattr__ = dict.__delitem__


class _QueryArgs(ctypes.Structure):
    _fields_ = [
        ("embeddings", _PTR),
        ("offsets", _PTR),
        ("grid_indices", _PTR),
        ("cell_indices", _PTR),
        ("masks", _PTR),
        ("lut_grid_nb2grid_idx", _PTR),
        ("lut_cell_nb2cell_idx", _PTR),
        ("lut_cell_nb2grid_nb", _PTR),
        ("num_queries", _I64),
        ("num_embeddings", _I64),
        ("cells_per_grid", _I64),
        ("embedding_dim", _I64),
        ("interpolation", ctypes.c_int32),
        ("dtype", ctypes.c_int32),
    ]


# name -> (restype, argtypes); mirrors include/ash_hip.h
_SIGNATURES = {
    "ash_last_error": (ctypes.c_char_p, []),
    "ash_abi_version": (ctypes.c_int, []),
    "ash_source_fingerprint": (ctypes.c_char_p, []),
    "ash_map_workspace_bytes": (
        ctypes.c_int,
        [ctypes.c_int, _I64, ctypes.POINTER(_I64), ctypes.POINTER(_I64)],
    ),
    "ash_map_create": (
        ctypes.c_int,
        [ctypes.c_int, _I64, _PTR, _PTR, _I64, ctypes.c_int, _PTR, ctypes.POINTER(_PTR)],
    ),
    "ash_map_attach_general": (ctypes.c_int, [_PTR, _PTR, _I64, _PTR]),
    "ash_map_destroy": (ctypes.c_int, [_PTR]),
    "ash_map_find": (ctypes.c_int, [_PTR, _PTR, _I64, _PTR, _PTR, _PTR]),
    "ash_grid_query": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, ctypes.c_int, _PTR, _PTR, _PTR, _PTR, _PTR],
    ),
    "ash_grid_forward": (
        ctypes.c_int,
        [_PTR, _PTR, _PTR, ctypes.c_float, ctypes.c_int, ctypes.POINTER(_QueryArgs), _PTR, _PTR, _PTR,
         _PTR, _PTR, _PTR],
    ),
    "ash_grid_activate": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int,
         _PTR, _PTR, _PTR, _PTR],
    ),
    "ash_grid_activate_static": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int,
         _PTR, _PTR, _PTR],
    ),
    "ash_grid_activate_positions": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, _PTR, ctypes.c_float, ctypes.c_int, ctypes.c_int, ctypes.c_int,
         ctypes.c_int, ctypes.c_int, _PTR, _PTR, _PTR],
    ),
    "ash_grid_integrate_depth_flagged": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, ctypes.c_int, ctypes.c_int, _PTR, _PTR, ctypes.c_float,
         ctypes.POINTER(ctypes.c_float), _PTR, _PTR, _PTR, _PTR, ctypes.c_int, ctypes.c_int,
         ctypes.c_float, ctypes.c_float, _PTR],
    ),
    "ash_grid_fuse_frame": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, _PTR, ctypes.c_float, ctypes.c_int, ctypes.c_int, ctypes.c_int,
         ctypes.c_int, _PTR, _PTR, _PTR, _I64, ctypes.c_int, ctypes.c_int, ctypes.c_float]
        + [_PTR] * 5 + [ctypes.c_int, ctypes.c_int, ctypes.c_float, ctypes.c_float, _PTR, _PTR],
    ),
    "ash_grid_integrate_depth": (
        ctypes.c_int,
        [_PTR, _I64, ctypes.c_int, ctypes.c_int, _PTR, _PTR, _I64, ctypes.c_float,
         ctypes.POINTER(ctypes.c_float), _PTR, _PTR, _PTR, _PTR, ctypes.c_int, ctypes.c_int,
         ctypes.c_float, ctypes.c_float, _PTR],
    ),
    "ash_grid_integrate_depth_touched": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, ctypes.c_int, ctypes.c_int, _PTR, _PTR, ctypes.c_float,
         ctypes.POINTER(ctypes.c_float), _PTR, _PTR, _PTR, _PTR, ctypes.c_int, ctypes.c_int,
         ctypes.c_float, ctypes.c_float, _PTR],
    ),
    "ash_ray_find_near_far": (
        ctypes.c_int,
        [_PTR, _PTR, _PTR, _PTR, _PTR, _I64, ctypes.c_float, ctypes.c_float, ctypes.c_float,
         ctypes.c_float, _PTR, _PTR, _PTR],
    ),
    "ash_ray_sample": (
        ctypes.c_int,
        [_PTR, _PTR, _PTR, _PTR, _PTR, _I64, _I64, ctypes.c_float, _PTR, _PTR, _PTR, _PTR, _PTR,
         _PTR],
    ),
    "ash_ray_sample_staged": (
        ctypes.c_int,
        [_PTR] * 5 + [_I64, _I64, ctypes.c_float, _PTR, _PTR, _I64, _PTR],
    ),
    "ash_ray_sample_compact": (ctypes.c_int, [_PTR] * 3 + [_I64, _I64] + [_PTR] * 4),
    "ash_ray_volume_bytes": (_I64, [ctypes.c_int, ctypes.c_int, _I64, ctypes.c_int]),
    "ash_map_ray_volume_bytes": (_I64, [_PTR, ctypes.c_int, ctypes.c_int, _I64, _I64]),
    "ash_ray_volume_kept": (ctypes.c_int, [_PTR, _PTR]),
    "ash_ray_find_near_far_world": (
        ctypes.c_int,
        [_PTR, _PTR, ctypes.c_int, ctypes.c_int] + [_PTR] * 3
        + [ctypes.c_float, _PTR, _PTR, _I64] + [ctypes.c_float] * 3 + [_PTR] * 3,
    ),
    "ash_ray_find_near_far_marked": (
        ctypes.c_int,
        [_PTR, _PTR] + [ctypes.c_int] * 3 + [_PTR] * 3
        + [ctypes.c_float, _PTR, _PTR, _I64] + [ctypes.c_float] * 3 + [_PTR] * 3,
    ),
    "ash_surface_block8_workspace_bytes": (_I64, [_I64, _I64]),
    "ash_surface_block8_classify": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, _PTR, _I64, _PTR, _PTR, _I64, _I64, ctypes.c_float, ctypes.c_float,
         ctypes.c_int32, _PTR, _PTR, _PTR],
    ),
    "ash_surface_block8_extract": (
        ctypes.c_int,
        [_PTR, _I64] + [_PTR] * 3 + [_I64, _I64, ctypes.c_float, ctypes.c_int32, _PTR, _I64, _I64,
                                     ctypes.c_int, ctypes.c_float, _PTR, _PTR, _PTR, _PTR],
    ),
    "ash_ray_sample_groups": (_I64, [_I64]),
    "ash_ray_sample_march": (
        ctypes.c_int,
        [_PTR, _PTR, ctypes.c_int, ctypes.c_int] + [_PTR] * 3
        + [ctypes.c_float, _PTR, _PTR, ctypes.c_float, ctypes.c_float, _I64, _I64,
           ctypes.c_float, _PTR, _PTR, _PTR, _I64, ctypes.POINTER(_I64), _PTR],
    ),
    "ash_ray_sample_march_marked": (
        ctypes.c_int,
        [_PTR, _PTR] + [ctypes.c_int] * 3 + [_PTR] * 3
        + [ctypes.c_float, _PTR, _PTR, ctypes.c_float, ctypes.c_float, _I64, _I64,
           ctypes.c_float, _PTR, _PTR, _PTR, _I64, ctypes.POINTER(_I64), _PTR],
    ),
    "ash_ray_sample_place": (
        ctypes.c_int, [_PTR] * 3 + [_I64, _I64, ctypes.c_float] + [_PTR] * 5,
    ),
    "ash_map_insert_keys": (ctypes.c_int, [_PTR, _PTR, _I64, _PTR]),
    "ash_map_insert_needs_scratch": (ctypes.c_int, [ctypes.c_int, ctypes.POINTER(_I64)]),
    "ash_map_insert": (
        ctypes.c_int,
        [
            _PTR,
            _PTR,
            _I64,
            ctypes.c_int,
            ctypes.POINTER(_PTR),
            ctypes.POINTER(_PTR),
            ctypes.POINTER(_I64),
            _PTR,
            _PTR,
        ],
    ),
    "ash_map_bulk_workspace_bytes": (
        ctypes.c_int,
        [_PTR, _I64, ctypes.c_int, ctypes.POINTER(_I64), ctypes.POINTER(_I64),
         ctypes.POINTER(ctypes.c_int)],
    ),
    "ash_map_insert_bulk": (
        ctypes.c_int,
        [
            _PTR,
            _PTR,
            _I64,
            ctypes.c_int,
            ctypes.POINTER(_PTR),
            ctypes.POINTER(_PTR),
            ctypes.POINTER(_I64),
            _PTR,
            _I64,
            _PTR,
        ],
    ),
    "ash_map_neighbors": (
        ctypes.c_int, [_PTR, _I64, ctypes.c_int, ctypes.c_int, _PTR, _PTR, _PTR]),
    "ash_map_items_in_index_order": (ctypes.c_int, [_PTR, ctypes.POINTER(ctypes.c_int)]),
    "ash_map_erase": (ctypes.c_int, [_PTR, _PTR, _I64, _PTR]),
    "ash_map_erase_bulk_query": (
        ctypes.c_int, [_PTR, _I64, ctypes.POINTER(_I64), ctypes.POINTER(ctypes.c_int)]
    ),
    "ash_map_erase_bulk": (ctypes.c_int, [_PTR, _PTR, _I64, _PTR, _I64, _PTR]),
    "ash_map_clear": (ctypes.c_int, [_PTR, _PTR]),
    "ash_map_clear_rows": (
        ctypes.c_int,
        [_PTR, ctypes.c_int, ctypes.POINTER(_PTR), ctypes.POINTER(_I64), _PTR],
    ),
    "ash_map_status": (ctypes.c_int, [_PTR, ctypes.POINTER(_I64), _PTR]),
    "ash_map_counters": (ctypes.c_int, [_PTR, _PTR, ctypes.POINTER(_I64), _PTR]),
    "ash_map_counters_pending": (ctypes.c_int, [_PTR]),
    "ash_map_known_size": (ctypes.c_int, [_PTR, ctypes.POINTER(_I64)]),
    "ash_map_set_staging": (ctypes.c_int, [_PTR, _PTR]),
    "ash_map_insert_scratch_bytes": (
        ctypes.c_int,
        [_PTR, _I64, ctypes.c_int, ctypes.POINTER(_I64), ctypes.c_int, ctypes.POINTER(_I64)],
    ),
    "ash_map_insert_auto": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, ctypes.c_int, ctypes.POINTER(_PTR), ctypes.POINTER(_PTR),
         ctypes.POINTER(_I64), _PTR, _I64, ctypes.c_int, _PTR, _PTR],
    ),
    "ash_map_erase_scratch_bytes": (
        ctypes.c_int, [_PTR, _I64, ctypes.c_int, ctypes.POINTER(_I64)]
    ),
    "ash_map_erase_auto": (ctypes.c_int, [_PTR, _PTR, _I64, _PTR, _I64, ctypes.c_int, _PTR]),
    "ash_map_upkeep": (ctypes.c_int, [_PTR, _I64, _PTR, _I64, _PTR, _PTR]),
    "ash_grid_collect_touched": (ctypes.c_int, [_PTR] * 6),
    "ash_map_size": (ctypes.c_int, [_PTR, ctypes.POINTER(_I64), _PTR]),
    "ash_map_items": (ctypes.c_int, [_PTR, _PTR, _PTR, _I64, _PTR]),
    "ash_map_items_rows": (
        ctypes.c_int,
        [_PTR, _PTR, _PTR, _I64, ctypes.c_int, ctypes.POINTER(_PTR), ctypes.POINTER(_PTR),
         ctypes.POINTER(_I64), ctypes.POINTER(_I64), _PTR],
    ),
    "ash_map_load": (ctypes.c_int, [_PTR, _PTR, _PTR, _I64, _PTR, _PTR]),
    "ash_map_should_rebuild": (ctypes.c_int, [_PTR, _I64, _I64, _I64]),
    "ash_map_rebuild": (ctypes.c_int, [_PTR, _PTR, _PTR, _I64, _PTR]),
    "ash_scatter_rows": (ctypes.c_int, [_PTR, _PTR, _PTR, _I64, _I64, _PTR]),
    "ash_gather_rows": (
        ctypes.c_int,
        [ctypes.c_int, ctypes.POINTER(_PTR), ctypes.POINTER(_PTR), ctypes.POINTER(_I64),
         ctypes.POINTER(_I64), _PTR, _I64, _PTR],
    ),
    "ash_map_find_rows": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, ctypes.c_int, ctypes.POINTER(_PTR), ctypes.POINTER(_PTR),
         ctypes.POINTER(_I64), ctypes.POINTER(_I64), ctypes.c_int, _PTR, _PTR, _PTR],
    ),
    "ash_map_find_rows_scratch_bytes": (
        _I64, [_PTR, _I64, ctypes.c_int, ctypes.POINTER(_I64), ctypes.POINTER(_I64)]
    ),
    "ash_map_find_rows_scratch": (
        ctypes.c_int,
        [_PTR, _PTR, _I64, ctypes.c_int, ctypes.POINTER(_PTR), ctypes.POINTER(_PTR),
         ctypes.POINTER(_I64), ctypes.POINTER(_I64), ctypes.c_int, _PTR, _PTR, _PTR, _I64, _PTR],
    ),
    "ash_add_rows": (
        ctypes.c_int,
        [_PTR, _PTR, _PTR, _I64, _I64, ctypes.c_int, _PTR, _I64, _PTR],
    ),
    "ash_isosurface_workspace_ints": (ctypes.c_int64, [_I64, _I64]),
    "ash_isosurface_classify": (
        ctypes.c_int,
        [_PTR] * 7 + [_I64] * 3
        + [ctypes.c_int, ctypes.c_float, ctypes.c_float, ctypes.c_int32] + [_PTR] * 3,
    ),
    "ash_isosurface_points": (
        ctypes.c_int,
        [_PTR] * 7 + [_I64] * 3 + [ctypes.c_int, ctypes.c_float, ctypes.c_int32]
        + [_PTR] * 2 + [_I64] + [_PTR] * 2,
    ),
    "ash_convolution_forward": (
        ctypes.c_int,
        [_PTR] * 9 + [_I64] * 6 + [ctypes.c_int32, _PTR],
    ),
    "ash_convolution_forward_listed": (
        ctypes.c_int,
        [_PTR] * 9 + [_I64] * 6 + [ctypes.c_int32, _PTR, _PTR],
    ),
    "ash_convolution_cube_supported": (
        ctypes.c_int, [_I64, ctypes.c_int, ctypes.c_int, _I64, ctypes.c_int32]
    ),
    "ash_convolution_cube": (
        ctypes.c_int,
        [_PTR] * 5 + [_I64, _I64, ctypes.c_int, ctypes.c_int, _I64, ctypes.c_int32, _PTR, _PTR],
    ),
    "ash_marching_cubes_workspace_ints": (ctypes.c_int64, [_I64, _I64]),
    "ash_marching_cubes_classify": (
        ctypes.c_int,
        [_PTR] * 7 + [_I64] * 3
        + [ctypes.c_int, ctypes.c_float, ctypes.c_float, ctypes.c_int32] + [_PTR] * 4,
    ),
    "ash_marching_cubes_extract": (
        ctypes.c_int,
        [_PTR] * 7 + [_I64] * 3 + [ctypes.c_int, ctypes.c_float, ctypes.c_int32]
        + [_PTR] * 3 + [_I64] * 2 + [_PTR] * 3,
    ),
    "ash_query_forward": (ctypes.c_int, [ctypes.POINTER(_QueryArgs), _PTR, _PTR]),
    "ash_query_backward_forward": (
        ctypes.c_int,
        [ctypes.POINTER(_QueryArgs), _PTR, _PTR, _PTR, _PTR],
    ),
    "ash_query_backward_backward": (
        ctypes.c_int,
        [ctypes.POINTER(_QueryArgs), _PTR, _PTR, _PTR, _PTR, _PTR],
    ),
    "ash_query_backward_forward_accumulate": (
        ctypes.c_int,
        [ctypes.POINTER(_QueryArgs), _PTR, _PTR, _PTR, _PTR],
    ),
    "ash_query_backward_both": (
        ctypes.c_int,
        [ctypes.POINTER(_QueryArgs)] + [_PTR] * 5 + [ctypes.c_int32, _PTR],
    ),
    "ash_query_backward_forward_scaled": (
        ctypes.c_int,
        [ctypes.POINTER(_QueryArgs), _PTR, _PTR, _PTR, _PTR, _PTR, ctypes.c_double, ctypes.c_int32, _PTR],
    ),
    "ash_query_backward_backward_scaled": (
        ctypes.c_int,
        [ctypes.POINTER(_QueryArgs), _PTR, _PTR, _PTR, _PTR, ctypes.c_double, ctypes.c_int32, _PTR],
    ),
    "ash_query_backward_backward_accumulate": (
        ctypes.c_int,
        [ctypes.POINTER(_QueryArgs), _PTR, _PTR, _PTR, _PTR, _PTR],
    ),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)

# Stamps of the tables' contents: a table takes a new one whenever its keys may
# have changed, and no two tables ever share one (a table made by `resize` may
# sit at the address of the one it replaces), so that what callers derive from
# the keys can be kept under the stamp alone.
_VERSIONS = itertools.count(1)

# Largest number of staged sample slots (rays x stride, 8 bytes each) for which
# ray_sample keeps the samples of its allocation pass; beyond it the march is
# run twice as in the reference.
RAY_STAGE_LIMIT = 1 << 30
# Staged slots per ray beyond max_samples_per_ray.
RAY_STAGE_EXTRA = 2
# Largest table whose touched rows ash_grid_collect_touched lists (the header's
# ASH_COLLECT_MAX_BLOCKS).
COLLECT_MAX_BLOCKS = 1 << 20
# Words of scratch for the count of a fusion frame (the header's ASH_FLAGGED_GROUPS).
FLAGGED_GROUPS = 8192
# Size of a second region that is attached before any key has asked for it
# (2^16 slots of 20 bytes).
GENERAL_JUST_IN_CASE_BYTES = 20 << 16
# Which inserts (and erases) take the streaming path of the library (batch split
# by bucket range, ranges handled in LDS) instead of the per-key kernel:
# "auto" = when the library says the batch is large enough relative to the
# table, "always" = whenever the path applies, "never".
BULK_INSERT = os.environ.get("ASH_BULK_INSERT", "auto")
BULK_ERASE = os.environ.get("ASH_BULK_ERASE", "auto")
_POLICY = {"auto": 0, "always": 1, "never": 2}   # the header's ASH_STREAMING_*
_INSERT_POLICY = {**_POLICY, "auto": 3}          # ... ASH_STREAMING_EARLY
NEEDS_GENERAL = 2                                # the header's ASH_NEEDS_GENERAL
_DTYPE = {torch.float32: 0, torch.float64: 1}


def library_path() -> str:
    return os.environ.get("ASH_HIP_LIBRARY", os.path.join(_LIB_DIR, _LIB_NAME))


def load_library(path: Optional[str] = None) -> ctypes.CDLL:
    """dlopen the C-ABI library and attach the prototypes."""
    lib = ctypes.CDLL(path or library_path())
    for name, (restype, argtypes) in _SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    return lib


def load_host(lib: ctypes.CDLL):
    """The native host module, calling into `lib`."""
    path = os.path.join(_LIB_DIR, _HOST_NAME)
    if not os.path.exists(path):
        raise OSError(f"{path} does not exist")
    spec = importlib.util.spec_from_file_location("_ash_host", path)
    host = importlib.util.module_from_spec(spec)
    try:
        spec.loader.exec_module(host)
    except ImportError as exc:
        raise OSError(f"{_HOST_NAME}: {exc}") from exc
    host.bind(lib._handle)
    return host


def _stream_of(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def _require_hip(t: torch.Tensor, what: str) -> None:
    if not t.is_cuda:
        raise RuntimeError(f"{what} must live on a HIP device, got {t.device}")


def stands_alone(t: torch.Tensor) -> bool:
    """Whether a kernel may take `t` by its address and a graph node of the
    package's own may stand for torch's operations on it.  Not for a subclass,
    inside a function transform (vmap and the like), with a forward-mode tangent
    or while a trace is recorded: there torch's operations have to be seen."""
    return (
        type(t) in (torch.Tensor, torch.nn.Parameter)
        and torch._C._functorch.peek_interpreter_stack() is None
        and not torch._C._is_tracing()
        and (forward_ad._current_level < 0 or forward_ad.unpack_dual(t).tangent is None)
    )


class _Backend:
    """Stands where the reference's `__ash` extension module stands."""

    def __init__(self, lib: ctypes.CDLL):
        self.lib = lib
        self.host = load_host(lib)
        backend = self

        class HashMap(_HashMap):
            _backend = backend

        self.HashMap = HashMap

    # -- error plumbing -------------------------------------------------
    def check(self, status: int) -> None:
        if status != 0:
            msg = self.lib.ash_last_error()
            raise RuntimeError(msg.decode() if msg else "libash_hip call failed")

    # -- iso-surface points (ash/src/pybind.cpp:30) --------------------------
    def isosurface_extraction(
        self, sdfs, weights, grid_indices, grid_coords_table, lut_grid_nb2grid_idx,
        cell_coords_table, lut_cell_nb2cell_idx, lut_cell_nb2grid_nb, grid_dim, iso_value,
        weight_thr,
    ) -> torch.Tensor:
        """Zero crossings of `sdfs - iso_value` on the +x/+y/+z edges of the
        listed blocks' cells, (P, 3) float32 in cell units, in the order of the
        listing."""
        _require_hip(sdfs, "sdfs")
        dev = sdfs.device
        if sdfs.dtype not in _DTYPE:
            raise RuntimeError("sdfs must be float32 or float64")
        b, m = sdfs.shape[0], sdfs.shape[1]
        sdfs = sdfs.reshape(b, m).contiguous()
        weights = weights.to(dev, sdfs.dtype).reshape(b, m).contiguous()
        gi = grid_indices.reshape(-1).to(dev, torch.int64).contiguous()
        gc = grid_coords_table.to(dev, torch.int32).contiguous()
        cc = cell_coords_table.to(dev, torch.int32).contiguous()
        lut_g = lut_grid_nb2grid_idx.to(dev, torch.int64).contiguous()
        lut_c2c = lut_cell_nb2cell_idx.to(dev, torch.int64).contiguous()
        lut_c2g = lut_cell_nb2grid_nb.to(dev, torch.int64).contiguous()
        if gc.shape != (b, 3) or cc.shape != (m, 3) or lut_g.shape != (b, 8):
            raise RuntimeError("coordinate / neighbour tables do not match the grid")
        if lut_c2c.shape != (m, 8) or lut_c2g.shape != (m, 8):
            raise RuntimeError("cell neighbour tables must be (cells_per_grid, 8)")
        flags = torch.empty(b * m, dtype=torch.uint8, device=dev)
        workspace = torch.empty(
            self.lib.ash_isosurface_workspace_ints(gi.numel(), m), dtype=torch.int32, device=dev
        )
        with torch.cuda.device(dev):
            self.check(
                self.lib.ash_isosurface_classify(
                    sdfs.data_ptr(), weights.data_ptr(), gi.data_ptr(), lut_g.data_ptr(),
                    cc.data_ptr(), lut_c2c.data_ptr(), lut_c2g.data_ptr(), gi.numel(), b, m,
                    int(grid_dim), float(iso_value), float(weight_thr), _DTYPE[sdfs.dtype],
                    flags.data_ptr(), workspace.data_ptr(), _stream_of(dev),
                )
            )
            n_points = int(workspace[0].item())
            positions = torch.empty((n_points, 3), dtype=torch.float32, device=dev)
            if n_points:
                self.check(
                    self.lib.ash_isosurface_points(
                        sdfs.data_ptr(), gi.data_ptr(), gc.data_ptr(), lut_g.data_ptr(),
                        cc.data_ptr(), lut_c2c.data_ptr(), lut_c2g.data_ptr(), gi.numel(), b, m,
                        int(grid_dim), float(iso_value), _DTYPE[sdfs.dtype], flags.data_ptr(),
                        workspace.data_ptr(), n_points, positions.data_ptr(), _stream_of(dev),
                    )
                )
        return positions

    # -- marching cubes (ash/src/pybind.cpp:31) ------------------------------
    def marching_cubes(
        self, sdfs, weights, grid_indices, grid_coords_table, lut_grid_nb2grid_idx,
        cell_coords_table, lut_cell_nb2cell_idx, lut_cell_nb2grid_nb, grid_dim, iso_value,
        weight_thr,
    ) -> Tuple[torch.Tensor, torch.Tensor]:
        """Triangle mesh of the surface `sdfs == iso_value` over the listed
        blocks: (triangles int32 (T, 3), vertices float32 (V, 3) in cell units).
        A cell contributes when its eight corners exist and weigh at least
        `weight_thr`.  Vertices and triangles follow the order of `grid_indices`."""
        _require_hip(sdfs, "sdfs")
        dev = sdfs.device
        if sdfs.dtype not in _DTYPE:
            raise RuntimeError("sdfs must be float32 or float64")
        b, m = sdfs.shape[0], sdfs.shape[1]
        sdfs = sdfs.reshape(b, m).contiguous()
        weights = weights.to(dev, sdfs.dtype).reshape(b, m).contiguous()
        gi = grid_indices.reshape(-1).to(dev, torch.int64).contiguous()
        gc = grid_coords_table.to(dev, torch.int32).contiguous()
        cc = cell_coords_table.to(dev, torch.int32).contiguous()
        lut_g = lut_grid_nb2grid_idx.to(dev, torch.int64).contiguous()
        lut_c2c = lut_cell_nb2cell_idx.to(dev, torch.int64).contiguous()
        lut_c2g = lut_cell_nb2grid_nb.to(dev, torch.int64).contiguous()
        if gc.shape != (b, 3) or cc.shape != (m, 3) or lut_g.shape != (b, 8):
            raise RuntimeError("coordinate / neighbour tables do not match the grid")
        if lut_c2c.shape != (m, 8) or lut_c2g.shape != (m, 8):
            raise RuntimeError("cell neighbour tables must be (cells_per_grid, 8)")
        cases = torch.empty(b * m, dtype=torch.uint8, device=dev)
        slots = torch.empty(b * m, dtype=torch.int32, device=dev)
        counters = torch.empty(
            self.lib.ash_marching_cubes_workspace_ints(gi.numel(), m), dtype=torch.int32, device=dev
        )
        with torch.cuda.device(dev):
            self.check(
                self.lib.ash_marching_cubes_classify(
                    sdfs.data_ptr(), weights.data_ptr(), gi.data_ptr(), lut_g.data_ptr(),
                    cc.data_ptr(), lut_c2c.data_ptr(), lut_c2g.data_ptr(), gi.numel(), b, m,
                    int(grid_dim), float(iso_value), float(weight_thr), _DTYPE[sdfs.dtype],
                    cases.data_ptr(), slots.data_ptr(), counters.data_ptr(), _stream_of(dev),
                )
            )
            n_triangles, n_vertices = counters[:2].tolist()
            triangles = torch.empty((n_triangles, 3), dtype=torch.int32, device=dev)
            vertices = torch.empty((n_vertices, 3), dtype=torch.float32, device=dev)
            if n_vertices:
                self.check(
                    self.lib.ash_marching_cubes_extract(
                        sdfs.data_ptr(), gi.data_ptr(), gc.data_ptr(), lut_g.data_ptr(),
                        cc.data_ptr(), lut_c2c.data_ptr(), lut_c2g.data_ptr(), gi.numel(), b, m,
                        int(grid_dim), float(iso_value), _DTYPE[sdfs.dtype], cases.data_ptr(),
                        slots.data_ptr(), counters.data_ptr(), n_vertices, n_triangles,
                        vertices.data_ptr(), triangles.data_ptr() if n_triangles else None,
                        _stream_of(dev),
                    )
                )
        return triangles, vertices

    def surface_mesh_block8(
        self, hashmap, sdfs, weights, grid_indices, grid_coords_table, lut_grid_nb2grid_idx,
        grid_dim, iso_value, weight_thr, to_world,
    ):
        """marching_cubes for blocks of 8^3 cells and the tables that
        SparseDenseGrid builds (the per-cell ones are then not needed), or None
        for other block sizes.  `sdfs` and `weights` may be channels of wider
        rows; `to_world`: (scale, origin or None) to apply to the vertices, or
        None."""
        if int(grid_dim) != 8 or sdfs.dtype not in _DTYPE:
            return None
        _require_hip(sdfs, "sdfs")
        dev = sdfs.device
        b = sdfs.shape[0]

        def channel(t):
            t = t.reshape(b, 512)
            step = t.stride(1)
            return t if t.stride(0) == 512 * step and 1 <= step <= 64 else t.contiguous()

        scale, origin = (1.0, None) if to_world is None else to_world
        return self.host.surface_mesh(
            hashmap._address, hashmap._index, channel(sdfs), channel(weights.to(dev, sdfs.dtype)),
            grid_indices.reshape(-1).to(dev, torch.int64).contiguous(),
            grid_coords_table.to(dev, torch.int32).contiguous(),
            lut_grid_nb2grid_idx.to(dev, torch.int64).contiguous(), float(iso_value),
            float(weight_thr), to_world is not None, scale, origin)

    # -- sparse convolution (ash/src/pybind.cpp:33) -------------------------
    def convolution_forward(
        self, inputs, weights, masks, grid_indices, cell_indices, lut_grid_nb2grid_idx,
        lut_cell_nb2cell_idx, lut_cell_nb2grid_nb, grid_dim,
    ) -> torch.Tensor:
        """outputs[row] = sum over window taps k of inputs[row of neighbour k] *
        weights[k], per channel; same shape as `inputs`, zero rows for blocks
        that are not listed."""
        _require_hip(inputs, "inputs")
        dev = inputs.device
        if inputs.dtype not in _DTYPE or inputs.dim() != 3 or not inputs.is_contiguous():
            raise RuntimeError("inputs must be contiguous float32/float64 (B, M, E)")
        b, m, e = inputs.shape
        weights = weights.to(dev, inputs.dtype).contiguous()
        lut_g = lut_grid_nb2grid_idx.to(dev, torch.int64).contiguous()
        lut_c2c = lut_cell_nb2cell_idx.to(dev, torch.int64).contiguous()
        lut_c2g = lut_cell_nb2grid_nb.to(dev, torch.int64).contiguous()
        k = lut_c2c.shape[1]
        if weights.shape != (k, e):
            raise RuntimeError(f"weights must be ({k}, {e}), got {tuple(weights.shape)}")
        if lut_c2c.shape != (m, k) or lut_c2g.shape != (m, k) or lut_g.shape[0] != b:
            raise RuntimeError("neighbour tables do not match the inputs")
        gi = grid_indices.reshape(-1).to(dev, torch.int64).contiguous()
        ci = cell_indices.reshape(-1).to(dev, torch.int64).contiguous()
        if ci.numel() != m:
            raise RuntimeError("cell_indices must list every cell of a block")
        masks = masks.to(dev, torch.bool).contiguous()
        if masks.numel() < gi.numel() * m:
            raise RuntimeError("masks must cover every listed cell")
        outputs = torch.empty_like(inputs)
        # one scratch byte per block: the library then clears only the rows of
        # the blocks that are not listed
        listed = torch.empty(b, dtype=torch.uint8, device=dev)
        with torch.cuda.device(dev):
            self.check(
                self.lib.ash_convolution_forward_listed(
                    inputs.data_ptr(), weights.data_ptr(), masks.data_ptr(), gi.data_ptr(),
                    ci.data_ptr(), lut_g.data_ptr(), lut_c2c.data_ptr(), lut_c2g.data_ptr(),
                    outputs.data_ptr(), gi.numel(), b, m, e, k, lut_g.shape[1],
                    _DTYPE[inputs.dtype], listed.data_ptr(), _stream_of(dev),
                )
            )
        return outputs

    def convolution_cube(self, inputs, weights, grid_indices, lut_grid_nb2grid_idx, grid_dim):
        """convolution_forward of every cell of the listed blocks for a cube
        window and the tables that SparseDenseGrid builds (of which only the
        per-block one is needed), or None for sizes that
        `convolution_forward` takes."""
        b, m, e = inputs.shape
        window = weights.shape[0]
        if inputs.dtype not in _DTYPE or not self.lib.ash_convolution_cube_supported(
            b, grid_dim, window, e, _DTYPE[inputs.dtype]
        ) or inputs.data_ptr() % 16:
            return None
        _require_hip(inputs, "inputs")
        dev = inputs.device
        if not inputs.is_contiguous() or m != grid_dim**3:
            raise RuntimeError("inputs must be contiguous (B, grid_dim^3, E)")
        weights = weights.to(dev, inputs.dtype).contiguous()
        if weights.shape != (window, window, window, e):
            raise RuntimeError(f"weights must be ({window}, {window}, {window}, {e})")
        lut_g = lut_grid_nb2grid_idx.to(dev, torch.int64).contiguous()
        if lut_g.shape != (b, 27):
            raise RuntimeError("neighbour table does not match the inputs")
        gi = grid_indices.reshape(-1).to(dev, torch.int64).contiguous()
        outputs = torch.empty_like(inputs)
        listed = torch.empty(b, dtype=torch.uint8, device=dev)
        self.check(
            self.lib.ash_convolution_cube(
                inputs.data_ptr(), weights.data_ptr(), gi.data_ptr(), lut_g.data_ptr(),
                outputs.data_ptr(), gi.numel(), b, grid_dim, window, e, _DTYPE[inputs.dtype],
                listed.data_ptr(), _stream_of(dev),
            )
        )
        return outputs

    # -- rays (ash/src/pybind.cpp:35-37) ----------------------------------
    @staticmethod
    def _rays(hashmap, ray_origins, ray_directions):
        dev = hashmap.device()
        o = ray_origins.to(dev, torch.float32).contiguous()
        d = ray_directions.to(dev, torch.float32).contiguous()
        if o.dim() != 2 or o.shape[1] != 3 or d.shape != o.shape:
            raise RuntimeError("ray origins and directions must both be (N, 3)")
        return dev, o, d

    def ray_find_near_far(
        self, hashmap, ray_origins, ray_directions, bbox_min, bbox_max, t_min, t_max, t_step,
        grid2cell_multiplier,
    ) -> Tuple[torch.Tensor, torch.Tensor]:
        """Per ray, the parameter range that contains active blocks (cell
        units); near = -1 where the ray meets none."""
        dev, o, d = self._rays(hashmap, ray_origins, ray_directions)
        lo = bbox_min.to(dev, torch.float32).contiguous()
        hi = bbox_max.to(dev, torch.float32).contiguous()
        n = o.shape[0]
        nears = torch.zeros(n, dtype=torch.float32, device=dev)
        fars = torch.zeros(n, dtype=torch.float32, device=dev)
        with torch.cuda.device(dev):
            self.check(
                self.lib.ash_ray_find_near_far(
                    hashmap._handle, o.data_ptr(), d.data_ptr(), lo.data_ptr(), hi.data_ptr(), n,
                    float(t_min), float(t_max), float(t_step), float(grid2cell_multiplier),
                    nears.data_ptr(), fars.data_ptr(), _stream_of(dev),
                )
            )
        return nears, fars

    def ray_find_near_far_world(
        self, hashmap, ray_origins, ray_directions, origin, cell_size, bbox_min, bbox_max, t_min,
        t_max, grid2cell_multiplier, block_bounds=(0, -1),
    ) -> Tuple[torch.Tensor, torch.Tensor]:
        """ray_find_near_far of world rays with cell units = (x - origin) /
        cell_size: the transforms of rays, box and results in the same launch
        (t_min and t_max in cell units).  block_bounds: where the blocks of the
        grid lie (lo, hi; a range that is small enough speeds the look-ups up)."""
        return self.host.ray_near_far(hashmap._address, hashmap._index, hashmap._volumes, ray_origins, ray_directions,
                                      origin, cell_size, bbox_min, bbox_max, t_min, t_max,
                                      grid2cell_multiplier, *block_bounds)

    def ray_sample_world(
        self, hashmap, ray_origins, ray_directions, origin, cell_size, ray_nears, ray_fars,
        max_samples_per_ray, grid2cell_multiplier, block_bounds=(0, -1),
    ):
        """ray_sample of world rays, everything in world units; None where the
        samples do not fit a staging area (`ray_sample` takes such rays)."""
        stride = max(1, int(max_samples_per_ray) + RAY_STAGE_EXTRA)
        if ray_origins.shape[0] * stride > RAY_STAGE_LIMIT:
            return None
        return self.host.ray_sample(hashmap._address, hashmap._index, hashmap._volumes, ray_origins, ray_directions,
                                    origin, cell_size, ray_nears, ray_fars, int(max_samples_per_ray),
                                    grid2cell_multiplier, stride, *block_bounds)

    def ray_sample(
        self, hashmap, ray_origins, ray_directions, ray_nears, ray_fars, bbox_min, bbox_max,
        max_samples_per_ray, grid2cell_multiplier,
    ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
        """(ray_indices int64[M], t_nears fp32[M], t_fars fp32[M], inclusive
        prefix sum of the per-ray sample counts int64[N])."""
        dev, o, d = self._rays(hashmap, ray_origins, ray_directions)
        n = o.shape[0]

        def per_ray(t):
            if not torch.is_tensor(t):
                return torch.full((n,), float(t), dtype=torch.float32, device=dev)
            return t.to(dev, torch.float32).expand(n).contiguous()

        nears, fars = per_ray(ray_nears), per_ray(ray_fars)
        counts = torch.zeros(n, dtype=torch.int64, device=dev)
        fixed = (hashmap._handle, o.data_ptr(), d.data_ptr(), nears.data_ptr(), fars.data_ptr(), n,
                 int(max_samples_per_ray), float(grid2cell_multiplier))
        # One march: the allocation pass keeps its samples, the assignment pass
        # copies them.  A ray takes at most max_samples steps of its own size
        # (+ rounding), so the staging stride below is never exceeded; the
        # two-march path of the reference remains for the case that it is.
        stride = max(1, int(max_samples_per_ray) + RAY_STAGE_EXTRA)
        staged = n * stride <= RAY_STAGE_LIMIT
        if staged:
            stage = torch.empty((n, stride, 2), dtype=torch.float32, device=dev)
            with torch.cuda.device(dev):
                self.check(
                    self.lib.ash_ray_sample_staged(*fixed, counts.data_ptr(), stage.data_ptr(),
                                                   stride, _stream_of(dev))
                )
        else:
            with torch.cuda.device(dev):
                self.check(
                    self.lib.ash_ray_sample(*fixed, counts.data_ptr(), None, None, None, None,
                                            _stream_of(dev))
                )
        prefix = torch.cumsum(counts, 0)
        if n:
            total, most = torch.stack([prefix[-1], counts.max()]).tolist()
        else:
            total, most = 0, 0
        ray_indices = torch.empty(total, dtype=torch.int64, device=dev)
        t_nears = torch.empty(total, dtype=torch.float32, device=dev)
        t_fars = torch.empty(total, dtype=torch.float32, device=dev)
        if total:
            with torch.cuda.device(dev):
                if staged and most <= stride:
                    self.check(
                        self.lib.ash_ray_sample_compact(
                            counts.data_ptr(), prefix.data_ptr(), stage.data_ptr(), stride, n,
                            ray_indices.data_ptr(), t_nears.data_ptr(), t_fars.data_ptr(),
                            _stream_of(dev),
                        )
                    )
                else:
                    self.check(
                        self.lib.ash_ray_sample(
                            *fixed, None, prefix.data_ptr(), ray_indices.data_ptr(),
                            t_nears.data_ptr(), t_fars.data_ptr(), _stream_of(dev),
                        )
                    )
        return ray_indices, t_nears, t_fars, prefix

    # -- depth integration (no pybind counterpart: the reference's demo does
    #    this with torch expressions, demo/rgbd_fusion.py:76-110,216-254) -----
    def integrate_depth(
        self,
        embeddings: torch.Tensor,
        grid_indices: torch.Tensor,
        grid_coords: torch.Tensor,
        grid_dim: int,
        cell_size: float,
        origin: Optional[torch.Tensor],
        intrinsic: torch.Tensor,
        extrinsic: torch.Tensor,
        depth: torch.Tensor,
        color: Optional[torch.Tensor],
        trunc: float,
        depth_max: float,
        counted_by=None,
        flagged_by=None,
    ) -> None:
        """In-place TSDF update of the cells of the listed blocks.  With
        `counted_by` (a map whose latest deferred activation made the listing)
        the number of listed blocks is read on the device; with `flagged_by` (a
        map whose latest `activate_positions` left flags) there is no listing
        and the kernel goes by the map's flags, which it takes down."""
        _require_hip(embeddings, "embeddings")
        dev = embeddings.device
        if embeddings.dtype != torch.float32 or not embeddings.is_contiguous():
            raise RuntimeError("embeddings must be contiguous float32")
        if embeddings.dim() != 3 or embeddings.shape[1] != grid_dim**3:
            raise RuntimeError("embeddings must be (num_embeddings, grid_dim^3, embedding_dim)")
        if flagged_by is not None:
            if flagged_by._device != dev or getattr(flagged_by, "_touched", None) is None:
                raise RuntimeError("no activation has flagged rows of this map on this device")
            if embeddings.shape[0] < flagged_by.capacity:
                raise RuntimeError("one embedding row per index of the map is needed")
        else:
            grid_indices = grid_indices.reshape(-1).to(dev, torch.int64).contiguous()
            grid_coords = grid_coords.reshape(-1, 3).to(dev, torch.int32).contiguous()
            if grid_coords.shape[0] != grid_indices.shape[0]:
                raise RuntimeError("one coordinate row per block index is needed")
        if counted_by is not None and grid_indices.shape[0] != counted_by.capacity:
            raise RuntimeError("a listing counted on the device has one row per block of the map")
        intrinsic = intrinsic.to(dev, torch.float32).contiguous()
        extrinsic = extrinsic.to(dev, torch.float32).contiguous()
        if intrinsic.shape != (3, 3) or extrinsic.shape != (4, 4):
            raise RuntimeError("intrinsic must be 3x3 and extrinsic 4x4")
        depth = depth.to(dev, torch.float32).contiguous()
        if depth.dim() != 2:
            raise RuntimeError("depth must be (H, W)")
        if color is not None:
            color = color.to(dev, torch.float32).contiguous()
            if color.shape != (*depth.shape, 3):
                raise RuntimeError("color must be (H, W, 3)")
        c_origin = None
        if origin is not None:
            c_origin = (ctypes.c_float * 3)(*[float(v) for v in origin.reshape(-1).tolist()])
        tail = (float(cell_size), c_origin, intrinsic.data_ptr(), extrinsic.data_ptr(),
                depth.data_ptr(), color.data_ptr() if color is not None else None,
                depth.shape[0], depth.shape[1], float(trunc), float(depth_max), _stream_of(dev))
        with torch.cuda.device(dev):
            if flagged_by is not None:
                self.check(
                    self.lib.ash_grid_integrate_depth_flagged(
                        flagged_by._handle, embeddings.data_ptr(), embeddings.shape[0],
                        int(grid_dim), embeddings.shape[2], flagged_by._touched.data_ptr(),
                        flagged_by._block_coords.data_ptr(), *tail,
                    )
                )
            elif counted_by is not None:
                self.check(
                    self.lib.ash_grid_integrate_depth_touched(
                        counted_by._handle, embeddings.data_ptr(), embeddings.shape[0],
                        int(grid_dim), embeddings.shape[2], grid_indices.data_ptr(),
                        grid_coords.data_ptr(), *tail,
                    )
                )
            else:
                self.check(
                    self.lib.ash_grid_integrate_depth(
                        embeddings.data_ptr(), embeddings.shape[0], int(grid_dim),
                        embeddings.shape[2], grid_indices.data_ptr(), grid_coords.data_ptr(),
                        grid_indices.shape[0], *tail,
                    )
                )

    # -- value rows by index (ash/hashmap.py:87-95,138-146) -------------------
    def gather_rows(self, tables: Dict[str, torch.Tensor], indices: Optional[torch.Tensor],
                    first: int = 0) -> Dict[str, torch.Tensor]:
        """{name: table[indices]} for value tables on a HIP device, four tables
        per launch; with indices None, {name: copy of table[:first]}.  Tables
        the kernel does not take (rows that are not a multiple of 4 bytes,
        non-contiguous storage) are indexed by torch."""
        out: Dict[str, torch.Tensor] = {}
        names, batch = [], []
        n = indices.numel() if indices is not None else int(first)
        for name, table in tables.items():
            fits = (table.is_cuda and table.is_contiguous() and table.numel() > 0
                    and table.numel() // table.shape[0] * table.element_size() % 4 == 0
                    and not table.requires_grad
                    and (indices is None
                         or (indices.device == table.device and indices.dtype == torch.int64)))
            if fits:
                names.append(name)
                batch.append(table)
            else:
                out[name] = table[indices.reshape(-1)] if indices is not None else table[:n].clone()
        if batch:
            out.update(zip(names, self.host.gather_rows(batch, indices, n)))
        return {name: out[name] for name in tables}

    # -- look-up with rows (ash/hashmap.py:82-95, ash/embedding.py:30-38) -----
    def finds_rows_of(self, tables, device) -> bool:
        """Whether `find_rows` takes these tables (a list of tensors)."""
        return self.host.finds_rows_of(tables, device.index)

    def find_rows(self, hashmap, keys, tables, zero_misses: bool = False,
                  need_indices: bool = True):
        """(indices or None, masks, [table[indices] for each table]) in one
        launch, large batches on several tables in three with scratch memory;
        rows of keys that are not stored are row 0 of the table, or zeros with
        `zero_misses`."""
        return self.host.find_rows(hashmap._address, hashmap.key_dim, hashmap._index, keys, tables,
                                   zero_misses, need_indices)

    def embedding_rows(self, hashmap, keys, embedding) -> torch.Tensor:
        """Rows of `embedding` under `keys`, zeros for keys that are not stored;
        differentiable, to any order, with respect to the embedding."""
        return self.host.embedding_rows(embedding, hashmap._address, hashmap.key_dim, hashmap._index, keys)

    # -- trilinear queries (ash/src/pybind.cpp:25-29) ---------------------
    def query_forward(
        self,
        embeddings,
        offsets,
        grid_indices,
        cell_indices,
        masks,
        lut_grid_nb2grid_idx,
        lut_cell_nb2cell_idx,
        lut_cell_nb2grid_nb,
        grid_dim,
        interpolation,
    ) -> torch.Tensor:
        return self.host.query_forward(
            [embeddings, offsets, grid_indices, cell_indices, masks, lut_grid_nb2grid_idx,
             lut_cell_nb2cell_idx, lut_cell_nb2grid_nb], interpolation)

    def grid_forward(
        self,
        hashmap,
        x,
        embeddings,
        lut_grid_nb2grid_idx,
        lut_cell_nb2cell_idx,
        lut_cell_nb2grid_nb,
        grid_dim,
        interpolation,
        need_operands: bool = True,
        origin: Optional[torch.Tensor] = None,
        cell_size: float = 1.0,
    ):
        """`SparseDenseGrid.query` and `query_forward` in one kernel: positions x
        (float32 (N, 3); cell units = (x - origin) / cell_size, evaluated as
        torch does on the device) -> (features (N, E), masks (N,),
        grid_indices, cell_indices, offsets).  The last three are what a
        backward pass needs; with need_operands False they are not produced
        (None)."""
        return self.host.grid_forward(
            hashmap._address, hashmap._index, x, embeddings, lut_grid_nb2grid_idx,
            lut_cell_nb2cell_idx, lut_cell_nb2grid_nb, grid_dim, interpolation, need_operands,
            origin, cell_size)

    def query_backward_forward(
        self,
        z,
        embeddings,
        offsets,
        grid_indices,
        cell_indices,
        masks,
        lut_grid_nb2grid_idx,
        lut_cell_nb2cell_idx,
        lut_cell_nb2grid_nb,
        grid_dim,
        interpolation,
        need_embeddings: bool = True,
        need_offsets: bool = True,
        accumulate_into: Optional[torch.Tensor] = None,
        along=(),
        cell_size: float = 1.0,
    ) -> Tuple[Optional[torch.Tensor], Optional[torch.Tensor]]:
        """(grad_embeddings, grad_offsets); an output that is not needed is
        None and its work (for grad_embeddings: dense zero fill + atomics) is
        skipped.  With `accumulate_into` (a gradient of the embeddings' shape
        that already holds other contributions) the embedding gradient is added
        to that tensor, which is also what is returned.  `along`: what
        query_backward_backward has put off for the same queries, pairs
        (grad_grad_offsets, z), taken along in grad_embeddings -- the first pair
        in the same pass over the queries.  `cell_size`: the offsets are positions
        divided by it, and the gradients with respect to the offsets, here and in
        `along`, are those with respect to the positions."""
        operands = [embeddings, offsets, grid_indices, cell_indices, masks, lut_grid_nb2grid_idx,
                    lut_cell_nb2cell_idx, lut_cell_nb2grid_nb]
        if not along:
            return self.host.query_backward_forward(
                z, operands, interpolation, need_embeddings, need_offsets, accumulate_into, cell_size)
        grad_embeddings, grad_offsets = self.host.query_backward_both(
            z, *along[0], operands, interpolation, need_offsets, accumulate_into, cell_size)
        for pair in along[1:]:
            self.host.query_backward_backward(*pair, operands, interpolation, False, True, grad_embeddings,
                                              cell_size)
        return grad_embeddings, grad_offsets

    def query_backward_forward_onto(self, grad_embeddings, z, *operands, need_offsets: bool = True, **along):
        """query_backward_forward whose embedding gradient is added to
        `grad_embeddings`, a tensor that no one else holds; returns
        grad_offsets."""
        return _Backend.query_backward_forward(self, z, *operands, need_offsets=need_offsets,
                                               accumulate_into=grad_embeddings, **along)[1]

    def query_backward_backward_onto(self, grad_embeddings, grad_grad_offsets, z, *operands,
                                     cell_size: float = 1.0) -> None:
        """query_backward_backward with no other result than an embedding
        gradient added to `grad_embeddings`."""
        _Backend.query_backward_backward(self, None, grad_grad_offsets, z, *operands, need_z=False,
                                         accumulate_into=grad_embeddings, need_offsets=False,
                                         cell_size=cell_size)

    def query_backward_backward(
        self,
        grad_grad_embeddings,
        grad_grad_offsets,
        z,
        embeddings,
        offsets,
        grid_indices,
        cell_indices,
        masks,
        lut_grid_nb2grid_idx,
        lut_cell_nb2cell_idx,
        lut_cell_nb2grid_nb,
        grid_dim,
        interpolation,
        need_z: bool = True,
        need_embeddings: bool = True,
        accumulate_into: Optional[torch.Tensor] = None,
        need_offsets: bool = True,
        later: bool = False,
        cell_size: float = 1.0,
    ) -> Tuple[Optional[torch.Tensor], Optional[torch.Tensor], Optional[torch.Tensor]]:
        """(grad_z, grad_embeddings, zero grad_offsets); outputs that are not
        needed are None and their work is skipped.  `accumulate_into` as for
        query_backward_forward.  `later`: grad_embeddings comes without the
        contributions of this call (zeros, or `accumulate_into` as it is); the
        caller has query_backward_forward or query_backward_backward_onto add
        them.  There is no grad_z then.  `cell_size` as there."""
        operands = [embeddings, offsets, grid_indices, cell_indices, masks, lut_grid_nb2grid_idx,
                    lut_cell_nb2cell_idx, lut_cell_nb2grid_nb]
        if later:
            grad_z, grad_embeddings = None, self.host.query_gradient_later(
                grad_grad_offsets, z, operands, interpolation, accumulate_into)
        else:
            grad_z, grad_embeddings = self.host.query_backward_backward(
                grad_grad_offsets, z, operands, interpolation, need_z, need_embeddings, accumulate_into,
                cell_size)
        # the offsets second-order term is not produced (ash/src/grid.cu:417-418)
        zeros = embeddings.new_zeros(grid_indices.shape[0], 3) if need_offsets else None
        return grad_z, grad_embeddings, zeros

    # for callers that drop the zero grad_offsets above
    WITHOUT_OFFSETS = {"need_offsets": False}
    # the backward functions take `cell_size`
    TAKES_CELL_SIZE = True


class _HashMap:
    """Same surface as the pybind class `HashMap` (ash/src/pybind.cpp:9-23).

    Owns the table workspace as torch tensors and a native handle.  `heap` is
    the caller's int32[capacity] buffer and is mutated in place by the kernels.
    Which insert path a batch takes, the upkeep of the table and what is known
    of its counters on the host are the library's business (ash_map_insert_auto,
    ash_map_counters); this class allocates what the calls ask for.
    """

    _backend: "_Backend" = None
    _COUNTERS = ("size", "dropped", "tombstones", "exotic_pending", "load_duplicates", "touched",
                 "general_live")

    def __init__(self, key_dim: int, capacity: int, heap: torch.Tensor, device):
        device = torch.device(device)
        if device.type != "cuda":
            # the reference has no CPU map either (ash/src/hashmap_cpu.cpp:8)
            raise RuntimeError("Not implemented: ash hash maps exist on HIP devices only")
        if heap.dtype != torch.int32 or heap.numel() != capacity or not heap.is_contiguous():
            raise RuntimeError("heap must be a contiguous int32 tensor of `capacity` elements")
        _require_hip(heap, "heap")
        lib = self._backend.lib
        self._lib = lib
        self._handle = None
        self._device = heap.device
        self.key_dim = int(key_dim)
        self.capacity = int(capacity)
        self._heap = heap
        table_bytes, general_bytes = _I64(0), _I64(0)
        self._check(
            lib.ash_map_workspace_bytes(
                self.key_dim, self.capacity, ctypes.byref(table_bytes), ctypes.byref(general_bytes)
            )
        )
        self._general_bytes = general_bytes.value
        self._table = torch.empty(table_bytes.value, dtype=torch.uint8, device=self._device)
        self._general = None
        # counts the calls that may have changed the stored keys; lets callers
        # keep results derived from the key set (orderings, tables) while it stands
        self.version = next(_VERSIONS)
        handle = _PTR()
        with torch.cuda.device(self._device):
            self._check(
                lib.ash_map_create(
                    self.key_dim,
                    self.capacity,
                    heap.data_ptr(),
                    self._table.data_ptr(),
                    table_bytes.value,
                    self._device.index,
                    self._stream(),
                    ctypes.byref(handle),
                )
            )
        self._handle = handle
        self._address, self._index = handle.value, self._device.index
        self._volumes = self._backend.host.Volumes()

    def __del__(self):
        handle, self._handle = getattr(self, "_handle", None), None
        if handle:
            # (waits for counters that the device is still to leave on the host)
            self._lib.ash_map_destroy(handle)

    # -- helpers ---------------------------------------------------------
    def _check(self, status: int) -> None:
        self._backend.check(status)

    def _stream(self) -> int:
        return _stream_of(self._device)

    def _keys(self, keys: torch.Tensor) -> torch.Tensor:
        if keys.dim() != 2 or keys.shape[1] != self.key_dim:
            raise RuntimeError(f"keys must be (N, {self.key_dim}), got {tuple(keys.shape)}")
        if keys.device != self._device:
            raise RuntimeError(f"keys are on {keys.device}, the map on {self._device}")
        return keys.to(torch.int32).contiguous()

    def _scratch(self, nbytes: int) -> Optional[torch.Tensor]:
        return torch.empty(nbytes, dtype=torch.uint8, device=self._device) if nbytes else None

    def _attach_general(self, just_in_case: bool = False) -> None:
        """Hands the table its second region (keys that do not fit the packed
        code live there): sized for the capacity once such a key has shown up,
        or -- `just_in_case`, ahead of time by a path that cannot come back for
        it -- for a few thousand of them."""
        if self._general is not None:
            raise RuntimeError("internal error: unpackable keys pending with region attached")
        nbytes = min(self._general_bytes, GENERAL_JUST_IN_CASE_BYTES) if just_in_case \
            else self._general_bytes
        self._general = torch.empty(nbytes, dtype=torch.uint8, device=self._device)
        with torch.cuda.device(self._device):
            self._check(
                self._lib.ash_map_attach_general(
                    self._handle, self._general.data_ptr(), nbytes, self._stream()
                )
            )

    def _upkeep(self, incoming: int) -> None:
        """Before the entry points that insert without ash_map_insert_auto."""
        nbytes = _I64(0)
        self._check(self._lib.ash_map_insert_scratch_bytes(
            self._handle, 0, 0, None, _POLICY["never"], ctypes.byref(nbytes)))
        scratch = self._scratch(nbytes.value)
        with torch.cuda.device(self._device):
            self._check(self._lib.ash_map_upkeep(
                self._handle, incoming, scratch.data_ptr() if scratch is not None else None,
                nbytes.value, None, self._stream()))

    # -- pybind surface --------------------------------------------------
    def device(self) -> torch.device:
        return self._device

    def counters(self) -> Dict[str, int]:
        """The table's counters as the handle knows them; copied from the
        device only when no earlier call has left them on the host."""
        return dict(zip(self._COUNTERS, self._read_counters()))

    def _read_counters(self):
        return self._backend.host.counters(self._address, self._index)

    def status(self) -> Dict[str, int]:
        """The counters by a copy from the device, whatever the handle knows."""
        out = (_I64 * 5)()
        with torch.cuda.device(self._device):
            self._check(self._lib.ash_map_status(self._handle, out, self._stream()))
        fresh = dict(zip(self._COUNTERS[:5], out))
        fresh.update({k: v for k, v in self.counters().items() if k not in fresh})
        return fresh

    def status_after_insert(self) -> Dict[str, int]:
        """The counters after the latest insert: every insert reads them (or
        queues their read-back), which saves the caller a read-back of its own."""
        return self.counters()

    @property
    def counters_queued(self) -> bool:
        """Whether the latest insert returned with the read-back of the
        counters still queued behind it."""
        return bool(self._lib.ash_map_counters_pending(self._handle))

    def known_size(self) -> Optional[int]:
        """The size if it is known on the host (from the latest read-back, or
        zero after a clear), else None; never asks the device for it."""
        n = _I64(0)
        rc = self._lib.ash_map_known_size(self._handle, ctypes.byref(n))
        if rc < 0:
            self._check(1)
        return n.value if rc == 1 else None

    def size(self) -> int:
        return self._read_counters()[0]

    def find(self, keys: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
        return self._backend.host.find(self._address, self.key_dim, self._index, keys)

    def query_cells(
        self, x: torch.Tensor, grid_dim: int
    ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
        """Fused front end of `SparseDenseGrid.query`: positions in cell units ->
        (grid_indices, cell_indices, offsets, masks) in one kernel."""
        return self._backend.host.query_cells(self._address, self._index, x, grid_dim)

    def _activation_buffers(self, cells: torch.Tensor) -> torch.Tensor:
        if self.key_dim != 3:
            raise RuntimeError("block activation needs 3-d keys")
        if cells.dim() != 2 or cells.shape[1] != 3 or cells.dtype != torch.float32:
            raise RuntimeError("positions must be float32 (N, 3)")
        if cells.device != self._device:
            raise RuntimeError(f"positions are on {cells.device}, the map on {self._device}")
        if getattr(self, "_touched", None) is None:
            self._touched = torch.zeros(self.capacity, dtype=torch.uint8, device=self._device)
            self._block_coords = torch.zeros(
                (self.capacity, 3), dtype=torch.int32, device=self._device
            )
        return cells.contiguous()

    def activate_blocks(
        self,
        cells: torch.Tensor,
        grid_dim: int,
        dilation: int,
        bidirectional: bool,
        bound_lo: int,
        bound_hi: int,
    ) -> Tuple[torch.Tensor, torch.Tensor]:
        """Fused body of `SparseDenseGrid.spatial_init_`: inserts the blocks
        around the positions `cells` (fp32, cell units) and returns the touched
        blocks as (grid_coords int32[n,3], grid_indices int64[n])."""
        cells = self._activation_buffers(cells)
        self._upkeep(cells.shape[0])
        # the touched rows are listed on the device and their count travels with
        # the read-back that ends the activation (tables beyond the listing
        # kernel's limit take torch's nonzero and a second read-back)
        listing = self.capacity <= COLLECT_MAX_BLOCKS
        if listing:
            rows = torch.empty(self.capacity, dtype=torch.int64, device=self._device)
            coords = torch.empty((self.capacity, 3), dtype=torch.int32, device=self._device)
        for _ in range(2):
            with torch.cuda.device(self._device):
                # (positions in cell units: no origin, cell size 1)
                self._check(
                    self._lib.ash_grid_activate_positions(
                        self._handle, cells.data_ptr(), cells.shape[0], None, 1.0,
                        int(grid_dim), int(dilation), int(bool(bidirectional)), int(bound_lo),
                        int(bound_hi), self._touched.data_ptr(), self._block_coords.data_ptr(),
                        self._stream(),
                    )
                )
                if listing:
                    self._check(
                        self._lib.ash_grid_collect_touched(
                            self._handle, self._touched.data_ptr(), self._block_coords.data_ptr(),
                            rows.data_ptr(), coords.data_ptr(), self._stream(),
                        )
                    )
            self.version = next(_VERSIONS)
            counters = self.counters()
            if counters["exotic_pending"] == 0:
                break
            # blocks beyond the packed range: they need the second region
            self._attach_general()
        if listing:
            n = counters["touched"]
            return coords[:n], rows[:n]
        grid_indices = self._touched.nonzero().view(-1)
        grid_coords = self._block_coords[grid_indices]
        self._touched[grid_indices] = 0
        return grid_coords, grid_indices

    def activate_blocks_deferred(
        self,
        cells: torch.Tensor,
        grid_dim: int,
        dilation: int,
        bidirectional: bool,
        bound_lo: int,
        bound_hi: int,
    ) -> Tuple[torch.Tensor, torch.Tensor]:
        """activate_blocks without its read-back: the blocks are inserted and
        the touched ones listed on the device, and (grid_coords int32[capacity,3],
        grid_indices int64[capacity]) are returned whole -- how many of their
        rows the listing filled stays in the table's counters, where
        ash_grid_integrate_depth_touched reads it.  Nothing here waits for the
        device (every 64th call in a row looks at the counters for the table's
        upkeep), so the launches can be captured into a graph; keys refused for
        lack of capacity show in the counters at the next call that reads them
        (`counters`, `size`, any insert).  Both tensors are reused by the next
        deferred activation of this map."""
        if self.capacity > COLLECT_MAX_BLOCKS:
            raise RuntimeError("deferred activation lists at most 2^20 blocks")
        cells = self._activation_buffers(cells)
        n = cells.shape[0]
        if getattr(self, "_listing", None) is None:
            self._listing = (
                torch.empty((self.capacity, 3), dtype=torch.int32, device=self._device),
                torch.empty(self.capacity, dtype=torch.int64, device=self._device),
            )
        if self._general is None:
            # a key beyond the packed range would otherwise wait for a read-back
            # that this path does not make
            self._attach_general(just_in_case=True)
        self._upkeep(n)
        coords, rows = self._listing
        with torch.cuda.device(self._device):
            # (positions in cell units: no origin, cell size 1; no scratch)
            self._check(
                self._lib.ash_grid_activate_positions(
                    self._handle, cells.data_ptr(), n, None, 1.0, int(grid_dim), int(dilation),
                    int(bool(bidirectional)), int(bound_lo), int(bound_hi),
                    self._touched.data_ptr(), self._block_coords.data_ptr(), self._stream(),
                )
            )
            self._check(
                self._lib.ash_grid_collect_touched(
                    self._handle, self._touched.data_ptr(), self._block_coords.data_ptr(),
                    rows.data_ptr(), coords.data_ptr(), self._stream(),
                )
            )
        self.version = next(_VERSIONS)
        return coords, rows

    def activate_positions(
        self,
        positions: torch.Tensor,
        origin: Optional[torch.Tensor],
        cell_size: float,
        grid_dim: int,
        dilation: int,
        bidirectional: bool,
        bound_lo: int,
        bound_hi: int,
    ) -> None:
        """The activation of `activate_blocks` from world positions (cell units
        = (positions - origin) / cell_size), two launches and nothing else: the
        touched rows stay flagged in the map's own arrays for
        `integrate_depth(flagged_by=map)`, which takes the flags down again.
        Nothing waits for the device and nothing is allocated once the map's
        arrays exist, so the launches can be captured into a graph; keys
        refused for lack of capacity show in the counters at the next call that
        reads them."""
        positions = self._activation_buffers(positions)
        n = positions.shape[0]
        if self._general is None:
            # a key beyond the packed range would otherwise wait for a read-back
            # that this path does not make
            self._attach_general(just_in_case=True)
        self._upkeep(n)
        with torch.cuda.device(self._device):
            self._check(self._lib.ash_grid_activate_positions(
                self._handle, positions.data_ptr(), n,
                origin.data_ptr() if origin is not None else None, float(cell_size),
                int(grid_dim), int(dilation), int(bool(bidirectional)), int(bound_lo),
                int(bound_hi), self._touched.data_ptr(), self._block_coords.data_ptr(),
                self._stream()))
        self.version = next(_VERSIONS)

    def fuse_frame(
        self,
        positions: torch.Tensor,
        origin: Optional[torch.Tensor],
        cell_size: float,
        dilation: int,
        bidirectional: bool,
        bounds: Tuple[int, int],
        embeddings: torch.Tensor,
        grid_dim: int,
        cell_to_world: Tuple[float, Optional[torch.Tensor]],
        intrinsic: torch.Tensor,
        extrinsic: torch.Tensor,
        depth: torch.Tensor,
        color: Optional[torch.Tensor],
        trunc: float,
        depth_max: float,
        count: bool,
    ) -> None:
        """The activation of `activate_blocks` from world positions (cell units
        = (positions - origin) / cell_size) and the depth integration over the
        rows it touches, two launches; with `count` one between them leaves the
        counters, the number of touched blocks among them, where `counters`
        finds them (it does not wait for the integration).
        Nothing waits for the device and nothing is allocated once the map's
        arrays exist, so the launches can (without `count`) be captured into a
        graph; keys refused for lack of capacity show in the counters at the
        next call that reads them."""
        self._activation_buffers(positions)
        counts = None
        if count:
            counts = getattr(self, "_group_counts", None)
            if counts is None:
                counts = self._group_counts = torch.empty(FLAGGED_GROUPS, dtype=torch.int32,
                                                          device=self._device)
        if self._general is None:
            # a key beyond the packed range would otherwise wait for a read-back
            # that this path does not make
            self._attach_general(just_in_case=True)
        self._backend.host.fuse_frame(
            self._address, self._index, positions, origin, cell_size, dilation, bool(bidirectional),
            *bounds, self._touched, self._block_coords, embeddings, grid_dim, *cell_to_world,
            intrinsic, extrinsic, depth, color, trunc, depth_max, counts)
        self.version = next(_VERSIONS)

    def insert_keys(self, keys: torch.Tensor) -> None:
        self._insert(keys, [], [], [])

    def insert(
        self,
        keys: torch.Tensor,
        values: Dict[str, torch.Tensor],
        external_values: Dict[str, torch.Tensor],
    ) -> None:
        self._insert(keys, list(values), list(values.values()), [external_values[name] for name in values])

    def _insert(self, keys, names, values, stores) -> None:
        """One ash_map_insert_auto (a second one after the second region has
        been attached, the first time a key does not fit the packed code)."""
        policy = _INSERT_POLICY[BULK_INSERT]
        for _ in range(2):
            waiting = self._backend.host.insert(self._address, self.key_dim, self._index, self.capacity,
                                                keys, names, values, stores, policy)
            self.version = next(_VERSIONS)
            if not waiting:
                return
            self._attach_general()
        raise RuntimeError("internal error: unpackable keys pending with region attached")

    def erase(self, keys: torch.Tensor) -> None:
        streaming = self._backend.host.erase(self._address, self.key_dim, self._index, keys,
                                             _POLICY[BULK_ERASE])
        self.last_erase_path = "streaming" if streaming else "per-key"
        self.version = next(_VERSIONS)

    def zeroes(self, t: torch.Tensor) -> bool:
        """Whether `clear` can zero `t` along with the table."""
        return stands_alone(t) and self._backend.host.can_zero(t, self._index)

    def clear(self, rows=()) -> None:
        """`rows`: up to four tensors (`zeroes`) to be zeroed in the same launch."""
        self._backend.host.clear(self._address, self._index, list(rows))
        self.version = next(_VERSIONS)

    def _listed(self) -> int:
        """The number of entries that a listing has now."""
        n = self.size()
        # whether entry i is listed under index i: the value rows of the listing
        # are then the first n rows of every value tensor (HashMap.items)
        dense = ctypes.c_int(0)
        self._check(self._lib.ash_map_items_in_index_order(self._handle, ctypes.byref(dense)))
        self.last_items_in_index_order = bool(dense.value)
        return n

    def items(self) -> Tuple[torch.Tensor, torch.Tensor]:
        return self._backend.host.items(self._address, self.key_dim, self._index, self._listed())

    def items_rows(self, tables):
        """(keys, indices, [table[indices] for each table]): the listing and the
        value rows of its entries, for tables that `finds_rows_of` takes."""
        return self._backend.host.items_rows(self._address, self.key_dim, self._index, self._listed(), tables)

    def neighbor_rows(
        self, num_rows: int, radius: int, bidirectional: bool
    ) -> Optional[Tuple[torch.Tensor, torch.Tensor]]:
        """(coords int32 (num_rows, 3), lut int64 (num_rows, K)): key of every
        index and the indices of the keys at its offsets, -1 where there are
        none; None for windows that one launch does not take."""
        if self.key_dim != 3 or not 0 <= radius <= 15:
            return None
        return self._backend.host.neighbors(self._address, self._index, num_rows, radius,
                                            bool(bidirectional))

    def load_states(self, states: Dict[str, torch.Tensor]) -> None:
        keys = self._keys(states["active_keys"])
        indices = states["active_indices"].to(self._device, torch.int64).contiguous()
        heap = states["heap"].to(self._device, torch.int32).contiguous()
        n = keys.shape[0]
        if indices.numel() != n:
            raise RuntimeError("active_keys and active_indices differ in length")
        if heap.numel() != self.capacity:
            raise RuntimeError("heap length differs from the capacity")
        for _ in range(2):
            with torch.cuda.device(self._device):
                self._check(
                    self._lib.ash_map_load(
                        self._handle,
                        keys.data_ptr() if n else None,
                        indices.data_ptr() if n else None,
                        n,
                        heap.data_ptr(),
                        self._stream(),
                    )
                )
            self.version = next(_VERSIONS)
            counters = self.counters()
            if counters["exotic_pending"] == 0:
                break
            self._attach_general()
        refused = counters["load_duplicates"]
        if refused:
            # The reference prints "Error loading, should never reach here!"
            # (ash/src/hashmap_gpu.cuh:420-422) for a repeated key and goes on
            # with a heap counter that no longer matches the stored entries; an
            # index or heap entry outside 0 .. capacity-1 makes its later calls
            # write out of bounds.  Here such a state is refused: the map is
            # left empty.
            self.clear()
            raise RuntimeError(
                f"load_states: {refused} pairs were refused (duplicate keys, or indices / heap "
                "entries outside the capacity); nothing was loaded"
            )


class _MissingBackend:
    """Placeholder used when libash_hip.so cannot be loaded: every use raises."""

    def __init__(self, reason: str):
        self._reason = reason

    def __getattr__(self, name):
        raise RuntimeError(
            f"libash_hip.so is not available ({self._reason}); build it with "
            "`python torch-ash_amd/build.py`. There is no CPU or PyTorch fallback."
        )


_BACKEND = None


def _get_c_extension():
    """Counterpart of ash/common.py:4-15: returns the native backend object."""
    global _BACKEND
    if _BACKEND is None:
        try:
            _BACKEND = _Backend(load_library())
        except OSError as exc:
            warnings.warn(f"HIP extension {_LIB_NAME} could not be loaded: {exc}")
            _BACKEND = _MissingBackend(str(exc))
    return _BACKEND

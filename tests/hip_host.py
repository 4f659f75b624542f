"""libgbr.so over tests/cpp/hip_host.cpp: the library's host code with HIP calls
served from host memory.  Import it before habitat_sim_amd loads the library, in
a process of its own (tests/test_host_runtime.py starts one per case)."""
import ctypes
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "habitat-sim_amd"), os.path.join(ROOT, "tests")):
    if p not in sys.path:
        sys.path.insert(0, p)

LIB = os.path.join(ROOT, "tests", "cpp", "_build", "libhip_host.so")
_lib = ctypes.CDLL(LIB, mode=ctypes.RTLD_GLOBAL)
_lib.hip_host_calls.restype = ctypes.c_int64
_lib.hip_host_used.restype = ctypes.c_int64
_lib.hip_host_blocks.restype = ctypes.c_int64
_HOOK = ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.POINTER(ctypes.c_uint32), ctypes.POINTER(ctypes.c_void_p))
_hook = None


class InputArgs(ctypes.Structure):
    """gbr_device.h InputArgs, the argument of k_inputs."""
    _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p * 6), ("end", ctypes.c_uint32 * 6),
                ("nodes", ctypes.POINTER(ctypes.c_uint32)), ("transforms", ctypes.POINTER(ctypes.c_float)),
                ("local", ctypes.c_void_p), ("n_nodes", ctypes.c_uint32)]


class RasterItem(ctypes.Structure):
    """gbr_device.h RasterItem: a bin, in the second argument of k_raster_lane."""
    _fields_ = [("scene", ctypes.c_uint32), ("gbin", ctypes.c_uint32), ("rect", ctypes.c_int16 * 4),
                ("bin_cap", ctypes.c_uint32), ("plane_offset", ctypes.c_uint32), ("size", ctypes.c_int32 * 2),
                ("entries", ctypes.c_uint64), ("rec_base", ctypes.c_uint64), ("stride", ctypes.c_int32),
                ("planes", ctypes.c_uint32), ("pad", ctypes.c_uint32 * 2)]


class RedwoodArgs(ctypes.Structure):
    """The head of gbr_noise.hip RedwoodArgs, the argument of k_redwood."""
    _fields_ = [("depth", ctypes.c_void_p), ("model", ctypes.c_void_p), ("normals", ctypes.c_void_p),
                ("out", ctypes.c_void_p), ("total", ctypes.c_uint32), ("npx", ctypes.c_uint32),
                ("W", ctypes.c_uint32), ("by_npx", ctypes.c_uint32 * 2), ("by_w", ctypes.c_uint32 * 2),
                ("xmax", ctypes.c_float), ("ymax", ctypes.c_float)]


def on_call(function) -> None:
    """Calls function(name, grid, arguments) at each launch (the kernel's
    mangled name), event record and event wait (the call's name, the event)."""
    global _hook
    _hook = _HOOK(lambda name, grid, args: function(name.decode(), tuple(grid[:3]), args))
    _lib.hip_host_hook(_hook)


def on_launch(kernel: str, argument, function) -> None:
    """Calls function(arguments[0] as an `argument` structure, grid, arguments)
    at each launch of a kernel whose (mangled) name holds `kernel`."""
    on_call(lambda name, grid, args: kernel in name and function(
        argument.from_address(args[0]) if argument else None, grid, args))


def fail(call: str, after: int = 0) -> None:
    """The HIP call of this name fails once, after `after` more that succeed."""
    _lib.hip_host_fail(call.encode(), ctypes.c_int64(after))


def calls(call: str) -> int:
    return _lib.hip_host_calls(call.encode())


def device_memory(limit: int) -> None:
    """hipMalloc fails beyond `limit` bytes in all."""
    _lib.hip_host_memory(ctypes.c_int64(limit))


def device_memory_used() -> int:
    return _lib.hip_host_used()


def memory_blocks() -> int:
    """Device and pinned allocations not yet freed."""
    return _lib.hip_host_blocks()


def runtime():
    """The runtime itself, for calls a user's program makes."""
    return _lib

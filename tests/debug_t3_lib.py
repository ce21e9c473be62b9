"""ctypes view of the T3 path's test-only diagnostics library
(tests/native/cbx_debug_t3.h, built by `make -C tests/native`)."""
import ctypes
import os

import pkg

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "native", "_build", "libcbx_debug_t3.so")

_lib = None


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB):
            raise FileNotFoundError(f"{LIB} is not built; run `make -C tests/native`")
        pkg.load().load_library()  # torch's HIP runtime first, as for the product library
        L = ctypes.CDLL(LIB)
        vp, i64 = ctypes.c_void_p, ctypes.c_int64
        L.cbx_debug_t3_gelu.argtypes = [vp, vp, i64, vp]
        L.cbx_debug_t3_groups.argtypes = [vp, vp, ctypes.c_int32, ctypes.c_int32, vp, vp]
        _lib = L
    return _lib


def _stream():
    import torch
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _ok(rc, name):
    if rc != 0:
        raise RuntimeError(f"{name} returned {rc}")


def gelu(x, out):
    _ok(lib().cbx_debug_t3_gelu(x.data_ptr(), out.data_ptr(), x.numel(), _stream()), "gelu")


def groups(act, slots, n_slots):
    """t3_group_rows on device int32 act and slots: [groups, 16] row numbers, -1 for none."""
    import torch
    n = slots.numel()
    G = lib().cbx_debug_t3_groups(None, None, n, n_slots, None, None)
    rows = torch.full((G, 16), -7, dtype=torch.int32, device=slots.device)
    if lib().cbx_debug_t3_groups(act.data_ptr(), slots.data_ptr(), n, n_slots, rows.data_ptr(),
                                 _stream()) != G:
        raise RuntimeError("groups failed")
    return rows

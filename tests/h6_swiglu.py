"""The Q4_K product of many rows that applies SwiGLU where it stores.  Only a decoder's prompt reaches it through the C interface, with no
trace of which kernel ran, so tests call the library's own function."""
import ctypes

import numpy as np

from joshua_amd import capi


def swiglu_product(blocks, n, lhs):
    """(its return code, -1 for a call that it declines; its output with a row behind it, NaN where nothing is stored) of n weight rows,
    gate and up in turn, and the activation rows `lhs`."""
    import torch
    f = capi.lib()._ZN3jqh14gemm_h6_swigluEjPKhmPKfPfmmmP12ihipStream_t
    f.argtypes = [ctypes.c_uint32, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t,
                  ctypes.c_size_t, ctypes.c_void_p]
    m, k = lhs.shape
    w = capi.Weight.upload(capi.Q4_K, blocks, n, k)
    x, y = torch.from_numpy(np.ascontiguousarray(lhs)).cuda(), torch.full((m + 1, n // 2), float("nan"), device="cuda")
    torch.cuda.synchronize()
    rc = f(capi.Q4_K, w.device_ptr, k // 256 * 144, x.data_ptr(), y.data_ptr(), m, k, n, None)
    torch.cuda.synchronize()
    return rc, y.cpu().numpy()

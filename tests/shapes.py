"""ctypes binding of tests/cpp/shapes.cpp: the 2D kernels by tile shape."""
import ctypes as C

import dropin

J5, BOX9, LIFE8, CLOUD = 1, 2, 3, 5  # kernel patterns


class Job(C.Structure):
    _fields_ = [("src", C.c_void_p), ("dst", C.c_void_p), ("ring", C.c_void_p), ("prev", C.c_void_p),
                ("partials", C.c_void_p), ("wx", C.c_void_p), ("wy", C.c_void_p), ("pitch", C.c_uint64),
                ("xpitch", C.c_uint64), ("ypitch", C.c_uint64), ("W", C.c_int32), ("H", C.c_int32),
                ("pattern", C.c_int32), ("k", C.c_int32), ("coeff", C.c_float), ("wt", C.c_float * 9)]


def lib():
    l = C.CDLL(dropin.driver("libshapes.so"))
    assert l.shapes_job_size() == C.sizeof(Job)
    l.shapes_rtile_blocks.restype = l.shapes_points_blocks.restype = C.c_uint64
    l.shapes_points.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_int,
                                C.c_uint64, C.c_int, C.c_float, C.c_int, C.c_uint32, C.c_uint64]
    l.shapes_plan.argtypes = [C.c_int, C.c_int, C.c_int, C.c_uint64, C.c_int, C.POINTER(C.c_int32)]
    return l


def plan(l, pattern, w, h, rem, odd=False):
    out = (C.c_int32 * 3)()
    l.shapes_plan(pattern, w, h, rem, int(odd), out)
    return tuple(out)

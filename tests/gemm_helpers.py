"""The block decoders' prompt product and its plans through tests/gemm_harness.cpp."""
import ctypes as C
import os

from conftest import ROOT

F32, ELEM, RELU2, SWIGLU, DECAY = range(5)
TILES = [(256, 256), (256, 192), (128, 256), (128, 192), (128, 128), (64, 256), (64, 128)]  # rows and columns of each kind


class Call(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in "A W C bias".split()] + [(n, C.c_int64) for n in "lda ldw ldc section_a slab slab_room".split()] + \
               [(n, C.c_int32) for n in "M N K epilogue section_n may_split".split()]


def harness():
    path = os.path.join(ROOT, "tests", "libshim_harness.so")
    assert os.path.exists(path), "tests/libshim_harness.so is not built (python -c 'import __graft_entry__ as g; g.build()')"
    h = C.CDLL(path)
    h.gemm_run.argtypes = [C.POINTER(Call), C.POINTER(C.c_int32), C.c_void_p]
    h.gemm_plan.argtypes = [C.POINTER(Call), C.POINTER(C.c_int32)]
    h.gemm_plan.restype = None
    return h


def plan(M, N, K, epilogue=F32, section=0, slabs=0):
    """(K splits, workgroups, [(kind, first workgroup, row, column, end of columns, row tiles, column tiles)]); no regions: 64 x 64 tiles.
    slabs > 0: the caller takes up to so many partial sums."""
    kp = (K + 63) // 64 * 64
    c = Call(M=M, N=N, K=K, lda=kp, ldw=kp, ldc=N, epilogue=epilogue, section_n=section, slab=M * N, slab_room=M * N * slabs, may_split=int(slabs > 0))
    out = (C.c_int32 * 32)()
    harness().gemm_plan(C.byref(c), out)
    return out[0], out[1], [tuple(out[3 + 7 * i:10 + 7 * i]) for i in range(out[2])]

"""How the products of a K-quant run are cut: the library's rule (an internal entry point, called by its C++ name) and the cuts that its
sums are held to."""
import ctypes as C

from guffin_amd import hip, synth


class Matrix(C.Structure):
    _fields_ = [("dtype", C.c_int), ("tiles", C.c_void_p), ("N", C.c_uint32)]


class Split(C.Structure):
    _fields_ = [("row_tiles", C.c_uint32), ("slices", C.c_uint32), ("halves", C.c_uint32)]


Q4, Q6 = synth.Q4_K, synth.Q6_K
# K, (format, N) of each matrix of a launch of the 12B shapes, plain blocks and those all in four bits
PRODUCTS = {"qkv": (3840, ((Q4, 4096), (Q4, 2048), (Q6, 2048))), "qkv4": (3840, ((Q4, 4096), (Q4, 2048), (Q4, 2048))),
            "o": (4096, ((Q4, 3840),)), "gate_up": (3840, ((Q4, 15360), (Q4, 15360))), "down": (15360, ((Q6, 3840),)),
            "down4": (15360, ((Q4, 3840),))}
# from which run on (rows) how many slices: the cuts by the costs of long runs, whose sums' error no other cut of a run of up to 192 rows may
# exceed
BAR = {"qkv": ((5, 15), (14, 8), (49, 4), (65, 5), (97, 4), (129, 5), (145, 3), (161, 5)),
       "qkv4": ((5, 15), (13, 8), (49, 4), (65, 5), (94, 4), (129, 5), (145, 3), (161, 5), (188, 3)),
       "o": ((5, 16), (24, 8), (111, 4), (129, 8), (145, 4)), "gate_up": ((5, 4), (60, 3), (65, 2), (145, 1)),
       "down": ((5, 15), (129, 10)), "down4": ((5, 15), (129, 10))}


def bar(name, rows):
    return [s for first, s in BAR[name] if first <= rows][-1]


def cut_of(K, parts, rows):
    """The library's cut of a run of `rows` through one launch of `parts` ((format, N))."""
    f = hip.lib()._ZN6guffin13prefill_splitEPKNS_13PrefillMatrixEjjj
    f.argtypes, f.restype = [C.POINTER(Matrix), C.c_uint32, C.c_uint32, C.c_uint32], Split
    return f((Matrix * len(parts))(*[Matrix(dtype, None, n) for dtype, n in parts]), len(parts), rows, K)


def split(name, rows):
    K, parts = PRODUCTS[name]
    return cut_of(K, parts, rows)


def planes(parts, image, M, K, cut):
    """The planes of each of `parts` ((format, tiles, N), one launch), cut so, on the current stream."""
    import torch
    f = hip.lib()._ZN6guffin19prefill_gemm_planesEP12ihipStream_tPKNS_13PrefillMatrixEjPKhPKPfjjNS_12PrefillSplitE
    f.argtypes, f.restype = [C.c_void_p, C.POINTER(Matrix), C.c_uint32, C.c_void_p, C.POINTER(C.c_void_p), C.c_uint32, C.c_uint32, Split], C.c_int
    y = [torch.full((cut.slices, M, N), float("nan"), device="cuda") for _, _, N in parts]
    m = (Matrix * len(parts))(*[Matrix(dtype, tiles.data_ptr(), N) for dtype, tiles, N in parts])
    hip.check(f(hip._raw_stream(), m, len(m), image.data_ptr(), (C.c_void_p * len(y))(*[p.data_ptr() for p in y]), M, K, cut))
    return y

"""ctypes mirror of libSpMM_API.so, with the reference's names and argument order.

The functions here add nothing to the C ABI: they convert numpy arrays and
device pointers, call through, and turn error codes into exceptions.  There is
no CPU fallback: if the library has not been built, loading fails.

Reference interfaces mirrored (paths relative to the reference checkout):
  InitSparseMatrixA_API   build/SpMM_API.cuh:55, csrc/SpMM_API.cu:241-438
  SpMM_SplitK_API         third_party/ft.patch:2833-2843, csrc/SpMM_API.cu:79-208
  GenSparseMatrixBinFile  csrc/SpMM_API.cu:1565-1620,
                          end2end_inference/ft_tools/huggingface_opt_convert_Phase2.py:36-59
  decompose               kernel_benchmark/spmm_decompose.h:12-51  (HeteroSparse_Decompose)
  2:4 part + residual     kernel_benchmark/spmm_test.cu:285-330,462-560, csrc/SpMM_API.cu:1127-1553
                          (HeteroSparse_PackA1, HeteroSparse_SpMM_API)
"""
import ctypes
import os
import subprocess

import numpy as np

_PKG = os.path.dirname(os.path.abspath(__file__))
# SPMM_LIB_PATH selects another build of the same library (used to compare kernel variants).
_LIB_PATH = os.environ.get("SPMM_LIB_PATH") or os.path.join(_PKG, "lib", "libSpMM_API.so")

_u16p = ctypes.POINTER(ctypes.c_uint16)
_u32p = ctypes.POINTER(ctypes.c_uint32)
_i32p = ctypes.POINTER(ctypes.c_int)
_ALLOCATE = ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t)

EXPORTED_SYMBOLS = (
    "InitSparseMatrixA_API",
    "InitSparseMatrixA_API_NoReorder",
    "SpMM_EncodeInto",
    "SpMM_SplitK_API",
    "SpMM_SplitK_API_StaticWorkspace",
    "GenSparseMatrixBinFile",
    "SpMM_FreeHost",
    "SpMM_GetErrorString",
    "SpMM_SuggestSplitK",
    "SpMM_SuggestSplitK_Bytes",
    "SpMM_PlanLaunch",
    "SpMM_PlanReductionInLaunch",
    "SpMM_SplitK_API_Planned",
    "SpMM_SplitK_API_RowMajor",
    "SpMM_SplitK_API_RowMajor_Flags",
    "SpMM_SplitK_API_Strided",
    "SpMM_DeviceEncodeOffsets",
    "SpMM_DeviceEncodeItems",
    "SpMM_SynthWeights",
    "SpMM_SynthActivations",
    "SpMM_SynthHarnessWeights",
    "SpMM_SynthHarnessActivations",
    "SpMM_CalibrationCopy",
    "SpMM_SplitK_API_Events",
    "SpMM_SplitK_Partials",
    "SpMM_EventCreate",
    "SpMM_EventDestroy",
    "SpMM_EventRecord",
    "SpMM_EventElapsedMs",
    "HeteroSparse_Decompose",
    "HeteroSparse_PackedBytes",
    "HeteroSparse_PackA1",
    "HeteroSparse_SpMM_API",
    "HeteroSparse_SuggestSplitK",
    "HeteroSparse_A1_Partials",
    "HeteroSparse_DeviceSplitPack",
    "HeteroSparse_PackA2",
    "HeteroSparse_DevicePackA2_Offsets",
    "HeteroSparse_DevicePackA2_Words",
    "HeteroSparse_Fused_SpMM_API",
    "HeteroSparse_Fused_SpMM_API_Strided",
    "HeteroSparse_SpMM_API_RowMajor",
    "HeteroSparse_Fused_SpMM_API_RowMajor",
)


class SpMMError(RuntimeError):
    """A non-zero code from the library."""

    def __init__(self, where, code, text=""):
        super().__init__(f"{where} failed with code {code}" + (f" ({text})" if text else ""))
        self.code = code


def library_path():
    return _LIB_PATH


def build_library():
    """Compile the library in-tree with hipcc (always recompiles)."""
    csrc = os.path.join(_PKG, "csrc")
    subprocess.run(["make", "-s", "-C", csrc, "clean"], check=True)
    subprocess.run(["make", "-s", "-C", csrc, "-j8"], check=True)
    return _LIB_PATH


_lib = None


def load_library():
    """Load libSpMM_API.so; raises if it is missing (no fallback)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(_LIB_PATH):
        raise FileNotFoundError(
            f"{_LIB_PATH} not found: build it with graphneuralnetproj_amd.build_library() "
            "or `make -C graphneuralnetproj_amd/csrc`")
    # A process must hold ONE HIP runtime.  Device memory and streams come from
    # PyTorch here, and PyTorch ships its own libamdhip64 (same soname as the
    # system one): importing it first makes the loader bind this library to that
    # copy instead of mapping a second runtime that cannot see the device.
    try:
        import torch  # noqa: F401
    except ImportError:
        pass
    lib = ctypes.CDLL(_LIB_PATH)
    lib.InitSparseMatrixA_API.restype = ctypes.c_int
    lib.InitSparseMatrixA_API.argtypes = [_u16p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.POINTER(_u32p),
                                          ctypes.POINTER(_i32p)]
    lib.InitSparseMatrixA_API_NoReorder.restype = ctypes.c_int
    lib.InitSparseMatrixA_API_NoReorder.argtypes = lib.InitSparseMatrixA_API.argtypes
    lib.SpMM_EncodeInto.restype = ctypes.c_int
    lib.SpMM_EncodeInto.argtypes = [_u16p, ctypes.c_int, ctypes.c_int, ctypes.c_int, _ALLOCATE, ctypes.c_void_p, _i32p]
    lib.SpMM_SplitK_API.restype = ctypes.c_int
    lib.SpMM_SplitK_API.argtypes = [ctypes.c_void_p] * 6 + [ctypes.c_int] * 3 + [ctypes.c_void_p, ctypes.c_int]
    lib.SpMM_SplitK_API_StaticWorkspace.restype = ctypes.c_int
    lib.SpMM_SplitK_API_StaticWorkspace.argtypes = [ctypes.c_void_p] * 6 + [ctypes.c_int] * 4
    lib.GenSparseMatrixBinFile.restype = ctypes.c_int
    lib.GenSparseMatrixBinFile.argtypes = [ctypes.c_char_p, ctypes.c_int, ctypes.c_int, ctypes.c_char_p,
                                           ctypes.c_char_p, ctypes.c_char_p]
    lib.SpMM_FreeHost.restype = None
    lib.SpMM_FreeHost.argtypes = [ctypes.c_void_p]
    lib.SpMM_GetErrorString.restype = ctypes.c_char_p
    lib.SpMM_GetErrorString.argtypes = [ctypes.c_int]
    lib.SpMM_SuggestSplitK.restype = ctypes.c_int
    lib.SpMM_SuggestSplitK.argtypes = [ctypes.c_int] * 3
    lib.SpMM_SuggestSplitK_Bytes.restype = ctypes.c_int
    lib.SpMM_SuggestSplitK_Bytes.argtypes = [ctypes.c_int] * 3 + [ctypes.c_long]
    lib.SpMM_PlanLaunch.restype = ctypes.c_int
    lib.SpMM_PlanLaunch.argtypes = [ctypes.c_int] * 4 + [_i32p] * 4 + [ctypes.POINTER(ctypes.c_double)]
    lib.SpMM_PlanReductionInLaunch.restype = ctypes.c_int
    lib.SpMM_PlanReductionInLaunch.argtypes = [ctypes.c_int] * 4
    lib.SpMM_SplitK_API_Planned.restype = ctypes.c_int
    lib.SpMM_SplitK_API_Planned.argtypes = ([ctypes.c_void_p] * 5 + [ctypes.c_int] * 3 + [ctypes.c_void_p]
                                            + [ctypes.c_int] * 6)
    lib.SpMM_SplitK_API_Strided.restype = ctypes.c_int
    lib.SpMM_SplitK_API_Strided.argtypes = ([ctypes.c_void_p] * 4 + [ctypes.c_long, ctypes.c_void_p, ctypes.c_long]
                                            + [ctypes.c_int] * 3 + [ctypes.c_void_p, ctypes.c_int, ctypes.c_int])
    lib.SpMM_DeviceEncodeOffsets.restype = ctypes.c_int
    lib.SpMM_DeviceEncodeOffsets.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    lib.SpMM_DeviceEncodeItems.restype = ctypes.c_int
    lib.SpMM_DeviceEncodeItems.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p,
                                           ctypes.c_void_p]
    lib.SpMM_SplitK_API_RowMajor.restype = ctypes.c_int
    lib.SpMM_SplitK_API_RowMajor.argtypes = lib.SpMM_SplitK_API.argtypes
    lib.SpMM_SplitK_API_RowMajor_Flags.restype = ctypes.c_int
    lib.SpMM_SplitK_API_RowMajor_Flags.argtypes = [ctypes.c_void_p] * 5 + [ctypes.c_int] * 3 + [ctypes.c_void_p, ctypes.c_int,
                                                                                              ctypes.c_int]
    lib.SpMM_SynthWeights.restype = None
    lib.SpMM_SynthWeights.argtypes = [_u16p, ctypes.c_int, ctypes.c_int, ctypes.c_double, ctypes.c_int,
                                      ctypes.c_uint64]
    lib.SpMM_SynthActivations.restype = None
    lib.SpMM_SynthActivations.argtypes = [_u16p, ctypes.c_long, ctypes.c_uint64]
    lib.SpMM_SynthHarnessWeights.restype = None
    lib.SpMM_SynthHarnessWeights.argtypes = lib.SpMM_SynthWeights.argtypes
    lib.SpMM_SynthHarnessActivations.restype = None
    lib.SpMM_SynthHarnessActivations.argtypes = lib.SpMM_SynthActivations.argtypes
    lib.SpMM_CalibrationCopy.restype = ctypes.c_int
    lib.SpMM_CalibrationCopy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long]
    lib.SpMM_SplitK_API_Events.restype = ctypes.c_int
    lib.SpMM_SplitK_API_Events.argtypes = lib.SpMM_SplitK_API.argtypes + [ctypes.c_void_p, ctypes.c_void_p]
    lib.SpMM_SplitK_Partials.restype = ctypes.c_int
    lib.SpMM_SplitK_Partials.argtypes = [ctypes.c_void_p] * 5 + [ctypes.c_int] * 4
    lib.SpMM_EventCreate.restype = ctypes.c_void_p
    lib.SpMM_EventCreate.argtypes = []
    lib.SpMM_EventDestroy.restype = None
    lib.SpMM_EventDestroy.argtypes = [ctypes.c_void_p]
    lib.SpMM_EventRecord.restype = ctypes.c_int
    lib.SpMM_EventRecord.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    lib.SpMM_EventElapsedMs.restype = ctypes.c_float
    lib.SpMM_EventElapsedMs.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    lib.HeteroSparse_Decompose.restype = ctypes.c_int
    lib.HeteroSparse_Decompose.argtypes = [_u16p, _u16p, _u16p, ctypes.c_long]
    lib.HeteroSparse_PackedBytes.restype = ctypes.c_long
    lib.HeteroSparse_PackedBytes.argtypes = [ctypes.c_int, ctypes.c_int]
    lib.HeteroSparse_PackA1.restype = ctypes.c_int
    lib.HeteroSparse_PackA1.argtypes = [_u16p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    lib.HeteroSparse_SpMM_API.restype = ctypes.c_int
    lib.HeteroSparse_SpMM_API.argtypes = [ctypes.c_void_p] * 6 + [ctypes.c_int] * 3 + [ctypes.c_void_p] + [ctypes.c_int] * 3
    lib.HeteroSparse_SuggestSplitK.restype = ctypes.c_int
    lib.HeteroSparse_SuggestSplitK.argtypes = [ctypes.c_int] * 3
    lib.HeteroSparse_DeviceSplitPack.restype = ctypes.c_int
    lib.HeteroSparse_DeviceSplitPack.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int,
                                                 ctypes.c_void_p, ctypes.c_void_p]
    lib.HeteroSparse_PackA2.restype = ctypes.c_int
    lib.HeteroSparse_PackA2.argtypes = [_u16p, ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.POINTER(ctypes.c_uint32)),
                                        ctypes.POINTER(ctypes.POINTER(ctypes.c_int)), ctypes.POINTER(ctypes.c_int)]
    lib.HeteroSparse_DevicePackA2_Offsets.restype = ctypes.c_int
    lib.HeteroSparse_DevicePackA2_Offsets.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p,
                                                      ctypes.c_void_p]
    lib.HeteroSparse_DevicePackA2_Words.restype = ctypes.c_int
    lib.HeteroSparse_DevicePackA2_Words.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p,
                                                    ctypes.c_void_p]
    lib.HeteroSparse_Fused_SpMM_API.restype = ctypes.c_int
    lib.HeteroSparse_Fused_SpMM_API.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int] + [ctypes.c_void_p] * 2 + [ctypes.c_int] * 3 + [
        ctypes.c_void_p, ctypes.c_int]
    lib.HeteroSparse_Fused_SpMM_API_Strided.restype = ctypes.c_int
    lib.HeteroSparse_Fused_SpMM_API_Strided.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int, ctypes.c_void_p, ctypes.c_long,
                                                        ctypes.c_void_p, ctypes.c_long] + [ctypes.c_int] * 3 + [
        ctypes.c_void_p, ctypes.c_int, ctypes.c_int]
    lib.HeteroSparse_SpMM_API_RowMajor.restype = ctypes.c_int
    lib.HeteroSparse_SpMM_API_RowMajor.argtypes = lib.HeteroSparse_SpMM_API.argtypes
    lib.HeteroSparse_Fused_SpMM_API_RowMajor.restype = ctypes.c_int
    lib.HeteroSparse_Fused_SpMM_API_RowMajor.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int] + [ctypes.c_void_p] * 2 + [ctypes.c_int] * 3 + [
        ctypes.c_void_p, ctypes.c_int, ctypes.c_int]
    lib.HeteroSparse_A1_Partials.restype = ctypes.c_int
    lib.HeteroSparse_A1_Partials.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int] * 7
    _lib = lib
    return lib


def _bits(a):
    a = np.ascontiguousarray(a)
    if a.dtype == np.float16:
        return a.view(np.uint16)
    if a.dtype != np.uint16:
        raise TypeError(f"expected float16 (or uint16 bit patterns), got {a.dtype}")
    return a


def InitSparseMatrixA_API_NoReorder(A_h, M=None, N=0, K=None):
    """InitSparseMatrixA_API without the bank-aware reordering of a tile's words."""
    return InitSparseMatrixA_API(A_h, M, N, K, _entry="InitSparseMatrixA_API_NoReorder")


def InitSparseMatrixA_API(A_h, M=None, N=0, K=None, _entry="InitSparseMatrixA_API"):
    """Encode a row-major fp16 M x K host matrix.

    Returns (Compressed_A uint32[4*TileOffsets[-1]], TileOffsets int32[(M/128)*(K/64)+2]);
    len(TileOffsets) is what the C function returns.  Raises SpMMError on a
    shape the reference would assert on.
    """
    a = _bits(A_h)
    if M is None or K is None:
        M, K = a.shape
    if a.size != M * K:
        raise ValueError(f"A_h has {a.size} elements, expected {M}*{K}")
    lib = load_library()
    if M <= 0 or K <= 0 or M % 128 or K % 64:
        raise SpMMError(_entry, -1)
    offsets = np.empty((M // 128) * (K // 64) + 2, dtype=np.int32)
    words = []

    # The words go straight into an array that owns them (a copy out of the library's memory, 41 MB on one
    # thread for 7168 x 7168 at 80 % sparsity, took longer than the encoding).
    def allocate(_, size):
        try:
            words.append(np.empty(size // 4, dtype=np.uint32))
        except MemoryError:
            return None
        return words[0].ctypes.data

    n = lib.SpMM_EncodeInto(a.ctypes.data_as(_u16p), M, K, _entry == "InitSparseMatrixA_API", _ALLOCATE(allocate), None,
                            offsets.ctypes.data_as(_i32p))
    if n < 0:
        raise SpMMError(_entry, n)
    return words.pop(), offsets


def _ptr(x):
    """Device pointer of a torch tensor, or a raw integer address, or None."""
    if x is None:
        return None
    if isinstance(x, int):
        return ctypes.c_void_p(x)
    return ctypes.c_void_p(x.data_ptr())


def SpMM_SplitK_API(stream, A, Compressed_A, TileOffsets, B, C, M_Global, N_Global, K_Global, Reduction_Workspace,
                    Split_K):
    """Enqueue C = A * B on `stream` (an integer hipStream_t or a torch stream; None = default).

    Tensor arguments are torch CUDA tensors (or raw device addresses); A is
    unused and may be None.  Returns 0; raises SpMMError with the hipError_t
    code otherwise.
    """
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.SpMM_SplitK_API(ctypes.c_void_p(stream) if stream else None, _ptr(A), _ptr(Compressed_A),
                             _ptr(TileOffsets), _ptr(B), _ptr(C), M_Global, N_Global, K_Global,
                             _ptr(Reduction_Workspace), Split_K)
    if rc != 0:
        raise SpMMError("SpMM_SplitK_API", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def SpMM_SplitK_API_StaticWorkspace(stream, A, Compressed_A, TileOffsets, B, C, M_Global, N_Global, K_Global, Split_K):
    """SpMM_SplitK_API on the library's static workspace (allocates nothing; Split_K*M*N*2 <= 32 MiB)."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.SpMM_SplitK_API_StaticWorkspace(ctypes.c_void_p(stream) if stream else None, _ptr(A), _ptr(Compressed_A),
                                             _ptr(TileOffsets), _ptr(B), _ptr(C), M_Global, N_Global, K_Global, Split_K)
    if rc != 0:
        raise SpMMError("SpMM_SplitK_API_StaticWorkspace", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def SpMM_SplitK_API_RowMajor(stream, A, Compressed_A, TileOffsets, B, C, M_Global, N_Global, K_Global,
                             Reduction_Workspace, Split_K):
    """SpMM_SplitK_API for row-major B (K x N) and C (M x N)."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.SpMM_SplitK_API_RowMajor(ctypes.c_void_p(stream) if stream else None, _ptr(A), _ptr(Compressed_A),
                                      _ptr(TileOffsets), _ptr(B), _ptr(C), M_Global, N_Global, K_Global,
                                      _ptr(Reduction_Workspace), Split_K)
    if rc != 0:
        raise SpMMError("SpMM_SplitK_API_RowMajor", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


SPMM_FLAG_RELU = 1
SPMM_FLAG_SEPARATE_REDUCTION = 2
SPMM_FLAG_ADAPTIVE_WAVES = 4  # SpMM_SplitK_API_Planned only


def SpMM_SplitK_API_Strided(stream, Compressed_A, TileOffsets, B, ldb, C, ldc, M_Global, N_Global, K_Global,
                            Reduction_Workspace, Split_K, Flags=0):
    """Column-major SpMM on token vectors ldb / ldc elements apart, optionally clamped at zero."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.SpMM_SplitK_API_Strided(ctypes.c_void_p(stream) if stream else None, _ptr(Compressed_A), _ptr(TileOffsets),
                                     _ptr(B), ldb, _ptr(C), ldc, M_Global, N_Global, K_Global,
                                     _ptr(Reduction_Workspace), Split_K, Flags)
    if rc != 0:
        raise SpMMError("SpMM_SplitK_API_Strided", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def encode_on_device(A_d, stream=None):
    """Tiled-CSL encode of a torch CUDA fp16 matrix on the GPU -> (items int32 tensor, offsets int32 tensor).

    Same bits as InitSparseMatrixA_API; synchronises once to size the word buffer.
    """
    import torch

    lib = load_library()
    M, K = A_d.shape
    if A_d.dtype != torch.float16 or not A_d.is_contiguous():
        raise TypeError("expected a contiguous float16 CUDA tensor")
    if stream is None:
        stream = torch.cuda.current_stream()
    sptr = ctypes.c_void_p(stream.cuda_stream) if stream.cuda_stream else None
    tiles = (M // 128) * (K // 64)
    offsets = torch.empty(max(tiles, 0) + 2, dtype=torch.int32, device=A_d.device)
    rc = lib.SpMM_DeviceEncodeOffsets(sptr, _ptr(A_d), M, K, _ptr(offsets))
    if rc != 0:
        raise SpMMError("SpMM_DeviceEncodeOffsets", rc, lib.SpMM_GetErrorString(rc).decode())
    vectors = int(offsets[-1].item())  # synchronises
    if vectors < 0:
        raise SpMMError("SpMM_DeviceEncodeOffsets", -5, "more than 2^31-1 vectors")
    items = torch.empty(max(vectors * 4, 4), dtype=torch.int32, device=A_d.device)
    rc = lib.SpMM_DeviceEncodeItems(sptr, _ptr(A_d), M, K, _ptr(offsets), _ptr(items))
    if rc != 0:
        raise SpMMError("SpMM_DeviceEncodeItems", rc, lib.SpMM_GetErrorString(rc).decode())
    return items[: vectors * 4], offsets


def GenSparseMatrixBinFile(DenseMatrixFileName, M, K, NZWeightsFileName, TileOffsetsFileName, OutputSizesFileName):
    lib = load_library()
    rc = lib.GenSparseMatrixBinFile(DenseMatrixFileName.encode(), M, K, NZWeightsFileName.encode(),
                                    TileOffsetsFileName.encode(), OutputSizesFileName.encode())
    if rc != 0:
        raise SpMMError("GenSparseMatrixBinFile", rc)
    return rc


def SpMM_SuggestSplitK(M_Global, N_Global, K_Global):
    return load_library().SpMM_SuggestSplitK(M_Global, N_Global, K_Global)


def SpMM_SuggestSplitK_Bytes(M_Global, N_Global, K_Global, Vectors):
    """SpMM_SuggestSplitK for a weight whose TileOffsets end at `Vectors`."""
    return load_library().SpMM_SuggestSplitK_Bytes(M_Global, N_Global, K_Global, int(Vectors))


def SpMM_PlanLaunch(M_Global, N_Global, K_Global, Split_K):
    """The planner's launch shape for a call: dict(mode, waves, stage_b, lds_bytes, estimated_us, paired, two_per_row).
    paired: both waves work on every tile (64 tokens); SpMM_SplitK_API_Planned launches that shape with StageB = 3.  two_per_row:
    `waves` counts tile rows, of two waves each (64 tokens); StageB = 4 there."""
    vals = [ctypes.c_int() for _ in range(4)]
    est = ctypes.c_double()
    rc = load_library().SpMM_PlanLaunch(M_Global, N_Global, K_Global, Split_K, *[ctypes.byref(v) for v in vals],
                                        ctypes.byref(est))
    if rc != 0:
        raise SpMMError("SpMM_PlanLaunch", rc)
    return {"mode": vals[0].value, "waves": vals[1].value, "stage_b": vals[2].value, "lds_bytes": vals[3].value,
            "estimated_us": est.value, "paired": (vals[0].value, vals[1].value, vals[3].value) == (0, 2, 3 * 16384),
            "two_per_row": N_Global == 64 and (vals[0].value, vals[1].value, vals[2].value, vals[3].value) == (0, 3, 0, 160 * 1024)}


def SpMM_PlanReductionInLaunch(M_Global, N_Global, K_Global, Split_K):
    """True if the planned call adds its slabs of partial sums up inside the main kernel's launch,
    False if it runs the reduction kernel (or Split_K is 1)."""
    rc = load_library().SpMM_PlanReductionInLaunch(M_Global, N_Global, K_Global, Split_K)
    if rc < 0:
        raise SpMMError("SpMM_PlanReductionInLaunch", rc)
    return bool(rc)


def SpMM_SplitK_API_RowMajor_Flags(stream, Compressed_A, TileOffsets, B, C, M_Global, N_Global, K_Global, Reduction_Workspace,
                                   Split_K, Flags=0):
    """SpMM_SplitK_API_RowMajor (B[K][N], C[M][N]) with Flags (SPMM_FLAG_RELU, SPMM_FLAG_SEPARATE_REDUCTION)."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.SpMM_SplitK_API_RowMajor_Flags(ctypes.c_void_p(stream) if stream else None, _ptr(Compressed_A), _ptr(TileOffsets),
                                            _ptr(B), _ptr(C), M_Global, N_Global, K_Global, _ptr(Reduction_Workspace), Split_K,
                                            Flags)
    if rc != 0:
        raise SpMMError("SpMM_SplitK_API_RowMajor_Flags", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def SpMM_SplitK_API_Planned(stream, Compressed_A, TileOffsets, B, C, M_Global, N_Global, K_Global,
                            Reduction_Workspace, Split_K, Mode, Waves, StageB, RowMajor=0, Flags=0):
    """SpMM_SplitK_API with a caller-chosen launch shape (tuning and tests)."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.SpMM_SplitK_API_Planned(ctypes.c_void_p(stream) if stream else None, _ptr(Compressed_A), _ptr(TileOffsets),
                                     _ptr(B), _ptr(C), M_Global, N_Global, K_Global, _ptr(Reduction_Workspace),
                                     Split_K, Mode, Waves, StageB, RowMajor, Flags)
    if rc != 0:
        raise SpMMError("SpMM_SplitK_API_Planned", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def synth_weights(M, K, sparsity, row_skewed=False, seed=0):
    """Deterministic synthetic fp16 weight, row-major M x K."""
    A = np.empty((M, K), dtype=np.uint16)
    load_library().SpMM_SynthWeights(A.ctypes.data_as(_u16p), M, K, float(sparsity), int(bool(row_skewed)), seed)
    return A.view(np.float16)


def synth_activations(N, K, seed=0):
    """Deterministic synthetic fp16 activations, one K vector per token (N x K)."""
    B = np.empty((N, K), dtype=np.uint16)
    load_library().SpMM_SynthActivations(B.ctypes.data_as(_u16p), N * K, seed)
    return B.view(np.float16)


def synth_harness_weights(M, K, sparsity, row_skewed=False, seed=0):
    """The reference harness's weights (kernel_benchmark/spmm_test_utils.h:111-123): kept values are
    exactly 1.0; the keep decisions are those of synth_weights with the same arguments."""
    A = np.empty((M, K), dtype=np.uint16)
    load_library().SpMM_SynthHarnessWeights(A.ctypes.data_as(_u16p), M, K, float(sparsity), int(bool(row_skewed)), seed)
    return A.view(np.float16)


def synth_harness_activations(N, K, seed=0):
    """The reference harness's activations (kernel_benchmark/spmm_test_utils.h:137-141): values in
    {-5, -3, -1, 1, 3}, one K vector per token (N x K)."""
    B = np.empty((N, K), dtype=np.uint16)
    load_library().SpMM_SynthHarnessActivations(B.ctypes.data_as(_u16p), N * K, seed)
    return B.view(np.float16)


# ---------------------------------------------------------------------------------------------
# 2:4 part on the sparse matrix cores + Tiled-CSL residual


HETERO_FLAG_TWO_STREAMS = 1


def HeteroSparse_Decompose(A_h):
    """(A1, A2) of a row-major fp16 matrix: at most two kept values per group of four in A1, the
    rest in A2 (kernel_benchmark/spmm_decompose.h:12-51, bit for bit)."""
    a = _bits(A_h)
    A1 = np.empty(a.shape, dtype=np.uint16)
    A2 = np.empty(a.shape, dtype=np.uint16)
    rc = load_library().HeteroSparse_Decompose(a.ctypes.data_as(_u16p), A1.ctypes.data_as(_u16p),
                                               A2.ctypes.data_as(_u16p), a.size)
    if rc != 0:
        raise SpMMError("HeteroSparse_Decompose", rc)
    return A1.view(np.float16), A2.view(np.float16)


def HeteroSparse_PackA1(A1_h, M=None, K=None):
    """Records of the 2:4 part in sparse-MFMA operand order -> uint8[(M/16)*(K/128)*2304]."""
    a = _bits(A1_h)
    if M is None or K is None:
        M, K = a.shape
    lib = load_library()
    size = lib.HeteroSparse_PackedBytes(M, K)
    if size < 0:
        raise SpMMError("HeteroSparse_PackedBytes", int(size))
    packed = np.empty(size, dtype=np.uint8)
    rc = lib.HeteroSparse_PackA1(a.ctypes.data_as(_u16p), M, K, packed.ctypes.data_as(ctypes.c_void_p))
    if rc != 0:
        raise SpMMError("HeteroSparse_PackA1", rc)
    return packed


def HeteroSparse_SuggestSplitK(M_Global, N_Global, K_Global):
    return load_library().HeteroSparse_SuggestSplitK(M_Global, N_Global, K_Global)


def HeteroSparse_SpMM_API(stream, Packed_A1, Compressed_A2, TileOffsets_A2, B, C, M_Global, N_Global, K_Global,
                          Reduction_Workspace, Split_K_A1, Split_K_A2, Flags=0):
    """Enqueue C = A1*B + A2*B (A1 as 2:4 records, A2 as Tiled-CSL or None) on `stream`."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.HeteroSparse_SpMM_API(ctypes.c_void_p(stream) if stream else None, _ptr(Packed_A1), _ptr(Compressed_A2),
                                   _ptr(TileOffsets_A2), _ptr(B), _ptr(C), M_Global, N_Global, K_Global,
                                   _ptr(Reduction_Workspace), Split_K_A1, Split_K_A2, Flags)
    if rc != 0:
        raise SpMMError("HeteroSparse_SpMM_API", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


HETERO_FUSED_MAX_LIST = 1024  # include/SpMM_API.h: what a block of a residual can hold
HETERO_FUSED_PIPELINED_ROUNDS = 5


def HeteroSparse_PackA2(A2_h, M=None, K=None):
    """Residual lists for HeteroSparse_Fused_SpMM_API -> (words uint32[NNZ + 64], offsets int32, longest list)."""
    a = _bits(A2_h)
    if M is None or K is None:
        M, K = a.shape
    lib = load_library()
    words = ctypes.POINTER(ctypes.c_uint32)()
    offsets = ctypes.POINTER(ctypes.c_int)()
    longest = ctypes.c_int(0)
    n = lib.HeteroSparse_PackA2(a.ctypes.data_as(_u16p), M, K, ctypes.byref(words), ctypes.byref(offsets),
                                ctypes.byref(longest))
    if n < 0:
        raise SpMMError("HeteroSparse_PackA2", n)
    try:
        offs = np.ctypeslib.as_array(offsets, shape=(n,)).copy()
        w = np.ctypeslib.as_array(words, shape=(int(offs[-1]) + 64,)).copy()
    finally:
        lib.SpMM_FreeHost(words)
        lib.SpMM_FreeHost(offsets)
    return w, offs, int(longest.value)


def HeteroSparse_Fused_SpMM_API(stream, Packed_A1, A2_Words, A2_Offsets, LongestList, B, C, M_Global, N_Global, K_Global,
                                Reduction_Workspace, Split_K):
    """Enqueue C = A1*B + A2*B as one launch (A1 as 2:4 records, A2 as residual lists) on `stream`."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.HeteroSparse_Fused_SpMM_API(ctypes.c_void_p(stream) if stream else None, _ptr(Packed_A1), _ptr(A2_Words),
                                         _ptr(A2_Offsets), LongestList, _ptr(B), _ptr(C), M_Global, N_Global, K_Global,
                                         _ptr(Reduction_Workspace), Split_K)
    if rc != 0:
        raise SpMMError("HeteroSparse_Fused_SpMM_API", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def HeteroSparse_Fused_SpMM_API_Strided(stream, Packed_A1, A2_Words, A2_Offsets, LongestList, B, ldb, C, ldc, M_Global, N_Global,
                                        K_Global, Reduction_Workspace, Split_K, Flags=0):
    """HeteroSparse_Fused_SpMM_API with token strides ldb / ldc (elements) and Flags (SPMM_FLAG_RELU)."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.HeteroSparse_Fused_SpMM_API_Strided(ctypes.c_void_p(stream) if stream else None, _ptr(Packed_A1), _ptr(A2_Words),
                                                 _ptr(A2_Offsets), LongestList, _ptr(B), ldb, _ptr(C), ldc, M_Global, N_Global,
                                                 K_Global, _ptr(Reduction_Workspace), Split_K, Flags)
    if rc != 0:
        raise SpMMError("HeteroSparse_Fused_SpMM_API_Strided", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def HeteroSparse_SpMM_API_RowMajor(stream, Packed_A1, Compressed_A2, TileOffsets_A2, B, C, M_Global, N_Global, K_Global,
                                   Reduction_Workspace, Split_K_A1, Split_K_A2, Flags=0):
    """HeteroSparse_SpMM_API for row-major operands: B[K][N], C[M][N] (and M x N slabs in the workspace)."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.HeteroSparse_SpMM_API_RowMajor(ctypes.c_void_p(stream) if stream else None, _ptr(Packed_A1), _ptr(Compressed_A2),
                                            _ptr(TileOffsets_A2), _ptr(B), _ptr(C), M_Global, N_Global, K_Global,
                                            _ptr(Reduction_Workspace), Split_K_A1, Split_K_A2, Flags)
    if rc != 0:
        raise SpMMError("HeteroSparse_SpMM_API_RowMajor", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def HeteroSparse_Fused_SpMM_API_RowMajor(stream, Packed_A1, A2_Words, A2_Offsets, LongestList, B, C, M_Global, N_Global, K_Global,
                                         Reduction_Workspace, Split_K, Flags=0):
    """HeteroSparse_Fused_SpMM_API for row-major operands (B[K][N], C[M][N]) with Flags (SPMM_FLAG_RELU, ...)."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.HeteroSparse_Fused_SpMM_API_RowMajor(ctypes.c_void_p(stream) if stream else None, _ptr(Packed_A1), _ptr(A2_Words),
                                                  _ptr(A2_Offsets), LongestList, _ptr(B), _ptr(C), M_Global, N_Global, K_Global,
                                                  _ptr(Reduction_Workspace), Split_K, Flags)
    if rc != 0:
        raise SpMMError("HeteroSparse_Fused_SpMM_API_RowMajor", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def HeteroSparse_A1_Partials(stream, Packed_A1, B, Partials, M_Global, N_Global, K_Global, Split_K, RowBlocks=0,
                             Waves=0, ShareB=0):
    """The 2:4 kernel alone, with a caller-chosen launch shape (0, 0 = the library's)."""
    lib = load_library()
    if stream is not None and not isinstance(stream, int):
        stream = stream.cuda_stream
    rc = lib.HeteroSparse_A1_Partials(ctypes.c_void_p(stream) if stream else None, _ptr(Packed_A1), _ptr(B),
                                      _ptr(Partials), M_Global, N_Global, K_Global, Split_K, RowBlocks, Waves, ShareB)
    if rc != 0:
        raise SpMMError("HeteroSparse_A1_Partials", rc, lib.SpMM_GetErrorString(rc).decode())
    return rc


def split_pack_on_device(A_d, want_residual=True, stream=None):
    """2:4 records (uint8 tensor) and dense residual (fp16 tensor, or None) of a torch CUDA fp16 matrix,
    made on the GPU; same bits as HeteroSparse_Decompose + HeteroSparse_PackA1."""
    import torch

    lib = load_library()
    M, K = A_d.shape
    if A_d.dtype != torch.float16 or not A_d.is_contiguous():
        raise TypeError("expected a contiguous float16 CUDA tensor")
    size = lib.HeteroSparse_PackedBytes(M, K)
    if size < 0:
        raise SpMMError("HeteroSparse_PackedBytes", int(size))
    if stream is None:
        stream = torch.cuda.current_stream()
    packed = torch.empty(size, dtype=torch.uint8, device=A_d.device)
    residual = torch.empty_like(A_d) if want_residual else None
    rc = lib.HeteroSparse_DeviceSplitPack(ctypes.c_void_p(stream.cuda_stream) if stream.cuda_stream else None, _ptr(A_d),
                                          M, K, _ptr(packed), _ptr(residual))
    if rc != 0:
        raise SpMMError("HeteroSparse_DeviceSplitPack", rc, lib.SpMM_GetErrorString(rc).decode())
    return packed, residual


def pack_residual_on_device(A2_d, stream=None):
    """Residual lists (words int32 tensor of T + 64, offsets int32 tensor, longest list) of a torch CUDA
    fp16 matrix, made on the GPU; same bits as HeteroSparse_PackA2.  Synchronises once, to size the words."""
    import torch

    lib = load_library()
    M, K = A2_d.shape
    if A2_d.dtype != torch.float16 or not A2_d.is_contiguous():
        raise TypeError("expected a contiguous float16 CUDA tensor")
    if stream is None:
        stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream) if stream.cuda_stream else None
    lists = (M // 16) * (K // 128)
    offsets = torch.empty(max(lists, 0) + 2, dtype=torch.int32, device=A2_d.device)  # the last int: the longest list
    rc = lib.HeteroSparse_DevicePackA2_Offsets(sp, _ptr(A2_d), M, K, _ptr(offsets), ctypes.c_void_p(offsets.data_ptr() + 4 * (lists + 1)))
    if rc != 0:
        raise SpMMError("HeteroSparse_DevicePackA2_Offsets", rc, lib.SpMM_GetErrorString(rc).decode())
    stream.synchronize()
    total, longest = (int(x) for x in offsets[lists:lists + 2].cpu())
    if total < 0:
        raise SpMMError("HeteroSparse_DevicePackA2_Offsets", -1, "more residual values than an int counts")
    if longest > 1024:
        raise SpMMError("HeteroSparse_DevicePackA2_Offsets", -1, "not a residual: a 16 x 128 block with more than 1024 kept values")
    words = torch.empty(total + 64, dtype=torch.int32, device=A2_d.device)
    rc = lib.HeteroSparse_DevicePackA2_Words(sp, _ptr(A2_d), M, K, _ptr(offsets), _ptr(words))
    if rc != 0:
        raise SpMMError("HeteroSparse_DevicePackA2_Words", rc, lib.SpMM_GetErrorString(rc).decode())
    return words, offsets[:lists + 1], longest


"""ctypes binding of libelf_stage.so (the C ABI declared in include/elf_stage.h).

The library is built in-tree by ``__graft_entry__.build()`` (or ``make -C elf_amd/csrc``).
There is no fallback: if the shared object is missing, loading raises.
"""

import ctypes
import logging
import os
from ctypes import c_int, c_int64, c_float, c_double, c_void_p, c_char_p, POINTER

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libelf_stage.so")

TORCH_LIB_PATH = os.path.join(_HERE, "libelf_torch.so")

logger = logging.getLogger("lib")

_lib = None
_torch_allocated = None  # not looked for yet; False: not to be had

# name -> (restype, argtypes); kept in one table so that tests can check the exported symbols
# against the header.
_P = c_void_p
_SIGNATURES = {
	"elf_last_error": (c_char_p, []),
	"elf_abi_version": (c_int, []),
	"elf_gemm_bf16": (c_int, [c_int, c_int, c_int, c_int, c_int, _P, c_int64, _P, c_int64, _P, c_int64, c_int, _P, c_int64, c_int, c_int, _P]),
	"elf_norm_fwd": (c_int, [c_int, _P, _P, _P, _P, _P, c_int, c_int, c_float, _P]),
	"elf_norm_bwd_workspace_floats": (c_int64, [c_int, c_int]),
	"elf_norm_bwd": (c_int, [c_int, _P, _P, _P, _P, _P, _P, _P, _P, _P, c_int, c_int, _P]),
	"elf_gemm_rope_bf16": (c_int, [c_int, c_int, c_int, _P, c_int64, _P, c_int64, _P, c_int64, _P, c_int, c_int, c_int, _P]),
	"elf_gemm_gelu_bwd_bf16": (c_int, [c_int, c_int, c_int, _P, _P, _P, _P, _P, _P]),
	"elf_gemm_way": (c_int, [c_int] * 5),
	"elf_colsum_workspace_floats": (c_int64, [c_int64, c_int]),
	"elf_colsum_bf16": (c_int, [_P, c_int64, _P, c_int64, c_int, _P, _P]),
	"elf_norm_bwd_noalloc": (c_int, [c_int, _P, _P, _P, _P, _P, _P, _P, _P, c_int, c_int, _P]),
	"elf_gelu_fwd": (c_int, [_P, _P, c_int64, _P]),
	"elf_gelu_bwd": (c_int, [_P, _P, _P, c_int64, _P]),
	"elf_gemm_act_bf16": (c_int, [c_int, c_int, c_int, c_int, _P, c_int64, _P, c_int64, _P, c_int64, _P, c_int64, _P]),
	"elf_gemm_swiglu_bwd_bf16": (c_int, [c_int, c_int, c_int, _P, c_int64, _P, c_int64, _P, c_int64, _P, c_int64, _P, _P]),
	"elf_swiglu_fwd": (c_int, [_P, _P, c_int64, c_int, _P]),
	"elf_swiglu_bwd": (c_int, [_P, _P, _P, c_int64, c_int, _P]),
	"elf_rope_table": (c_int, [_P, c_int, c_int, c_double, _P]),
	"elf_rope_apply": (c_int, [_P, _P, c_int64, c_int, c_int, c_int, c_int, c_int, _P]),
	"elf_scale_grads": (c_int, [_P, _P, c_int64, c_float, _P]),
	"elf_add_bf16": (c_int, [_P, _P, _P, c_int64, _P]),
	"elf_embedding_fwd": (c_int, [_P, _P, _P, c_int64, c_int, c_int, _P]),
	"elf_embedding_bwd": (c_int, [_P, _P, _P, c_int64, c_int, c_int, _P]),
	"elf_cross_entropy": (c_int, [_P, c_int64, _P, c_int64, c_int64, c_int64, c_float, _P, _P, _P, c_int64, _P]),
	"elf_cross_entropy_loss": (c_int, [_P, c_int64, c_int, _P, c_int64, c_int64, c_int64, c_float, c_int, _P, _P, _P, c_int64, _P, _P]),
	"elf_cross_entropy_dense": (c_int, [_P, _P, c_int64, c_int64, c_int64, c_float, _P, _P, _P, _P]),
	"elf_scale_by_bf16": (c_int, [_P, _P, _P, c_int64, _P]),
	"elf_cross_entropy_reduce": (c_int, [_P, _P, c_int64, c_int64, _P, _P]),
	"elf_attn_fwd": (c_int, [_P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int, c_int, c_int, c_int, c_int, c_int, c_float, _P]),
	"elf_attn_bwd_workspace_bytes": (c_int64, [c_int, c_int, c_int, c_int, c_int]),
	"elf_gemm_turn_giveups": (c_int, [POINTER(ctypes.c_uint64)]),
	"elf_linear_w_workspace_floats": (c_int64, [c_int, _P, c_int]),
	"elf_linear_w_way": (c_int, [c_int, _P, c_int]),
	"elf_linear_w_pass": (c_int, [c_int, _P, c_int, _P, _P]),
	"elf_gemm_dw_group": (c_int, [c_int, _P, c_int, c_float, _P]),
	"elf_hbm_probe": (c_int, [c_int, _P, _P, c_int64, _P]),
	"elf_prof_enable": (None, [c_int]),
	"elf_prof_collect": (c_int, [c_int, POINTER(c_double), POINTER(c_double)]),
	"elf_prof_launches": (c_int64, [c_int, POINTER(c_double)]),
	"elf_attn_bwd_shared_workspace_bytes": (c_int64, [c_int] * 6),
	"elf_attn_bwd_way": (c_int, [c_int64, _P] + [c_int64] * 3 + [c_int] * 6 + [POINTER(c_int)]),
	"elf_attn_bwd_shared": (c_int, [_P] * 10 + [c_int64] * 9 + [c_int] * 6 + [c_float, _P, _P]),
	"elf_attn_bwd": (c_int, [_P] * 10 + [c_int64] * 8 + [c_int] * 6 + [c_float, _P]),
	"elf_attn_bwd_rope": (c_int, [_P] * 10 + [c_int64] * 8 + [c_int] * 6 + [c_float, _P, _P]),
}


class ElfStageError(RuntimeError):
	"""A C-ABI call returned a negative status."""


def raw_stream():
	"""The current stream of the current device as the library takes it (``torch.cuda.current_stream().cuda_stream`` builds
	a Stream object for the same number: 9 us a call)."""
	return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def exported_symbols():
	return sorted(_SIGNATURES)


def register(name, restype, argtypes):
	"""Add a signature (used by modules that bind further entry points)."""
	_SIGNATURES[name] = (restype, argtypes)
	if _lib is not None:
		fn = getattr(_lib, name)
		fn.restype, fn.argtypes = restype, argtypes


def load():
	"""Load the shared object (once) and type every entry point. Raises if it is not built."""
	global _lib
	if _lib is not None:
		return _lib
	if not os.path.exists(LIB_PATH):
		raise ElfStageError(
			f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; g.build()'` "
			"or `make -C elf_amd/csrc`. There is no non-HIP fallback."
		)
	lib = ctypes.CDLL(LIB_PATH)
	for name, (restype, argtypes) in _SIGNATURES.items():
		fn = getattr(lib, name)
		fn.restype, fn.argtypes = restype, argtypes
	_lib = lib
	return lib


def _torch_reader():
	"""libelf_torch.so's reading of PyTorch's caching allocator, or False where the library is missing, does not load or was built for another
	PyTorch than this one."""
	if not os.path.exists(TORCH_LIB_PATH):
		return False
	try:
		lib = ctypes.CDLL(TORCH_LIB_PATH)
		lib.elf_torch_built_for.restype = c_char_p
		built_for, fn = lib.elf_torch_built_for().decode(), lib.elf_torch_allocated
	except (OSError, AttributeError) as e:
		logger.warning("%s is not used: %s", TORCH_LIB_PATH, e)
		return False
	if built_for != torch.__version__:
		logger.warning("%s is not used: built for PyTorch %s, this is %s", TORCH_LIB_PATH, built_for, torch.__version__)
		return False
	fn.restype, fn.argtypes = c_int, [c_int, _P]
	return fn


def torch_allocated(device):
	"""(allocated, peak) bytes of PyTorch's caching allocator on ``device`` through libelf_torch.so, or None without that library."""
	global _torch_allocated
	if _torch_allocated is None:
		_torch_allocated = _torch_reader()
	if _torch_allocated is False:
		return None
	out = (c_int64 * 2)()
	return (out[0], out[1]) if _torch_allocated(device, out) == 0 else None


def check(rc, what=""):
	if rc != 0:
		msg = load().elf_last_error().decode()
		raise ElfStageError(f"{what} failed (rc={rc}): {msg}")

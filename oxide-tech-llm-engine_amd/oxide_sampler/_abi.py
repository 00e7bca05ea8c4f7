"""ctypes view of include/oxide_sampler.h (the C ABI of liboxide_sampler.so).

The structures mirror the header field for field; `check_layout()` compares
their sizes with the C definitions compiled into the library's tests.
"""
from __future__ import annotations

import ctypes
import os
from pathlib import Path

PKG_ROOT = Path(__file__).resolve().parent.parent  # oxide-tech-llm-engine_amd/
LIB_PATH = PKG_ROOT / "lib" / "liboxide_sampler.so"

OXS_ABI_VERSION = 4

OXS_OK = 0
OXS_ERR_INVALID_ARGUMENT = -1
OXS_ERR_SHAPE_MISMATCH = -2
OXS_ERR_LIMITS = -3
OXS_ERR_HIP = -4
OXS_ERR_UNSUPPORTED = -5
OXS_ERR_NO_DEVICE = -6
OXS_ERR_TIMEOUT = -7

OXS_ROW_OK = 0
OXS_ROW_EMPTY = 1
OXS_ROW_HISTORY_FULL = 2
OXS_ROW_UNSUPPORTED = 3
OXS_ROW_MISSING_STATE = 4

OXS_MIROSTAT_DISABLED = 0
OXS_MIROSTAT_V1 = 1
OXS_MIROSTAT_V2 = 2

OXS_DTYPE_F32 = 0
OXS_DTYPE_BF16 = 1

OXS_FLAG_RECORD_HISTORY = 1
OXS_FLAG_SHARED_CONFIG = 2

OXS_PATH_BUCKETS = 0
OXS_PATH_SORT = 1
OXS_PATH_EXACT = 2
OXS_PATH_NONE = 3

OXS_STATIC_MAX_BATCH = 256
OXS_STATIC_MAX_VOCAB = 524288

# Exported symbols declared in include/oxide_sampler.h.
EXPORTED_SYMBOLS = (
    "oxs_abi_version",
    "oxs_status_string",
    "oxs_sampling_config_default",
    "oxs_rng_state_from_seed",
    "oxs_mirostat_mu_from_tau",
    "oxs_sampler_create",
    "oxs_sampler_destroy",
    "oxs_sampler_workspace_bytes",
    "oxs_sampler_count_paths",
    "oxs_sampler_path_counts",
    "oxs_sampler_record_rows",
    "oxs_read_floor",
    "oxs_sample_batch",
    "oxs_sample_batch_static",
    "oxs_decode_step",
    "oxs_argmax",
    "oxs_host_alloc",
    "oxs_host_free",
    "oxs_host_wait",
    "oxs_dfa_mask",
    "oxs_dfa_mask_gather",
    "oxs_gbnf_mask",
    "oxs_ascii_mask",
    "oxs_quantize_q8_1",
    "oxs_q8_0_packed_bytes",
    "oxs_pack_q8_0",
    "oxs_mmvq_q8_0",
)

OXS_DFA_ERROR_STATE = 0xFFFFFFFF


class OxsSamplingConfig(ctypes.Structure):
    _fields_ = [
        ("temperature", ctypes.c_float),
        ("top_k", ctypes.c_uint32),
        ("top_p", ctypes.c_float),
        ("min_p", ctypes.c_float),
        ("tfs_z", ctypes.c_float),
        ("typical_p", ctypes.c_float),
        ("xtc_threshold", ctypes.c_float),
        ("xtc_probability", ctypes.c_float),
        ("mirostat_mode", ctypes.c_int32),
        ("mirostat_tau", ctypes.c_float),
        ("mirostat_eta", ctypes.c_float),
        ("dry_multiplier", ctypes.c_float),
        ("dry_base", ctypes.c_float),
        ("dry_allowed_length", ctypes.c_uint32),
        ("dry_range", ctypes.c_uint32),
        ("repeat_penalty", ctypes.c_float),
        ("repeat_last_n", ctypes.c_uint32),
        ("frequency_penalty", ctypes.c_float),
        ("presence_penalty", ctypes.c_float),
        ("penalize_nl", ctypes.c_uint32),
        ("newline_penalty", ctypes.c_float),
        ("newline_token_id", ctypes.c_uint32),
        ("bias_offset", ctypes.c_uint32),
        ("bias_count", ctypes.c_uint32),
        ("ban_offset", ctypes.c_uint32),
        ("ban_count", ctypes.c_uint32),
    ]


class OxsLimits(ctypes.Structure):
    _fields_ = [
        ("max_batch", ctypes.c_uint32),
        ("max_vocab", ctypes.c_uint32),
        ("max_top_k", ctypes.c_uint32),
        ("max_dry_ids", ctypes.c_uint32),
    ]


class OxsBatch(ctypes.Structure):
    _fields_ = [
        ("batch", ctypes.c_uint32),
        ("vocab", ctypes.c_uint32),
        ("logits_dtype", ctypes.c_int32),
        ("flags", ctypes.c_uint32),
        ("logits_ld", ctypes.c_int64),
        ("logits", ctypes.c_void_p),
        ("configs", ctypes.c_void_p),
        ("bias_ids", ctypes.c_void_p),
        ("bias_values", ctypes.c_void_p),
        ("ban_ids", ctypes.c_void_p),
        ("allowed_mask", ctypes.c_void_p),
        ("mask_ld", ctypes.c_int64),
        ("history", ctypes.c_void_p),
        ("history_ld", ctypes.c_int64),
        ("history_len", ctypes.c_void_p),
        ("history_cap", ctypes.c_uint32),
        ("uniforms", ctypes.c_void_p),
        ("rng_state", ctypes.c_void_p),
        ("mirostat_mu", ctypes.c_void_p),
        ("out_tokens", ctypes.c_void_p),
        ("out_status", ctypes.c_void_p),
        ("out_kept_count", ctypes.c_void_p),
        ("out_kept_ids", ctypes.c_void_p),
        ("out_kept_probs", ctypes.c_void_p),
        ("kept_ld", ctypes.c_int64),
        ("logits_out", ctypes.c_void_p),
        ("logits_out_ld", ctypes.c_int64),
        ("logit_softcap", ctypes.c_float),
    ]


class OxsDfa(ctypes.Structure):
    _fields_ = [
        ("num_states", ctypes.c_uint32),
        ("transitions", ctypes.c_void_p),
    ]


class OxsTokenBytes(ctypes.Structure):
    _fields_ = [
        ("vocab", ctypes.c_uint32),
        ("num_bytes", ctypes.c_uint32),
        ("offsets", ctypes.c_void_p),
        ("bytes", ctypes.c_void_p),
    ]


class OxsGbnfRule(ctypes.Structure):
    _fields_ = [
        ("num_ranges", ctypes.c_uint32),
        ("ranges", ctypes.c_void_p),
        ("num_literals", ctypes.c_uint32),
        ("literal_offsets", ctypes.c_void_p),
        ("literal_bytes", ctypes.c_void_p),
    ]


class OxsDecodeIo(ctypes.Structure):
    _fields_ = [
        ("current_token", ctypes.c_void_p),
        ("current_position", ctypes.c_void_p),
        ("generated_count", ctypes.c_void_p),
        ("host_tokens", ctypes.c_void_p),
    ]


_lib = None


class LibraryMissing(RuntimeError):
    """Raised when liboxide_sampler.so has not been built: there is no fallback."""


def load_library(path: os.PathLike | str | None = None) -> ctypes.CDLL:
    """Loads liboxide_sampler.so and declares its prototypes. Fails loudly."""
    global _lib
    if _lib is not None and path is None:
        return _lib
    p = Path(path) if path else LIB_PATH
    if not p.exists():
        raise LibraryMissing(
            f"{p} is not built; run `make -C oxide-tech-llm-engine_amd` or "
            "`python -c 'import __graft_entry__; __graft_entry__.build()'`")
    lib = ctypes.CDLL(str(p))
    lib.oxs_abi_version.restype = ctypes.c_uint32
    lib.oxs_abi_version.argtypes = []
    lib.oxs_status_string.restype = ctypes.c_char_p
    lib.oxs_status_string.argtypes = [ctypes.c_int]
    lib.oxs_sampling_config_default.restype = None
    lib.oxs_sampling_config_default.argtypes = [ctypes.POINTER(OxsSamplingConfig)]
    lib.oxs_rng_state_from_seed.restype = ctypes.c_uint64
    lib.oxs_rng_state_from_seed.argtypes = [ctypes.c_int, ctypes.c_uint64]
    lib.oxs_mirostat_mu_from_tau.restype = ctypes.c_float
    lib.oxs_mirostat_mu_from_tau.argtypes = [ctypes.c_float]
    lib.oxs_sampler_create.restype = ctypes.c_int
    lib.oxs_sampler_create.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.POINTER(OxsLimits), ctypes.c_int]
    lib.oxs_sampler_destroy.restype = ctypes.c_int
    lib.oxs_sampler_destroy.argtypes = [ctypes.c_void_p]
    lib.oxs_sampler_workspace_bytes.restype = ctypes.c_size_t
    lib.oxs_sampler_workspace_bytes.argtypes = [ctypes.c_void_p]
    lib.oxs_sampler_count_paths.restype = ctypes.c_int
    lib.oxs_sampler_count_paths.argtypes = [ctypes.c_void_p, ctypes.c_int]
    lib.oxs_sampler_path_counts.restype = ctypes.c_int
    lib.oxs_sampler_path_counts.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_uint32)]
    lib.oxs_sampler_record_rows.restype = ctypes.c_int
    lib.oxs_sampler_record_rows.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_uint32)]
    lib.oxs_sample_batch.restype = ctypes.c_int
    lib.oxs_sample_batch.argtypes = [ctypes.c_void_p, ctypes.POINTER(OxsBatch), ctypes.c_void_p]
    lib.oxs_read_floor.restype = ctypes.c_int
    lib.oxs_read_floor.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_int64, ctypes.c_uint32,
                                   ctypes.c_void_p, ctypes.c_void_p]
    lib.oxs_sample_batch_static.restype = ctypes.c_int
    lib.oxs_sample_batch_static.argtypes = [ctypes.POINTER(OxsBatch), ctypes.c_void_p]
    lib.oxs_decode_step.restype = ctypes.c_int
    lib.oxs_decode_step.argtypes = [ctypes.c_void_p, ctypes.POINTER(OxsBatch), ctypes.POINTER(OxsDecodeIo),
                                    ctypes.c_void_p]
    lib.oxs_argmax.restype = ctypes.c_int
    lib.oxs_argmax.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_int64, ctypes.c_uint32, ctypes.c_void_p,
                               ctypes.c_void_p, ctypes.c_void_p]
    lib.oxs_host_alloc.restype = ctypes.c_int
    lib.oxs_host_alloc.argtypes = [ctypes.c_size_t, ctypes.POINTER(ctypes.c_void_p)]
    lib.oxs_host_free.restype = ctypes.c_int
    lib.oxs_host_free.argtypes = [ctypes.c_void_p]
    lib.oxs_host_wait.restype = ctypes.c_int
    lib.oxs_host_wait.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_void_p,
                                  ctypes.c_uint64]
    lib.oxs_dfa_mask.restype = ctypes.c_int
    lib.oxs_dfa_mask.argtypes = [ctypes.POINTER(OxsDfa), ctypes.POINTER(OxsTokenBytes), ctypes.c_void_p,
                                 ctypes.c_uint32, ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p]
    lib.oxs_dfa_mask_gather.restype = ctypes.c_int
    lib.oxs_dfa_mask_gather.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_int64, ctypes.c_uint32,
                                        ctypes.c_void_p, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_int64,
                                        ctypes.c_void_p]
    lib.oxs_gbnf_mask.restype = ctypes.c_int
    lib.oxs_gbnf_mask.argtypes = [ctypes.POINTER(OxsGbnfRule), ctypes.POINTER(OxsTokenBytes), ctypes.c_void_p,
                                  ctypes.c_void_p]
    lib.oxs_ascii_mask.restype = ctypes.c_int
    lib.oxs_ascii_mask.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint32, ctypes.c_void_p,
                                   ctypes.c_void_p]
    lib.oxs_quantize_q8_1.restype = ctypes.c_int
    lib.oxs_quantize_q8_1.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_void_p]
    lib.oxs_q8_0_packed_bytes.restype = ctypes.c_size_t
    lib.oxs_q8_0_packed_bytes.argtypes = [ctypes.c_uint32, ctypes.c_uint32]
    lib.oxs_pack_q8_0.restype = ctypes.c_int
    lib.oxs_pack_q8_0.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_void_p]
    lib.oxs_mmvq_q8_0.restype = ctypes.c_int
    lib.oxs_mmvq_q8_0.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint32,
                                  ctypes.c_uint32, ctypes.c_uint32, ctypes.c_void_p]
    if lib.oxs_abi_version() != OXS_ABI_VERSION:
        raise RuntimeError(f"liboxide_sampler ABI {lib.oxs_abi_version()} != {OXS_ABI_VERSION}")
    if path is None:
        _lib = lib
    return lib


class OxsError(RuntimeError):
    def __init__(self, code: int, what: str = ""):
        self.code = code
        lib = _lib
        text = lib.oxs_status_string(code).decode() if lib is not None else str(code)
        super().__init__(f"{what}: {text} ({code})" if what else f"{text} ({code})")


def check(code: int, what: str = "") -> None:
    if code != OXS_OK:
        raise OxsError(code, what)

"""Binding of include/mi355x_search.h for Python callers.  Device memory is supplied by the caller as torch CUDA
tensors; this module only passes pointers.  The per-step calls are methods of native base classes (the extension
module `_binding`, built from binding/torch_binding.cpp); what runs once -- creating, destroying, diagnostics -- goes
through ctypes.  There is no CPU fallback: if a shared library is missing, loading fails."""
import ctypes as C
import os

import torch

try:
    from . import _binding
    from ._binding import argmax_static  # noqa: F401
except ImportError as e:
    raise ImportError(f"the native binding _binding.so cannot be loaded ({e}): build it with __graft_entry__.build()") from e

_HERE = os.path.dirname(os.path.abspath(__file__))
MI355X_F32 = 1
MI355X_F16 = 10
MAX_EOS = 16


def library_path():
    return os.path.join(_HERE, "libmi355x_search.so")


class LogitsXformC(C.Structure):
    _fields_ = [("mask", C.c_void_p), ("history", C.c_void_p), ("history_stride", C.c_int32),
                ("history_len", C.c_int32), ("repetition_penalty", C.c_float), ("apply_min_length", C.c_int32),
                ("n_eos", C.c_int32), ("eos_ids", C.c_int32 * MAX_EOS), ("history_lens", C.c_void_p),
                ("min_length", C.c_int32), ("no_repeat_ngram_size", C.c_int32), ("mask_allowed_max", C.c_int32)]


class SampleParams(C.Structure):
    _fields_ = [("k", C.c_int32), ("p", C.c_float), ("temperature", C.c_float)]


_lib = None


def load_library():
    global _lib
    if _lib is not None:
        return _lib
    path = library_path()
    if not os.path.exists(path):
        raise RuntimeError(f"{path} is missing: build it with __graft_entry__.build() (hipcc, gfx950); "
                           "there is no CPU fallback")
    L = C.CDLL(path)
    vp, i32, i64, f32 = C.c_void_p, C.c_int, C.c_int64, C.c_float
    L.mi355x_search_create.argtypes = [i32, i32, i32, C.POINTER(vp)]
    L.mi355x_search_destroy.argtypes = [vp]
    L.mi355x_search_destroy.restype = None
    L.mi355x_search_last_error.restype = C.c_char_p
    L.mi355x_search_workspace_bytes.argtypes = [vp]
    L.mi355x_search_workspace_bytes.restype = C.c_size_t
    L.mi355x_process_logits.argtypes = [vp, vp, vp, i64, i32, i32, C.POINTER(LogitsXformC)]
    L.mi355x_argmax.argtypes = [vp, vp, vp, i32, i64, i32, i32, C.POINTER(LogitsXformC), vp]
    L.mi355x_argmax_static.argtypes = [vp, vp, i32, i64, i32, i32, C.POINTER(LogitsXformC), vp]
    L.mi355x_sample.argtypes = [vp, vp, vp, i64, i32, i32, C.POINTER(LogitsXformC), SampleParams,
                                C.POINTER(SampleParams), vp, vp, vp, vp, vp, i32]
    L.mi355x_sample_typed.argtypes = [vp, vp, vp, i32, i64, i32, i32, C.POINTER(LogitsXformC), SampleParams,
                                      C.POINTER(SampleParams), vp, vp, vp, vp, vp, i32]
    L.mi355x_sample_scattered.argtypes = [vp, vp, C.POINTER(vp), i32, i32, i32, C.POINTER(LogitsXformC), SampleParams,
                                          C.POINTER(SampleParams), vp, vp, vp, vp, vp, i32]
    L.mi355x_search_fallback_rows.argtypes = [vp, vp, C.POINTER(C.c_uint)]
    L.mi355x_search_wait_gave_up.argtypes = [vp, vp, C.POINTER(C.c_int)]
    L.mi355x_search_set_poll_limit.argtypes = [vp, C.c_int]
    L.mi355x_search_sum_waits_gave_up.argtypes = [vp, vp, C.POINTER(C.c_uint)]
    for name, args in {
        "mi355x_topk_scores": [vp, vp, vp, i32, i64, i32, i32, i32, vp, vp],
        "mi355x_softmax": [vp, vp, vp, i64, i32, i32, f32, i32],
        "mi355x_beam_select": [vp, vp, vp, i32, i64, i32, i32, i32, vp, vp, vp, vp],
        "mi355x_beam_scorer_create": [vp, i32, i32, i32, i32, C.POINTER(C.c_int32), i32, f32, i32, C.POINTER(vp)],
        "mi355x_beam_scorer_set_prompt": [vp, vp, C.POINTER(C.c_int32), i32],
        "mi355x_draw_in_order": [vp, vp, vp, vp, vp, i32, i32, vp, vp, vp, vp],
        "mi355x_beam_scorer_step": [vp, vp, vp, vp, vp],
        "mi355x_beam_search_step": [vp, vp, vp, i32, i64, i32],
        "mi355x_beam_scorer_is_done": [vp, vp, C.POINTER(C.c_int)],
        "mi355x_beam_scorer_hypothesis": [vp, vp, i32, i32, C.POINTER(C.c_int32), i32, C.POINTER(C.c_int),
                                          C.POINTER(C.c_float)],
        "mi355x_kv_gather": [vp, vp, C.POINTER(vp), C.POINTER(vp), i32, vp, i32, C.c_size_t],
        "mi355x_spec_verify": [vp, vp, vp, vp, vp, vp, vp, i32, i32, i32, vp, vp],
        "mi355x_spec_verify_sparse": [vp, vp, vp, vp, vp, i32, vp, vp, vp, i32, vp, vp, vp, i32, i32, i32, vp, vp, vp],
        "mi355x_greedy_tail": [vp, vp, vp, vp, i32, C.POINTER(C.c_int32), i32, i32, vp, i32, i32, vp],
        "mi355x_cast": [vp, vp, vp, i32, vp, i32, C.c_size_t],
        "mi355x_logits_handoff": [vp, vp, vp, i32, i32, i32, i32, C.POINTER(C.c_int32), vp, i64],
    }.items():
        if hasattr(L, name):
            getattr(L, name).argtypes = args
    if hasattr(L, "mi355x_beam_scorer_destroy"):
        L.mi355x_beam_scorer_destroy.argtypes = [vp]
        L.mi355x_beam_scorer_destroy.restype = None
        for n in ("next_scores", "next_tokens", "next_indices"):
            f = getattr(L, "mi355x_beam_scorer_" + n)
            f.argtypes = [vp]
            f.restype = vp
        L.mi355x_beam_scorer_sequences.argtypes = [vp, C.POINTER(C.c_int)]
        L.mi355x_beam_scorer_sequences.restype = vp
    _lib = L
    return L


class LogitsXform:
    """Python-side description of the fused logits processing (mask / min length / repetition penalty /
    no-repeat n-grams).  Holds references to the tensors so they outlive the asynchronous call.
    shared_history=True lets every row read the one history row given (stride 0), with history_lens
    telling how much of it each row sees: the verify rows of speculative decoding."""

    def __init__(self, mask=None, history=None, history_len=None, repetition_penalty=1.0, eos_ids=(),
                 apply_min_length=False, history_lens=None, min_length=0, no_repeat_ngram_size=0,
                 shared_history=False, mask_allowed_max=0):
        self.mask, self.history, self.history_lens = mask, history, history_lens
        c = self.c = LogitsXformC()
        self._addr = C.addressof(c)  # what the native calls read
        c.mask = mask.data_ptr() if mask is not None else None
        if mask is not None:
            assert mask.dtype == torch.int32 and mask.is_cuda and mask.is_contiguous()
        if history is not None:
            assert history.dtype == torch.int32 and history.is_cuda and history.is_contiguous() and history.dim() == 2
            c.history = history.data_ptr()
            c.history_stride = 0 if shared_history else history.shape[1]
            c.history_len = history.shape[1] if history_len is None else history_len
        if history_lens is not None:
            assert history_lens.dtype == torch.int32 and history_lens.is_cuda and history_lens.is_contiguous()
            c.history_lens = history_lens.data_ptr()
        c.repetition_penalty = repetition_penalty
        c.apply_min_length = int(apply_min_length)
        c.min_length = min_length
        c.no_repeat_ngram_size = no_repeat_ngram_size
        c.mask_allowed_max = mask_allowed_max
        c.n_eos = len(eos_ids)
        for i, e in enumerate(eos_ids):
            c.eos_ids[i] = e


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


class SearchContext(_binding.Context):
    """Owns a mi355x_search_ctx.  All tensor arguments must be CUDA tensors on the context's device.  The calls
    themselves (sample, argmax, softmax, ...) are methods of the native base class."""

    def __init__(self, max_rows, max_vocab, device=0):
        self.L = load_library()
        torch.cuda.init()
        h = C.c_void_p()
        self._check(self.L.mi355x_search_create(device, max_rows, max_vocab, C.byref(h)))
        self.h = h
        self.device = torch.device("cuda", device)
        self._attach(h.value, device)

    def close(self):
        if getattr(self, "h", None):
            self._attach(0, 0)
            self.L.mi355x_search_destroy(self.h)
            self.h = None

    __del__ = close

    def _check(self, rc):
        if rc != 0:
            raise RuntimeError(f"mi355x_search error {rc}: {self.L.mi355x_search_last_error().decode()}")

    def workspace_bytes(self):
        return self.L.mi355x_search_workspace_bytes(self.h)

    def fallback_rows(self):
        n = C.c_uint()
        self._check(self.L.mi355x_search_fallback_rows(self.h, _stream(), C.byref(n)))
        return n.value

    def wait_gave_up(self):
        g = C.c_int()
        self._check(self.L.mi355x_search_wait_gave_up(self.h, _stream(), C.byref(g)))
        return bool(g.value)

    def sum_waits_gave_up(self):
        n = C.c_uint()
        self._check(self.L.mi355x_search_sum_waits_gave_up(self.h, _stream(), C.byref(n)))
        return n.value

    def set_poll_limit(self, polls):
        self._check(self.L.mi355x_search_set_poll_limit(self.h, int(polls)))


class BeamScorer(_binding.Scorer):
    """Device-resident BeamSearchScorer + Sequences (mi355x_beam_scorer).  The steps and the views of the state (step,
    search_step, is_done, next_scores, next_tokens, next_indices, sequences) belong to the native base class."""

    def __init__(self, ctx, batch, beams, max_length, pad, eos, length_penalty=1.0, early_stopping=True):
        self.ctx, self.L = ctx, ctx.L
        self.batch, self.beams, self.max_length = batch, beams, max_length
        e = (C.c_int32 * max(1, len(eos)))(*eos)
        h = C.c_void_p()
        ctx._check(self.L.mi355x_beam_scorer_create(ctx.h, batch, beams, max_length, pad, e, len(eos),
                                                    length_penalty, int(early_stopping), C.byref(h)))
        self.h = h
        self._attach(h.value, ctx.device.index, batch * beams, max_length)

    def close(self):
        if getattr(self, "h", None):
            self._attach(0, 0, 0, 0)
            self.L.mi355x_beam_scorer_destroy(self.h)
            self.h = None

    __del__ = close

    def set_prompt(self, tokens):
        import numpy as np
        t = np.ascontiguousarray(tokens, dtype=np.int32)
        assert t.shape[0] == self.batch
        self.ctx._check(self.L.mi355x_beam_scorer_set_prompt(self.h, _stream(), t.ctypes.data_as(C.POINTER(C.c_int32)),
                                                             t.shape[1]))

    def next_scores_ptr(self):
        return self.L.mi355x_beam_scorer_next_scores(self.h)

    def hypothesis(self, batch, index):
        buf = (C.c_int32 * self.max_length)()
        n = C.c_int()
        sc = C.c_float()
        self.ctx._check(self.L.mi355x_beam_scorer_hypothesis(self.h, _stream(), batch, index, buf, self.max_length,
                                                             C.byref(n), C.byref(sc)))
        return list(buf[:n.value]), sc.value

"""The host library built over tests/gpu_stub.c (device calls on host memory):
its decisions about passes, buffers and fallbacks, tested without a GPU."""
import ctypes as C
import glob
import os
import subprocess

import numpy as np

import rustfox_amd as rf
from rustfox_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DONE = ["batch_gemv_rmsnorm", "batch_gate_up_silu"]
UNUSED = ["argmax", "dequant", "event_create", "event_destroy", "event_record", "event_record_copy",
          "event_sync", "event_wait", "gemv_i8", "gemv_multi", "graph_begin", "graph_end",
          "graph_free", "graph_launch", "kv_write", "quantize", "rope_store", "silu_mul",
          "stage_async", "tensor_load_async"]


def build(folder):
    so = os.path.join(folder, "libfox_stub.so")
    subprocess.run(["gcc", "-std=c11", "-O1", "-fPIC", "-shared", "-ffp-contract=off", "-D_GNU_SOURCE",
                    "-o", so, *sorted(glob.glob(os.path.join(ROOT, "rustfox_amd", "host", "*.c"))),
                    os.path.join(ROOT, "tests", "gpu_stub.c"), "-Wl,-Bsymbolic", "-lpthread", "-lm",
                    *[f"-Wl,--defsym,fox_gpu_{n}=stub_ok" for n in DONE],
                    *[f"-Wl,--defsym,fox_gpu_{n}=stub_refused" for n in UNUSED]], check=True)
    L = C.CDLL(so)
    vp, sz, u32p, f32p = C.c_void_p, C.c_size_t, C.POINTER(C.c_uint32), C.POINTER(C.c_float)
    for name, args, res in (("fox_model_open", [C.c_char_p, C.c_int, C.c_uint64, C.POINTER(vp)], C.c_int),
                            ("fox_model_close", [vp], None),
                            ("fox_context_create", [vp, C.POINTER(rf.ContextConfig), C.POINTER(vp)], C.c_int),
                            ("fox_context_destroy", [vp], None),
                            ("fox_context_set_position", [vp, C.c_uint32], C.c_int),
                            ("fox_context_position", [vp], C.c_uint32),
                            ("fox_eval", [vp, u32p, sz, C.POINTER(f32p)], C.c_int),
                            ("fox_eval_all", [vp, u32p, sz, f32p], C.c_int),
                            ("fox_last_error", [], C.c_char_p)):
        f = getattr(L, name)
        f.argtypes, f.restype = args, res
    return L


class StubModel:
    """A small ternary model opened through the stub."""

    def __init__(self, lib, path, **over):
        s = synth.spec("tiny-512", n_layer=2, n_vocab=600, **over)
        synth.write_gguf(path, s)
        self.lib, self.vocab = lib, s.n_vocab
        for name in ("fail_above", "mallocs", "live", "max_batch", "eights", "batches", "small_attn"):
            self.set(name, 0)
        self.set("head_rows", s.n_vocab)
        C.c_int.in_dll(lib, "stub_fail_attention").value = 0
        self.m = C.c_void_p()
        assert lib.fox_model_open(path.encode(), rf.WEIGHTS_DEVICE, 0, C.byref(self.m)) == 0

    def get(self, name):
        return C.c_size_t.in_dll(self.lib, "stub_" + name).value

    def set(self, name, v):
        C.c_size_t.in_dll(self.lib, "stub_" + name).value = v

    def fail_attention(self, n):
        C.c_int.in_dll(self.lib, "stub_fail_attention").value = n

    def context(self, n_ctx, n_batch):
        cfg = rf.ContextConfig(n_ctx=n_ctx, n_batch=n_batch, n_threads=0)
        c = C.c_void_p()
        assert self.lib.fox_context_create(self.m, C.byref(cfg), C.byref(c)) == 0
        return c

    def eval(self, c, ids):
        """(status, pointer to the logits)"""
        a = np.ascontiguousarray(ids, np.uint32)
        p = C.POINTER(C.c_float)()
        st = self.lib.fox_eval(c, a.ctypes.data_as(C.POINTER(C.c_uint32)), a.size, C.byref(p))
        return st, p

    def row(self, p):
        return np.ctypeslib.as_array(p, shape=(self.vocab,)).copy()

    def eval_all(self, c, ids):
        a = np.ascontiguousarray(ids, np.uint32)
        out = np.full((a.size, self.vocab), -1, np.float32)
        st = self.lib.fox_eval_all(c, a.ctypes.data_as(C.POINTER(C.c_uint32)), a.size,
                                   out.ctypes.data_as(C.POINTER(C.c_float)))
        return st, out

    def want(self, ids):
        """The stub's logits after each of these tokens."""
        ids = np.asarray(ids, np.float32)
        return ids[:, None] * np.float32(self.vocab) + np.arange(self.vocab, dtype=np.float32)

    def close(self):
        self.lib.fox_model_close(self.m)

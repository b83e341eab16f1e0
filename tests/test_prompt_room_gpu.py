"""Prompts on a card without room for the long pass (2048 tokens): they go through in
passes of 512, and the decoder does not try the long one again (every try frees all of the
pass's buffers).  The tuning build says how many rows there is room for."""
import ctypes
import os

import numpy as np
import pytest

from _util import rel_err
from test_wg_merge_gpu import _Cfg, _F16W, _model

pytestmark = pytest.mark.gpu
L, H, D, V, S = 2, 8, 128, 512, 2304


@pytest.fixture
def lib(gpu):
    import llm_capi
    lib = llm_capi.load_tune()
    lib.llm_decoder_create.argtypes = [ctypes.POINTER(_Cfg), ctypes.POINTER(ctypes.c_void_p)]
    lib.llm_decoder_set_f16_weights.argtypes = [ctypes.c_void_p, ctypes.POINTER(_F16W)]
    lib.llm_decoder_begin_synthetic.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int,
                                                ctypes.c_uint64, ctypes.c_int]
    lib.llm_decoder_prefill.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int]
    lib.llm_decoder_step.argtypes = [ctypes.c_void_p] * 5
    lib.llm_decoder_sync.argtypes = [ctypes.c_void_p]
    lib.llm_decoder_destroy.argtypes = [ctypes.c_void_p]
    lib.llm_decoder_destroy.restype = None
    yield lib
    os.environ.pop("LLM_PREFILL_ROOM", None)


class _Decoders:
    def __init__(self, lib):
        import torch
        self.lib, self.all = lib, []
        self.w = _model(np.random.default_rng(8), L, H, D, V)
        self.tok = np.random.default_rng(9).integers(0, V, S).astype(np.int32)
        self.logits = torch.empty((1, V), device="cuda")

    def make(self):
        import llm_capi
        cfg, dec = _Cfg(L, H, D, H * D, V, S, 0, 16, llm_capi.LLM_F16, 1, D ** -0.5, 0), ctypes.c_void_p()
        llm_capi.check(self.lib.llm_decoder_create(ctypes.byref(cfg), ctypes.byref(dec)), self.lib)
        self.all.append(dec)
        ww = _F16W(*[self.w[k].ctypes.data for k in ("emb", "ln1_g", "ln1_b", "ln2_g", "ln2_b", "wqkv",
                                                      "wo", "w1", "w2", "b1", "b2")])
        llm_capi.check(self.lib.llm_decoder_set_f16_weights(dec, ctypes.byref(ww)), self.lib)
        return dec

    def prompt(self, dec, n=1300):
        """(logits after a prompt of n tokens and one step, bytes of the card that it took)"""
        import torch
        import llm_capi
        lib, tok = self.lib, self.tok
        llm_capi.check(lib.llm_decoder_begin_synthetic(dec, 1, 0, 1, 0), lib)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        llm_capi.check(lib.llm_decoder_prefill(dec, 0, tok.ctypes.data, n), lib)
        taken = free - torch.cuda.mem_get_info()[0]
        llm_capi.check(lib.llm_decoder_step(dec, tok[n:].ctypes.data, self.logits.data_ptr(), None, None), lib)
        llm_capi.check(lib.llm_decoder_sync(dec), lib)
        return self.logits[0].cpu().numpy().copy(), taken


@pytest.fixture
def decoders(lib):
    d = _Decoders(lib)
    yield d
    for dec in d.all:
        lib.llm_decoder_destroy(dec)


def test_short_passes_and_no_second_try(decoders):
    import llm_capi
    d = decoders
    whole, took = d.prompt(d.make())
    os.environ["LLM_PREFILL_ROOM"] = "512"
    dec = d.make()
    short, first = d.prompt(dec)
    assert 0 < first < took
    # chunks split the sums of the attention otherwise: as whole prompts against steps
    assert rel_err(short, whole) < 1e-3
    del os.environ["LLM_PREFILL_ROOM"]
    again, more = d.prompt(dec)
    assert more == 0  # there would be room now, but no one asks
    np.testing.assert_array_equal(again, short)
    os.environ["LLM_PREFILL_ROOM"] = "100"  # nor is there room for the short pass
    dec = d.make()
    with pytest.raises(llm_capi.LlmError) as e:
        d.prompt(dec)
    assert e.value.status == llm_capi.LLM_ERR_OOM
    os.environ["LLM_PREFILL_ROOM"] = "512"  # later there is
    late, _ = d.prompt(dec)
    np.testing.assert_array_equal(late, short)


def test_growing_prompts(decoders):
    """The pass's buffers grow by whole short passes, not by each longer prompt."""
    dec = decoders.make()
    taken = [decoders.prompt(dec, n)[1] for n in (513, 600, 1000, 1024, 1025, 1500, 1030)]
    assert taken[0] > 0 and taken[4] > 0
    assert [t for i, t in enumerate(taken) if i not in (0, 4)] == [0] * 5, taken

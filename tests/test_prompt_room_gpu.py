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


def test_short_passes_and_no_second_try(lib):
    import torch
    import llm_capi
    w = _model(np.random.default_rng(8), L, H, D, V)
    tok = np.random.default_rng(9).integers(0, V, 1301).astype(np.int32)
    logits = torch.empty((1, V), device="cuda")

    def prompt(dec):
        """(logits after the prompt, bytes of the card that it took)"""
        llm_capi.check(lib.llm_decoder_begin_synthetic(dec, 1, 0, 1, 0), lib)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        llm_capi.check(lib.llm_decoder_prefill(dec, 0, tok.ctypes.data, tok.size - 1), lib)
        taken = free - torch.cuda.mem_get_info()[0]
        llm_capi.check(lib.llm_decoder_step(dec, tok[-1:].ctypes.data, logits.data_ptr(), None, None), lib)
        llm_capi.check(lib.llm_decoder_sync(dec), lib)
        return logits[0].cpu().numpy().copy(), taken

    decs = []

    def make():
        cfg, dec = _Cfg(L, H, D, H * D, V, S, 0, 16, llm_capi.LLM_F16, 1, D ** -0.5, 0), ctypes.c_void_p()
        llm_capi.check(lib.llm_decoder_create(ctypes.byref(cfg), ctypes.byref(dec)), lib)
        decs.append(dec)
        ww = _F16W(*[w[k].ctypes.data for k in ("emb", "ln1_g", "ln1_b", "ln2_g", "ln2_b", "wqkv",
                                                 "wo", "w1", "w2", "b1", "b2")])
        llm_capi.check(lib.llm_decoder_set_f16_weights(dec, ctypes.byref(ww)), lib)
        return dec

    try:
        whole, took = prompt(make())
        os.environ["LLM_PREFILL_ROOM"] = "512"
        dec = make()
        short, first = prompt(dec)
        assert 0 < first < took
        # chunks split the sums of the attention otherwise: as whole prompts against steps
        assert rel_err(short, whole) < 1e-3
        del os.environ["LLM_PREFILL_ROOM"]
        again, more = prompt(dec)
        assert more == 0  # there would be room now, but no one asks
        np.testing.assert_array_equal(again, short)
        os.environ["LLM_PREFILL_ROOM"] = "100"  # nor is there room for the short pass
        dec = make()
        with pytest.raises(llm_capi.LlmError) as e:
            prompt(dec)
        assert e.value.status == llm_capi.LLM_ERR_OOM
        os.environ["LLM_PREFILL_ROOM"] = "512"  # later there is
        late, _ = prompt(dec)
        np.testing.assert_array_equal(late, short)
    finally:
        for dec in decs:
            lib.llm_decoder_destroy(dec)

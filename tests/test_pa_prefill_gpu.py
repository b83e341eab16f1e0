"""Parity of the MFMA prefill attention (pa_prefill, via the C ABI): causal
paged attention of a prompt chunk, the reference's is_prefill pass
(attention/attention_cuda.hpp:21) with the maths of cpu_paged_attention_forward
(attention_cpu/cpu_attention_kernel.cpp:37-129) per query.

Oracle: the CPU restatement run as a decode batch of m rows with
beam_ids = row and context_lens = p0 + i + 1 — exactly the rows the decode
kernel computed per prompt token before this kernel existed.  Tolerance as
pa_decode: 1e-3 relative, tensor-normalised and elementwise.  The elementwise
floor is ATOL_FRAC = 4e-6 of the largest |output| (decode: 1e-6): q and p
enter the fp16 MFMAs as hi + lo halves, ~22 significant bits, so a score
carries ~2.4e-7 x sum|q_i k_i| of error and an output element ~1e-6 of the
output scale (measured 2e-7 .. 1.5e-6 of it, scripts/diag_prefill.py); an
element near zero is held to that floor, every other to 1e-3 of itself."""
import numpy as np
import pytest

from _util import assert_parity, rel_err

pytestmark = pytest.mark.gpu
RTOL = 1e-3
ATOL_FRAC = 4e-6


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _case(rng, *, rows, H, D, T, ts, missing=0.0, nan_tail=False):
    nt = (T + ts - 1) // ts
    num_pages = rows * H * nt + 7
    scale = D ** -0.25
    k_pool = (rng.standard_normal((num_pages, ts, D)) * scale).astype(np.float16)
    v_pool = rng.standard_normal((num_pages, ts, D)).astype(np.float16)
    perm = rng.permutation(num_pages)[: rows * H * nt].astype(np.int32)
    pt = np.full((rows, H, nt + 2), -1, np.int32)
    pt[:, :, :nt] = perm.reshape(rows, H, nt)
    if missing:
        m = rng.random(pt[:, :, :nt].shape) < missing
        pt[:, :, :nt][m] = -1
    if nan_tail and T % ts:
        # tokens past the context in the last page were never written: NaN there
        # must not reach the output (masked keys stage V = 0)
        for r in range(rows):
            for h in range(H):
                p = pt[r, h, nt - 1]
                if p >= 0:
                    k_pool[p, T % ts:] = np.nan
                    v_pool[p, T % ts:] = np.nan
    return k_pool, v_pool, pt


def _oracle(oracle, q, kp, vp, pt, row, p0, sm_scale=1.0):
    m = q.shape[0]
    T = p0 + m
    return oracle.paged_attention(
        q, kp.astype(np.float32), vp.astype(np.float32), pt, T=T,
        beam_ids=np.full(m, row, np.int32), context_lens=np.arange(p0 + 1, T + 1, dtype=np.int32),
        temperature=sm_scale ** -0.5)


@pytest.mark.parametrize("H,D,ts,p0,m,row", [
    (4, 64, 16, 0, 1, 0),       # one token, one key
    (4, 64, 16, 0, 37, 1),      # ragged query block, first chunk
    (12, 64, 16, 100, 64, 0),   # C2 heads
    (3, 128, 16, 0, 33, 2),
    (2, 128, 16, 1000, 200, 1), # later chunk: long prefix, ragged tail page
    (2, 128, 32, 517, 96, 0),   # page 32
    (2, 64, 32, 31, 1, 1),
    (16, 128, 16, 7680, 512, 0),  # C3 heads, the last chunk of an 8192-token prompt
])
@pytest.mark.parametrize("split", [True, False])
def test_pa_prefill_vs_oracle(gpu, oracle, H, D, ts, p0, m, row, split):
    """split: key range over several workgroups + the decode merge; else one pass."""
    import llm_capi
    rng = np.random.default_rng(p0 * 7 + m + D)
    kp, vp, pt = _case(rng, rows=3, H=H, D=D, T=p0 + m, ts=ts, nan_tail=True)
    q = (rng.standard_normal((m, H, D)) * D ** -0.25).astype(np.float32)
    out = llm_capi.pa_prefill(_dev(q), _dev(kp), _dev(vp), _dev(pt), row=row, p0=p0,
                              split=split).cpu().numpy()
    ref = _oracle(oracle, q, kp, vp, pt, row, p0)
    assert np.isfinite(out).all()
    assert_parity(out, ref, RTOL, ATOL_FRAC)
    # and the decode kernel on the same rows agrees
    dec = llm_capi.pa_decode(_dev(q), _dev(kp), _dev(vp), _dev(pt), T=p0 + m,
                             beam_ids=_dev(np.full(m, row, np.int32)),
                             context_lens=_dev(np.arange(p0 + 1, p0 + m + 1, dtype=np.int32)))
    assert_parity(out, dec.cpu().numpy(), RTOL, ATOL_FRAC)


@pytest.mark.parametrize("D,ts", [(64, 16), (64, 32), (128, 16), (128, 32)])
@pytest.mark.parametrize("p0,m", [
    (0, 63), (0, 64), (0, 65),      # a full tile, one query less and one more
    (0, 129), (95, 128),            # one query past a tile; a tile that ends inside a stage
    (1, 127), (448, 65), (449, 256),  # stages of 64 keys: first and last full or one key long
])
def test_pa_prefill_tile_edges(gpu, oracle, D, ts, p0, m):
    """Query tiles and key stages of 64, pages missing inside a stage, keys past
    the context never written; cut into pieces and in one pass."""
    import llm_capi
    rng = np.random.default_rng(p0 + 3 * m + D + ts)
    H = 3
    kp, vp, pt = _case(rng, rows=2, H=H, D=D, T=p0 + m, ts=ts, missing=0.1, nan_tail=True)
    q = (rng.standard_normal((m, H, D)) * D ** -0.25).astype(np.float32)
    ref = _oracle(oracle, q, kp, vp, pt, 1, p0)
    for split in (True, False):
        out = llm_capi.pa_prefill(_dev(q), _dev(kp), _dev(vp), _dev(pt), row=1, p0=p0,
                                  split=split).cpu().numpy()
        assert np.isfinite(out).all()
        assert_parity(out, ref, RTOL, ATOL_FRAC)


@pytest.mark.parametrize("H,D", [(2, 64), (7, 64), (12, 64), (16, 128), (31, 128), (33, 128)])
@pytest.mark.parametrize("p0,m", [(0, 300), (900, 70), (2000, 17)])
def test_pa_prefill_merges(gpu, oracle, H, D, p0, m):
    """Rows of one to many splits and of one to four quads a thread, some past the prompt
    merge's widest; rows whose pages are missing altogether."""
    import llm_capi
    rng = np.random.default_rng(H + p0 + m)
    kp, vp, pt = _case(rng, rows=1, H=H, D=D, T=p0 + m, ts=16)
    pt[0, H // 2] = -1
    q = (rng.standard_normal((m, H, D)) * D ** -0.25).astype(np.float32)
    out = llm_capi.pa_prefill(_dev(q), _dev(kp), _dev(vp), _dev(pt), row=0, p0=p0).cpu().numpy()
    assert (out[:, H // 2] == 0).all()
    at = np.r_[0:m:max(1, m // 5), m - 1]  # rows of their own contexts
    for i in at:
        ref = _oracle(oracle, q[i:i + 1], kp, vp, pt, 0, p0 + int(i))
        assert_parity(out[i:i + 1], ref, RTOL, ATOL_FRAC)


@pytest.mark.parametrize("H,p0,m", [(2, 0, 65), (2, 4095, 17), (2, 8190, 70), (12, 1000, 128), (16, 2040, 1), (33, 0, 1000)])
def test_pa_prefill_stages(gpu, oracle, H, p0, m):
    """One pass by stages of 64 keys where workgroups are few (of 32 past 512), splits of many
    short stages: contexts that end inside a stage, more than 16 splits' worth of keys."""
    import llm_capi
    rng = np.random.default_rng(p0 + m)
    kp, vp, pt = _case(rng, rows=1, H=H, D=128, T=p0 + m, ts=16, nan_tail=True)
    q = (rng.standard_normal((m, H, 128)) * 128 ** -0.25).astype(np.float32)
    k, v, t = _dev(kp), _dev(vp), _dev(pt)
    for split in (False, True):
        out = llm_capi.pa_prefill(_dev(q), k, v, t, row=0, p0=p0, split=split).cpu().numpy()
        for i in {0, m // 2, m - 1}:
            assert_parity(out[i:i + 1], _oracle(oracle, q[i:i + 1], kp, vp, pt, 0, p0 + i), RTOL, ATOL_FRAC)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("p0,m", [(0, 33), (0, 64), (31, 33), (50, 1)])
def test_pa_prefill_short_contexts_are_one_split(gpu, D, p0, m):
    """Up to 64 keys: the same bits with a workspace and without, no merge behind it."""
    import llm_capi
    rng = np.random.default_rng(p0 + m)
    kp, vp, pt = _case(rng, rows=1, H=16, D=D, T=p0 + m, ts=16)
    q = _dev((rng.standard_normal((m, 16, D)) * D ** -0.25).astype(np.float32))
    k, v, t = _dev(kp), _dev(vp), _dev(pt)
    whole, split = (llm_capi.pa_prefill(q, k, v, t, row=0, p0=p0, split=s).cpu().numpy() for s in (False, True))
    np.testing.assert_array_equal(split.view(np.uint32), whole.view(np.uint32))


def test_pa_prefill_missing_pages_and_scale(gpu, oracle):
    import llm_capi
    rng = np.random.default_rng(11)
    H, D, ts, p0, m = 3, 128, 16, 300, 70
    kp, vp, pt = _case(rng, rows=2, H=H, D=D, T=p0 + m, ts=ts, missing=0.15)
    # spiky scores: a large sm_scale stresses the running-max rescale
    q = (rng.standard_normal((m, H, D)) * 2.0).astype(np.float32)
    out = llm_capi.pa_prefill(_dev(q), _dev(kp), _dev(vp), _dev(pt), row=1, p0=p0,
                              sm_scale=0.5).cpu().numpy()
    ref = _oracle(oracle, q, kp, vp, pt, 1, p0, sm_scale=0.5)
    assert_parity(out, ref, RTOL, ATOL_FRAC)


def test_pa_prefill_all_missing_is_zero(gpu):
    import llm_capi
    rng = np.random.default_rng(3)
    kp, vp, pt = _case(rng, rows=1, H=2, D=64, T=40, ts=16)
    pt[:] = -1
    q = rng.standard_normal((40, 2, 64)).astype(np.float32)
    out = llm_capi.pa_prefill(_dev(q), _dev(kp), _dev(vp), _dev(pt), row=0, p0=0).cpu().numpy()
    np.testing.assert_array_equal(out, np.zeros_like(out))


def test_pa_prefill_strided_q_interleaved_pools(gpu, oracle):
    """q read in place from a wider row (the decoder's qkv rows) and K/V pages
    interleaved in one allocation (kv_cache's own layout)."""
    import torch
    import llm_capi
    rng = np.random.default_rng(5)
    H, D, ts, p0, m = 4, 128, 16, 64, 48
    kp, vp, pt = _case(rng, rows=1, H=H, D=D, T=p0 + m, ts=ts)
    kv = torch.empty((kp.shape[0], 2, ts, D), dtype=torch.float16, device="cuda")
    kv[:, 0] = _dev(kp)
    kv[:, 1] = _dev(vp)
    q = (rng.standard_normal((m, H, D)) * D ** -0.25).astype(np.float32)
    wide = torch.zeros((m, 3 * H * D), dtype=torch.float32, device="cuda")
    wide[:, :H * D] = _dev(q.reshape(m, H * D))
    out = llm_capi.pa_prefill(wide, kv[:, 0], kv[:, 1], _dev(pt), row=0, p0=p0).cpu().numpy()
    ref = _oracle(oracle, q, kp, vp, pt, 0, p0)
    assert_parity(out, ref, RTOL, ATOL_FRAC)


def test_pa_prefill_rejects_unsupported(gpu):
    import llm_capi
    rng = np.random.default_rng(1)
    kp, vp, pt = _case(rng, rows=1, H=2, D=32, T=20, ts=16)
    q = rng.standard_normal((20, 2, 32)).astype(np.float32)
    with pytest.raises(llm_capi.LlmError) as ei:
        llm_capi.pa_prefill(_dev(q), _dev(kp), _dev(vp), _dev(pt), row=0, p0=0)
    assert ei.value.status == llm_capi.LLM_ERR_UNSUPPORTED
    with pytest.raises(llm_capi.LlmError):  # positions past max_tiles
        kp, vp, pt = _case(rng, rows=1, H=2, D=64, T=20, ts=16)
        q = rng.standard_normal((100, 2, 64)).astype(np.float32)
        llm_capi.pa_prefill(_dev(q), _dev(kp), _dev(vp), _dev(pt), row=0, p0=0)


@pytest.mark.parametrize("H,D,m", [(4, 64, 113), (16, 64, 300), (16, 128, 300), (4, 64, 1024)])
def test_pa_prefill_as_exact_as_decode(gpu, H, D, m):
    """Small scores, so that the weights' own rounding decides: against 64 bits off no more
    than half as much again as the decode kernel over the same rows (whose weights stay
    fp32; with the scale of the weights' halves in their exponent it was twice as much)."""
    import torch
    import llm_capi
    g = torch.Generator(device="cuda").manual_seed(m)
    nt = -(-m // 16)
    kp, vp = (torch.randn((H * nt, 16, D), generator=g, device="cuda").half() for _ in "kv")
    pt = torch.randperm(H * nt, generator=g, device="cuda").int().view(1, H, nt).contiguous()
    q = torch.randn((m, H, D), generator=g, device="cuda") * 0.3 * D ** -0.5
    k, v = (x[pt[0].long()].reshape(H, -1, D)[:, :m].double() for x in (kp, vp))
    s = (q.double().transpose(0, 1) @ k.transpose(1, 2).contiguous()).masked_fill(
        torch.ones((m, m), dtype=torch.bool, device="cuda").triu(1), -float("inf"))
    e = torch.exp(s - s.amax(-1, keepdim=True))
    ref = ((e / (e.sum(-1, keepdim=True) + 1e-6)) @ v).transpose(0, 1)
    rows = torch.arange(m, dtype=torch.int32, device="cuda")
    outs = (llm_capi.pa_prefill(q, kp, vp, pt, row=0, p0=0),
            llm_capi.pa_decode(q, kp, vp, pt, T=m, beam_ids=torch.zeros_like(rows), context_lens=rows + 1))
    off = [((x.double() - ref).norm() / ref.norm()).item() for x in outs]
    assert off[0] <= 1.5 * off[1], off

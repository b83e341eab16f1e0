"""The block form of the layer-stack models' products (mm_impl.hpp) where it can go
wrong: one k-step and odd numbers of them, rows and columns that end inside a block,
heads that whole 16-byte stores fit and do not fit, blocks of one, a few and many
sequences at places of a page that are no multiple of four, short expert tiles."""
import numpy as np
import pytest

import _layer_stack as T
import _nubosun as N
from test_layer_stack_gpu import serve, tokens  # noqa: F401

pytestmark = pytest.mark.gpu

# width, attention, experts, portions of the sequences in each step
GEFARAX = {
    "one_k_step": (32, T.attn(heads=96, kv_heads=8, dim=24, vdim=16, rot=16), None,
                   [[17] * 7, [1] * 7, [31] * 7]),
    "odd_k_steps": (96, T.attn(heads=48, kv_heads=6, dim=40, vdim=24, rot=16),
                    T.moe(experts=4, top=2, ff=136, shared=200), [[70, 131, 50], [3, 2, 5], [61, 66, 129]]),
    "pairs": (128, T.attn(heads=64, kv_heads=4, dim=20, vdim=10, rot=12),
              T.moe(experts=8, top=3, ff=36, shared=40), [[33], [65], [130]]),
    "many_rows": (160, T.attn(heads=20, kv_heads=2, dim=72, vdim=64, rot=40),
                  T.moe(experts=3, top=2, ff=264, shared=300), [[127, 129, 1, 2, 60], [300]]),
    "wide": (1056, T.attn(heads=32, kv_heads=4, dim=64, vdim=64, rot=32),
             T.moe(experts=2, top=1, ff=520, shared=1032), [[391], [44, 28]]),
}


def check(serve, cfg, w, dtype, portions):  # noqa: F811
    n = max(len(p) for p in portions)
    lens = [sum(p[i] for p in portions if i < len(p)) for i in range(n)]
    requests = {i: tokens(cfg, lens[i], 7 + i) for i in range(n)}
    eng = serve(cfg, w, dtype, max_tokens=64 * n + sum(lens), max_seqs=n)
    got = T.replay(eng, requests, [list(enumerate(p)) for p in portions])
    for i in range(n):
        T.check_rows(got[i], T.logits(cfg, w, requests[i]), dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", GEFARAX)
def test_grouped_query_blocks(serve, name, dtype):  # noqa: F811
    width, a, m, portions = GEFARAX[name]
    cfg = T.config([(a, m)], width=width)
    w = T.weights(cfg, 3)
    check(serve, cfg, T.clear_choices(w) if dtype == "bfloat16" else w, dtype, portions)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("mixer", [N.latent(heads=48, dim=32, rot=16, vdim=24, rank=96),
                                   N.latent(heads=36, dim=20, rot=12, vdim=14, rank=72)],
                         ids=["whole", "pairs"])
def test_latent_blocks(serve, mixer, dtype):  # noqa: F811
    """Also the expansion of cached rows (portions of 65 tokens and more)."""
    cfg = N.config([(mixer, N.dense(ff=1100))], width=136)
    check(serve, cfg, N.weights(cfg, 5), dtype, [[70, 131, 90], [66, 1, 129]])


@pytest.mark.parametrize("ff,rows", [(4640, 385), (4668, 385)])
def test_two_blocks_a_cu(serve, ff, rows):  # noqa: F811
    """gate and up in 257 to 512 blocks of 64 x 128 (three stages), rows of 16 bytes and not."""
    cfg = N.config([(N.latent(heads=4, dim=32, rot=16, vdim=32, rank=64), N.dense(ff=ff))], width=96)
    check(serve, cfg, N.weights(cfg, 11), "bfloat16", [[rows]])


@pytest.mark.parametrize("ff,width", [(13000, 64), (13000, 96), (13000, 224), (9000, 160), (9000, 288),
                                      (9000, 320), (9000, 384), (9000, 448), (13000, 352), (9000, 1088),
                                      (9000, 1152)])
def test_strips(serve, ff, width):  # noqa: F811
    """gate and up by strips, 385 to 512 blocks of 128 x 256 or 513 to 768 of 128 x 128: one to seven stages
    and 17 and 18, a last k-step alone, rows and columns that end inside a block."""
    cfg = N.config([(N.latent(heads=4, dim=32, rot=16, vdim=32, rank=64), N.dense(ff=ff))], width=width)
    check(serve, cfg, N.weights(cfg, 13), "bfloat16", [[500]])


@pytest.mark.parametrize("ff,shared,width", [(7000, 1100, 160), (1056, 2080, 1056)])
def test_expert_strips(serve, ff, shared, width):  # noqa: F811
    """Tiles of 128 rows that end early; the routed and the shared experts' K at their own lengths."""
    cfg = T.config([(T.attn(heads=8, kv_heads=2, dim=32, vdim=32, rot=16), T.moe(experts=2, top=1, ff=ff, shared=shared))],
                   width=width)
    check(serve, cfg, T.clear_choices(T.weights(cfg, 17)), "bfloat16", [[500]])

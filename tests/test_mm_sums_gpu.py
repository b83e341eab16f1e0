"""The layer-stack models' products (mm_impl.hpp): the activation at gates of any size."""
import numpy as np
import pytest

import _layer_stack as T
import _nubosun as N
from test_layer_stack_gpu import run_whole, serve, tokens  # noqa: F401

pytestmark = pytest.mark.gpu


def far_gates(w, names):
    """Gates of one sign a column whatever the token, from 0.06 to 6e37: the first channel of
    every row is large, and only it reaches them."""
    w["embed"][:, 0] = 8.0
    for i, n in enumerate(names):
        k = np.resize(np.arange(-2, 38), len(w[n])) + 0.0
        w[n][:] = 0
        w[n][:, 0] = T.to_bf16((-1.0) ** (np.arange(len(k)) // 3 + i) * 10.0 ** k)
    return w


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows", [1, 16, 40, 300])
@pytest.mark.parametrize("kind", ["dense", "experts"])
def test_gates_far_from_zero(serve, kind, rows, dtype):  # noqa: F811
    """g / (1 + e^(-1.702 g)) is nothing where g is far below zero, however far."""
    if kind == "dense":
        cfg = N.config([(N.latent(), N.dense(ff=80))])
        w = far_gates(N.weights(cfg, 3), ["l0.mlp.gate"])
    else:
        cfg = T.config([(T.attn(), T.moe(experts=4, ff=80, shared=120))])
        w = far_gates(T.clear_choices(T.weights(cfg, 3)),
                      [f"l0.mlp.{e}.gate" for e in ("e0", "e1", "e2", "e3", "shared")])
    t = tokens(cfg, rows, rows)
    with np.errstate(over="ignore"):
        want = T.logits(cfg, w, t)
    T.check_rows(run_whole(serve(cfg, w, dtype), t), want, dtype)

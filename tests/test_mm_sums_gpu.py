"""Products of few rows in bf16 (mm_impl.hpp): the activation at gates of any size, and sums
over K that do not depend on what else the launch works on."""
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


@pytest.mark.parametrize("width,experts,rows", [(96, 2, 1), (96, 2, 5), (1088, 8, 1), (1088, 8, 16)])
def test_sums_of_experts_whatever_the_others_width(serve, width, experts, rows):  # noqa: F811
    """A shared expert of 64 k-steps beside routed ones of 16, 32 and 64, whose output is
    nothing: the same bits, by eight, four and two waves a workgroup (these past 640)."""
    first = base = None
    for ff in (2048, 1024, 512):
        cfg = T.config([(T.attn(), T.moe(experts=experts, ff=ff, shared=2048))], width=width)
        w = T.weights(cfg, 5)
        base = base or w
        w = {k: w[k] if ".mlp.e" in k else base[k] for k in w}
        for e in range(experts):
            w[f"l0.mlp.e{e}.down"] = 0 * w[f"l0.mlp.e{e}.down"]
        eng = serve(cfg, w, "bfloat16", name=f"m{ff}")
        s = eng.open_seq()
        tap = eng.step_taps([(s, tokens(cfg, rows, 6), [0])])[1]
        first = tap if first is None else first
        np.testing.assert_array_equal(tap.view(np.uint32), first.view(np.uint32))


@pytest.mark.parametrize("width", [72, 512])
def test_sums_of_the_head_whatever_its_width(serve, width):  # noqa: F811
    """Logits of the first tokens of heads of 999 column tiles and of more, one row to 16: the
    same bits."""
    cfg = T.config([(T.attn(), None)], width=width, vocab=32768)
    w = T.weights(cfg, 7)
    t = tokens({"vocab": 15984}, 16, 8)
    first = None
    for vocab in (15984, 16001, 32752, 32768):
        v = dict(w, embed=w["embed"][:vocab], head=w["head"][:vocab])
        eng = serve(dict(cfg, vocab=vocab), v, "bfloat16", name=f"m{vocab}")
        for rows in (range(16), [15], range(8), range(9)):
            s = eng.open_seq()
            out = eng.step([(s, t, list(rows))])[:, :15984]
            eng.close_seq(s)
            first = out if first is None else first
            np.testing.assert_array_equal(out.view(np.uint32), first[list(rows)].view(np.uint32))

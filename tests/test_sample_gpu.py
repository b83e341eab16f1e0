"""sample_rows where its segments, histograms and cells can go wrong: vocabularies at
their borders, ties, masked and unusable logits, thresholds that keep one or all."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def draw(logits, T, k, p, counter=0):
    import torch
    import llm_capi
    return llm_capi.sample_rows(torch.from_numpy(logits).cuda(), T, k, p, seed=5,
                                counter=counter).cpu().numpy()


@pytest.mark.parametrize("V", [1, 2, 63, 257, 4095, 4097, 8193, 16385, 32768, 53248, 53249, 65536])
@pytest.mark.parametrize("T,k,p", [(0.8, 40, 0.9), (1.0, 0, 0.999), (1.3, 2, 1.0), (1.0, 0, 1.0),
                                   (0.05, 300, 0.3), (0.0, 0, 1.0)])
def test_vocabulary_borders(gpu, V, T, k, p):
    from oracle.oracle import sample_rows
    logits = (np.random.default_rng(V + k).standard_normal((5, V)) * 2).astype(np.float32)
    for counter in (0, 9):
        ref, margin = sample_rows(logits, T, k, p, seed=5, counter=counter)
        got = draw(logits, T, k, p, counter)
        # a draw this close to a boundary of the distribution may fall on either side
        assert ((got == ref) | (margin < 1e-4)).all(), (got, ref, margin)


@pytest.mark.parametrize("segments", range(1, 17))
def test_every_number_of_segments(gpu, segments):
    """Rows of whole segments and of one token more than the form before takes."""
    from oracle.oracle import sample_rows
    for V in {4096 * segments, 4096 * (segments - 1) + 1}:
        logits = (np.random.default_rng(V).standard_normal((3, V)) * 2).astype(np.float32)
        logits[:, -1] = logits.max(1) + 3.0  # the last token is drawn now and then
        for counter in range(4):
            ref, margin = sample_rows(logits, 0.9, 60, 0.95, seed=5, counter=counter)
            got = draw(logits, 0.9, 60, 0.95, counter)
            assert ((got == ref) | (margin < 1e-4)).all(), (V, got, ref, margin)


def test_ties_stay_together(gpu):
    """Equal probabilities share a rank: all of them stay, nothing below does."""
    V = 20000
    logits = np.full((1, V), -3.0, np.float32)
    top = np.arange(17, V, 1999)
    logits[0, top] = 2.0
    seen = {int(draw(logits, 1.0, 3, 1.0, c)[0]) for c in range(200)}
    assert seen <= set(top.tolist()) and len(seen) == len(top)
    same = np.zeros((1, 300), np.float32)  # top_p of equal ones: the mass above each is 0
    assert len({int(draw(same, 1.0, 0, 0.1, c)[0]) for c in range(300)}) > 100


def test_masked_and_unusable_logits(gpu):
    V = 9000
    rng = np.random.default_rng(1)
    logits = rng.standard_normal((4, V)).astype(np.float32)
    logits[0, :] = -np.inf
    logits[0, [5, 8190, 8999]] = [0.0, 1.0, 0.5]  # all others masked
    logits[1, 77] = np.nan
    logits[2, :] = -np.inf
    logits[3, 4000] = 80.0  # the rest underflows to nothing
    for c in range(20):
        got = draw(logits, 1.0, 50, 0.95, c)
        assert got[0] in (5, 8190, 8999) and got[1] == 0 and got[2] == 0 and got[3] == 4000
    assert draw(logits, 1.0, 0, 0.3, 1)[0] == 8190


@pytest.mark.parametrize("p", [9e-16, 8e-16, 1e-16, 1e-20, 1.2e-38, 1e-42])
@pytest.mark.parametrize("k", [0, 50])
def test_top_p_below_any_probability(gpu, p, k):
    """A top_p that every mass exceeds leaves the most probable token, or its ties."""
    rng = np.random.default_rng(11)
    logits = rng.standard_normal((6, 9000)).astype(np.float32)
    logits[5, [3, 4100, 8999]] = logits[5].max() + 1.0
    logits[4] = 0.25
    for c in range(12):
        got = draw(logits, 1.0, k, p, c)
        assert (got[:4] == logits[:4].argmax(1)).all() and got[5] in (3, 4100, 8999)
    assert len({int(draw(logits[4:5], 1.0, k, p, c)[0]) for c in range(40)}) > 20  # all tied


@pytest.mark.parametrize("k", [2, 5, 63, 64, 65])
@pytest.mark.parametrize("p", [0.5, 0.97, 1.0])
@pytest.mark.parametrize("shape", ["spread", "one_group", "few_groups", "many_ties", "many_near", "flat",
                                   "some_near", "tiny"])
def test_few_tokens_left(gpu, shape, k, p):
    """A small top_k: its tokens spread out, in one group of eight threads, in fewer groups
    than top_k; 70 to 256 equal or near ones, and more than are ranked one against the other;
    all but one below the least normal number."""
    from oracle.oracle import sample_rows
    V = 12500
    rng = np.random.default_rng(k)
    logits = rng.standard_normal((3, V)).astype(np.float32)
    at = np.arange(V)
    group = (at // 256 % 16) * 8 + at % 64 // 8
    if shape == "one_group":
        logits[:, group == 19] += 6.0
    elif shape == "few_groups":
        logits[:, group >= 40] = -np.inf
    elif shape == "many_ties":
        logits[:, rng.permutation(V)[:900]] = 3.5
    elif shape == "many_near":
        logits[:, rng.permutation(V)[:2000]] = 3.0 + 1e-3 * rng.standard_normal((3, 2000)).astype(np.float32)
    elif shape == "some_near":
        logits[:, rng.permutation(V)[:190]] = 5.0 + 1e-3 * rng.standard_normal((3, 190)).astype(np.float32)
    elif shape == "tiny":
        logits[:, 777] = 66.0
    elif shape == "flat":
        logits[:] = 0.0
    for counter in range(6):
        ref, margin = sample_rows(logits, 0.7, k, p, seed=5, counter=counter)
        got = draw(logits, 0.7, k, p, counter)
        assert ((got == ref) | (margin < 1e-4)).all(), (got, ref, margin)


@pytest.mark.parametrize("V", [255, 1057, 1600, 2047, 2048, 2816, 4096])
@pytest.mark.parametrize("k", [2, 6, 24, 50, 64])
def test_short_rows(gpu, V, k):
    """Rows of about as many groups of eight threads as top_k, and of fewer."""
    from oracle.oracle import sample_rows
    logits = (2 * np.random.default_rng(V + k).standard_normal((5, V))).astype(np.float32)
    for p in (0.6, 1.0):
        ref, margin = sample_rows(logits, 0.8, k, p, seed=5, counter=k)
        got = draw(logits, 0.8, k, p, k)
        assert ((got == ref) | (margin < 1e-4)).all(), (got, ref, margin)


def test_exp_below_is_expf(gpu):
    """The sampler's exponential (tuning build) has expf's bits for every number that is not
    positive, minus infinity and NaN among them."""
    import ctypes
    import torch
    import llm_capi
    lib = llm_capi.load_tune()
    lib.exp_below_differs.argtypes = [ctypes.c_uint32, ctypes.c_uint, ctypes.c_void_p, ctypes.c_void_p]
    differ = torch.zeros(2, dtype=torch.int32, device="cuda")
    # 2^31 patterns with a sign; 0 and what comes with it in a workgroup, so small that it is 1; NaN
    for first, blocks in ((0x80000000, 1 << 23), (0, 1), (0x7F800001, (0x7FFFFFFF - 0x7F800001) // 256)):
        llm_capi.check(lib.exp_below_differs(first, blocks, differ.data_ptr(), None), lib)
        torch.cuda.synchronize()
        assert differ.tolist() == [0, 0], (hex(first), [hex(x & 0xFFFFFFFF) for x in differ.tolist()])

"""The block form of i8_gemm / f16_gemm (rows of a prompt) at the edges of its tiles:
exact int32 accumulators, fp16 sums within their rounding, rows with a stride, one
k-step and odd numbers of them, and the same rows at an address that only the stream
form takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# enough columns for more than 128 blocks of 64 x 64
SHAPES = [(65, 4352, 64), (127, 4160, 192), (129, 2832, 2048), (191, 2768, 320), (513, 1040, 64),
          (640, 2304, 768), (1025, 528, 448), (2048, 272, 1088), (2047, 2048, 128)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("shift", [0, 4])
def test_int8(gpu, M, N, K, shift):
    import torch
    import llm_capi
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(-127, 128, (M, K + 32), dtype=np.int8)
    W = rng.integers(-127, 128, (K, N), dtype=np.int8)
    sa = rng.uniform(0.5, 2.0, M).astype(np.float32)
    sw = rng.uniform(0.5, 2.0, N).astype(np.float32)
    bias = (100 * rng.standard_normal(N)).astype(np.float32)
    buf = torch.zeros(M * (K + 32) + 64, dtype=torch.int8, device="cuda")
    a = buf[shift:shift + M * (K + 32)].view(M, K + 32)
    a.copy_(torch.from_numpy(A))
    dev = [torch.from_numpy(x).cuda() for x in (sa, sw, bias)]
    packed = llm_capi.pack_weights(torch.from_numpy(W).cuda(), llm_capi.LLM_I8)
    acc, C = llm_capi.i8_gemm(a[:, :K], packed, N, sa=dev[0], sw=dev[1], bias=dev[2], act=1)
    ref = (torch.from_numpy(A[:, :K]).double() @ torch.from_numpy(W).double()).numpy()
    assert np.array_equal(acc.cpu().numpy(), ref.astype(np.int32))
    y = ref.astype(np.float32) * (sa[:, None] * sw) + bias
    assert np.array_equal(C.cpu().numpy(), np.maximum(y, 0))


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp16(gpu, M, N, K):
    import torch
    import llm_capi
    g = torch.Generator().manual_seed(M + K)
    A = torch.randn((M, K + 8), generator=g).half()
    W = torch.randn((K, N), generator=g).half()
    bias = torch.randn(N, generator=g)
    packed = llm_capi.pack_weights(W.cuda(), llm_capi.LLM_F16)
    C = llm_capi.f16_gemm(A.cuda()[:, :K], packed, N, bias=bias.cuda()).cpu().double()
    ref = A[:, :K].double() @ W.double() + bias.double()
    # fp32 sums of K exact products in some order: K roundings of the largest partial sum
    size = A[:, :K].double().abs() @ W.double().abs() + bias.double().abs()
    assert ((C - ref).abs() <= 2.0 ** -23 * (K ** 0.5 + 2) * size).all()


@pytest.mark.parametrize("M,N,K", [(257, 10944, 64), (257, 11024, 192), (257, 11248, 320)])
def test_two_blocks_a_cu(gpu, M, N, K):
    """257 to 512 blocks of 64 x 128: the form of three stages, with one k-step, odd and even
    numbers of stages."""
    test_int8(gpu, M, N, K, 0)
    test_fp16(gpu, M, N, K)


@pytest.mark.parametrize("M,N,K", [(700, 1024, 256), (512, 2304, 768), (320, 6144, 2048), (1024, 2048, 8192)])
def test_fp16_sums_as_exact_as_the_streams(gpu, M, N, K):
    """A block's sum over K goes in eight parts, as a stream's over its waves: off no more
    than a tenth beyond the stream of the same rows (one sum over all of K: 1.4 to 2.7
    times)."""
    import torch
    import llm_capi
    g = torch.Generator(device="cuda").manual_seed(K)
    A = torch.randn((M, K), generator=g, device="cuda").half()
    W = torch.randn((K, N), generator=g, device="cuda").half()
    packed = llm_capi.pack_weights(W, llm_capi.LLM_F16)
    ref = A.double() @ W.double()
    blocks = llm_capi.f16_gemm(A, packed, N).double()
    streams = torch.cat([llm_capi.f16_gemm(A[i:i + 64], packed, N).double() for i in range(0, M, 64)])
    off = [((x - ref).norm() / ref.norm()).item() for x in (blocks, streams)]
    assert off[0] <= 1.1 * off[1], off


@pytest.mark.parametrize("M,N,K", [(65, 4352, 64), (191, 2768, 320), (1025, 1040, 448)])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_activations_with_and_without_sums(gpu, M, N, K, act):
    """The activations of a block's epilogue, with whole sums at 16 bytes, beside them and not asked for:
    the same C, and scale, bias and activation of the exact sums (GELU within its erf's rounding)."""
    import torch
    import llm_capi
    rng = np.random.default_rng(M + N + act)
    A = torch.from_numpy(rng.integers(-127, 128, (M, K), dtype=np.int8))
    W = torch.from_numpy(rng.integers(-127, 128, (K, N), dtype=np.int8))
    sa, sw, bias = (torch.from_numpy(x.astype(np.float32)) for x in
                    (rng.uniform(0.5, 2.0, M) / 127, rng.uniform(0.5, 2.0, N) / 127, rng.standard_normal(N)))
    a, s, w, b = A.cuda(), sa.cuda(), sw.cuda(), bias.cuda()
    packed = llm_capi.pack_weights(W.cuda(), llm_capi.LLM_I8)
    lib, p = llm_capi.load(), llm_capi.ptr
    whole = A.double() @ W.double()
    y = whole.float() * (sa[:, None] * sw) + bias
    ref = y if act == 0 else y.relu() if act == 1 else 0.5 * y.double() * (1 + torch.erf(y.double() * 0.5 ** 0.5))
    out = []
    for shift in (0, 1, None):
        C = torch.empty((M, N), device="cuda")
        sums = torch.zeros(M * N + 4, dtype=torch.int32, device="cuda")
        at = None if shift is None else sums[shift:].data_ptr()
        llm_capi.check(lib.i8_gemm(p(a), K, p(packed), at, p(C), M, N, K, p(s), p(w), p(b), act,
                                   llm_capi.stream_ptr(None)))
        out.append(C.cpu())
        if shift is not None:
            assert torch.equal(sums[shift:shift + M * N].view(M, N).cpu().double(), whole)
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    if act < 2:
        assert torch.equal(out[0], ref)
    else:  # y / sqrt 2, erff and two products: a few roundings of y, and of 1 + erf where it cancels
        assert ((out[0].double() - ref).abs() <= 2.0 ** -21 * y.double().abs()).all()
    h = torch.randn((M, K), generator=torch.Generator().manual_seed(K)).half()
    w16 = (W.float() / 127).half()
    C = llm_capi.f16_gemm(h.cuda(), llm_capi.pack_weights(w16.cuda(), llm_capi.LLM_F16), N, bias=b, act=act).cpu().double()
    x = h.double() @ w16.double() + bias.double()
    ref = x if act == 0 else x.relu() if act == 1 else 0.5 * x * (1 + torch.erf(x * 0.5 ** 0.5))
    size = h.double().abs() @ w16.double().abs() + bias.double().abs()
    # as test_fp16; GELU's slope is at most 1.13
    assert ((C - ref).abs() <= 1.13 * 2.0 ** -23 * (K ** 0.5 + 2) * size + 2.0 ** -21 * x.abs()).all()

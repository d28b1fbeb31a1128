"""One row's add-norm made inside the gate_up product that reads it: the bits of the separate kernels, over both kinds of weights."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# rows of one wave, of four with a part of their last pieces, of two and four pieces a lane; 1, 2 and 4 tiles of channels a workgroup, as many as are taken
@pytest.mark.parametrize("k", [64, 448, 1024, 2048, 2112, 4096, 4160, 8192])
@pytest.mark.parametrize("n", [16, 48, 6160, 16384, 32768])
@pytest.mark.parametrize("quantized", [False, True])
def test_bits_of_the_separate_kernels(k, n, quantized):
    from tinyllmforge_amd import ops as P
    g = torch.Generator(device="cuda").manual_seed(n + k)
    x, residual = (torch.randn(1, k, generator=g, device="cuda").to(BF) * 3 for _ in range(2))
    norm = torch.rand(k, generator=g, device="cuda").to(BF) + 0.5
    if quantized:
        n = -(-n // 32) * 32
        w, scale = torch.randint(-127, 128, (n, k), dtype=torch.int8, device="cuda", generator=g), torch.rand(n, device="cuda", generator=g) * k ** -0.5 / 73
    else:
        w, scale = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(BF), None
    streamed = quantized and n * k >= 120_000_000           # by another kernel
    assert P.add_rms_norm_linear_silu_mul_supported(1, n, k, quantized) == (not streamed)
    if streamed:
        return
    normed, want_residual = P.add_rms_norm(x, residual, norm, 1e-6)
    want = P.w8a16_linear_silu_mul(normed, P.pack_w8(w), scale) if quantized else P.bf16_linear_silu_mul(normed, w)
    packed = P.pack_w8(w) if quantized else w
    got, got_residual = P.add_rms_norm_linear_silu_mul(x, residual, norm, 1e-6, packed, scale)
    assert torch.equal(got, want) and torch.equal(got_residual, want_residual)
    # stays so over replays of a graph, with eager work between them
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        again, again_residual = P.add_rms_norm_linear_silu_mul(x, residual, norm, 1e-6, packed, scale)
    for _ in range(3):
        again.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(again, want) and torch.equal(again_residual, want_residual)


def test_sizes_that_are_not_taken():
    from tinyllmforge_amd import _lib
    lib = _lib.load()
    supported = lib.tlf_add_rmsnorm_gemm_silu_mul_supported
    assert supported(1, 6144, 4096, 0) and not supported(2, 6144, 4096, 0) and not supported(1, 6144, 8256, 0) and not supported(1, 6152, 4096, 0) and not supported(1, 24576, 4096, 0) and not supported(1, 6144, 4000, 0)
    t = torch.zeros(1 << 16, dtype=BF, device="cuda")
    assert lib.tlf_add_rmsnorm_gemm_silu_mul(t.data_ptr(), t.data_ptr(), t.data_ptr(), t.data_ptr(), None, t.data_ptr(), t.data_ptr(), 2, 64, 64, 1e-6,
                                             torch.cuda.current_stream().cuda_stream) != 0

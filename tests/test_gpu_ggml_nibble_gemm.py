"""GPU parity of the matrix-core GEMM for the 32-value nibble types (Q4_0, Q5_0, IQ4_NL): rows
beyond the GEMV's against the oracle's exact dequant times x, at row- and column-tile edges, with
one and two column groups per wave and with K split; and the calls that stay on the GEMV."""
import numpy as np
import pytest

from webpytorch_amd import synth

pytestmark = pytest.mark.gpu

TYPES = ["Q4_0", "Q5_0", "IQ4_NL"]
# (M, K, N): smallest row count; tile tails; many K slices; two column groups (wide grid)
CASES = [(9, 256, 64), (64, 768, 70), (65, 1280, 1000), (77, 4096, 512), (520, 256, 7200)]


def _gemm(core, xt, lin, out_dtype):
    """The GEMM itself, at sizes below those the dispatch gives it too."""
    import torch
    M, K, N = xt.shape[0], lin.Kt, lin.Nt
    ws = core.workspace(core.ggml_gemm_workspace_bytes(M, K, N, core.dtype_code(xt), lin.type_name))
    out = torch.empty((M, N), dtype=out_dtype, device="cuda")
    core._lib.call("miq_ggml_nibble_gemm", core.ptr(xt), core.dtype_code(xt), core.ptr(lin.packed),
                   core._NATIVE_TYPES[lin.type_name][2], core.ptr(lin.bias), core.ptr(out), core.dtype_code(out), M, K, N,
                   core.ptr(ws), ws.numel(), core.stream_handle())
    return out.cpu().numpy()


@pytest.mark.parametrize("type_name", TYPES)
@pytest.mark.parametrize("M,K,N", CASES)
@pytest.mark.parametrize("xdt", [np.float16, np.float32])
def test_nibble_gemm(gpu, type_name, M, K, N, xdt):
    """fp32 accumulation of exact products: within 1e-5 of the largest output (the tolerance of
    the other types' GEMM); uniform random code bytes cover every code."""
    import torch
    from oracle import ggml
    from webpytorch_amd import core
    W = synth.ggml_layer(type_name, M + K + N, K, N)
    b = np.linspace(-1, 1, N).astype(np.float32)
    lin = core.GGMLLinear(W, type_name, K, N, bias=b)
    x = synth.activations(M + 1, M, K, xdt)
    xt = torch.from_numpy(x).cuda()
    assert core._nibble_gemm_taken(type_name, M, K, N, core.dtype_code(xt), lin.packed) == (M * K * N >= 1 << 28)
    ref = ggml.ggml_matmul(x.astype(np.float32), W, type_name, K, N) + b
    got = _gemm(core, xt, lin, torch.float32)
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
    got16 = _gemm(core, xt, lin, torch.float16).astype(np.float32)
    # the same sum rounded once more: half an fp16 step (2^-11 of the value, 2^-25 below its normal range)
    assert np.all(np.abs(got16 - got) <= np.abs(got) * 2.0 ** -11 + 2.0 ** -25)
    assert np.array_equal(_gemm(core, xt, lin, torch.float32), got)  # deterministic
    through = lin(xt).cpu().numpy()
    assert np.abs(through - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("type_name", TYPES)
def test_nibble_routes(gpu, type_name):
    """Rows whose K is no whole number of 256-value steps, weights off a 16-byte address and a
    workspace that would have to grow under graph capture keep the GEMV, with the same result."""
    import torch
    from oracle import ggml
    from webpytorch_amd import core
    M, N = 600, 1000
    for K in (32, 480, 512):
        W = synth.ggml_layer(type_name, K, K, N)
        x = synth.activations(K, M, K, np.float32)
        xt = torch.from_numpy(x).cuda()
        buf = torch.zeros(W.size + 16, dtype=torch.uint8, device="cuda")
        for off in (0, 2):
            packed = buf[off:off + W.size]
            packed.copy_(torch.from_numpy(W.reshape(-1)))
            assert core._nibble_gemm_taken(type_name, M, K, N, 0, packed) == (K == 512 and off == 0)
            if off:
                continue  # the GEMV asks for 16-byte aligned weights and says so
            got = core.ggml_matmul(xt, packed, type_name, K, N).cpu().numpy()
            ref = ggml.ggml_matmul(x, W, type_name, K, N)
            assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
    core.ggml_matmul(xt, buf[:W.size].clone(), type_name, K, N)  # checked before the capture
    packed, eager = buf[:W.size].clone(), None
    packed.copy_(torch.from_numpy(W.reshape(-1)))
    eager = core.ggml_matmul(xt, packed, type_name, K, N)
    out = torch.zeros_like(eager)
    st = torch.cuda.Stream()  # a stream without a workspace
    st.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        assert not core._nibble_gemm_taken(type_name, M, K, N, 0, packed)
        core.ggml_matmul(xt, packed, type_name, K, N, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert float((out - eager).abs().max()) <= 1e-5 * float(eager.abs().max())

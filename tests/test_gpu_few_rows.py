"""2 to 8 fp16 rows through the few-row matrix-core kernel: against the oracle at the edges of the
dispatch rule, and the calls beside it that keep the GEMV."""
import numpy as np
import pytest

from webpytorch_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,taken", [
    (2, 4096, 4096, True), (8, 4864, 896, True), (3, 4096, 8136, True), (8, 1024, 4104, True),
    (2, 16384, 1024, True), (7, 896, 4864, False), (2, 4224, 8136, False), (8, 16512, 512, False)])
def test_few_rows(gpu, M, K, N, taken):
    """fp32 sums of exact products: within 1e-5 of the largest output, as the other product paths."""
    import torch
    from oracle import gptq
    from webpytorch_amd import core
    L = synth.gptq_layer(M + K, K, N, 128, 4)
    b = np.linspace(-1, 1, N).astype(np.float32)
    ql = core.QuantizedLinear.from_autogptq(L["qweight"], L["qzeros"], L["scales"], b, 128, 4)
    x = synth.activations(K, M, K, np.float16)
    xt = torch.from_numpy(x).cuda()
    args = (ql.qweight, ql.scales, K, N, 128, 4, 1.0)
    assert core._few_rows_gemm_taken(xt, *args, None, None) == taken
    assert not core._few_rows_gemm_taken(xt.float(), *args, None, None)
    assert not core._few_rows_gemm_taken(xt, *args, None, torch.empty(0, dtype=torch.uint8, device="cuda")) \
        or core.gemm_workspace_bytes(M, K, N, 128, 4) == 0
    ref = x.astype(np.float32) @ gptq.dequant_closed_form(L["qweight"], L["qzeros"], L["scales"], 128, 4, 1.0) + b
    got = ql.forward(xt, out_dtype=torch.float32).cpu().numpy()
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
    assert np.array_equal(ql.forward(xt, out_dtype=torch.float32).cpu().numpy(), got)  # deterministic
    got16 = ql.forward(xt, out_dtype=torch.float16).cpu().numpy().astype(np.float32)
    assert np.all(np.abs(got16 - got) <= np.abs(got) * 2.0 ** -11 + 2.0 ** -25)


# products that split K over workgroups: 8, 22 and 32 slices, the last with a ragged column tile
SPLIT = [(2, 4096, 4096), (8, 11008, 1024), (3, 16384, 1000), (16, 4096, 1024)]


def _split_case(M, K, N, seed):
    from oracle import gptq
    from webpytorch_amd import core
    L = synth.gptq_layer(seed, K, N, 128, 4)
    sc = L["scales"].astype(np.float32)
    W = gptq.dequant_closed_form(L["qweight"], L["qzeros"], sc, 128, 4, 1.0).astype(np.float64)
    return L, sc, W, lambda s, x: core.QuantizedLinear.from_autogptq(L["qweight"], L["qzeros"], s, None, 128, 4).forward(x)


@pytest.mark.parametrize("weight_scale", [1.0, 0.01, 2.0 ** -20])
@pytest.mark.parametrize("M,K,N", SPLIT)
def test_split_products_at_every_magnitude(gpu, M, K, N, weight_scale):
    """Rows of one batch 2^-13 to 1 in size, layers of any scale: each row is as near its own float64
    product. An output passes at most about 140 fp32 roundings (16 steps of 32 k with up to 8 each,
    4 group folds, 4 waves; or 4 steps and up to 32 slices), each uniform within 2^-24 of a running
    sum that grows as a random walk: 2^-24 / sqrt(3) sqrt(140 / 2) = 2.9e-7 of the row's norm."""
    import torch
    L, sc, W, product = _split_case(M, K, N, M + N)
    size = 2.0 ** -np.array([0, 4, 7, 10, 13, 2, 9, 12] * 2)[:M]
    x = (synth.activations(N, M, K, np.float32) * size[:, None].astype(np.float32)).astype(np.float16)
    got = product(sc * np.float32(weight_scale), torch.from_numpy(x).cuda()).cpu().numpy().astype(np.float64)
    want = (x.astype(np.float64) @ W) * weight_scale
    for m in range(M):
        assert np.linalg.norm(got[m] - want[m]) < 3e-7 * np.linalg.norm(want[m]), m


@pytest.mark.parametrize("M,K,N", SPLIT)
def test_split_products_of_non_finite_and_huge_values(gpu, M, K, N):
    """NaN and infinities reach the outputs of their row as an fp32 sum has them, and a slice of
    1e9-sized products keeps fp32 accuracy beside the others."""
    import torch
    L, sc, W, product = _split_case(M, K, N, M + N)
    x = synth.activations(N, M, K, np.float16)
    bad = x.copy()
    bad[0, K - 5] = np.inf
    bad[1, 7] = np.nan
    got = product(sc, torch.from_numpy(bad).cuda()).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = bad[:2].astype(np.float64) @ W
    assert np.isnan(got[1]).all()
    assert np.array_equal(np.isnan(got[0]), np.isnan(want[0]))
    assert np.array_equal(np.sign(got[0][np.isinf(got[0])]), np.sign(want[0][np.isinf(want[0])]))
    clean = product(sc, torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(got[2:], clean[2:])
    sc[0] *= np.float32(1e9)
    big = W.copy()
    big[:128] *= 1e9
    got = product(sc, torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.linalg.norm(got - x.astype(np.float64) @ big) < 3e-7 * np.linalg.norm(x.astype(np.float64) @ big)


@pytest.mark.parametrize("M,K,N", [(6, 4096, 8136), (2, 4096, 11008)])
def test_captured_products_are_the_eager_ones(gpu, M, K, N):
    """A product that does not split K needs no workspace, so a capture on a stream without one
    records the kernel that an eager call runs: every replay has the eager call's bits."""
    import torch
    from webpytorch_amd import core
    L = synth.gptq_layer(M, K, N, 128, 4)
    ql = core.QuantizedLinear.from_autogptq(L["qweight"], L["qzeros"], L["scales"], None, 128, 4)
    x = torch.from_numpy(synth.activations(M, M, K, np.float16)).cuda()
    eager = ql.forward(x)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        out = ql.forward(x)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(ql.forward(x), eager)

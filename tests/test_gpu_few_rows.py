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

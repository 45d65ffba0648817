"""GPU: two threads on one stream. Products of several kernels stage their rows in the stream's one
workspace; a call's kernels are enqueued together, so each thread gets what it gets alone, bit for
bit."""
import threading

import numpy as np
import pytest

from webpytorch_amd import synth

pytestmark = pytest.mark.gpu


def _ggml(type_name, K, N):
    from webpytorch_amd import core
    return core.GGMLLinear(synth.ggml_layer(type_name, K, K, N), type_name, K, N)


def _gptq(K, N, act_order):
    from webpytorch_amd import core
    L = synth.gptq_layer(K, K, N, 128, 4, act_order=act_order)
    return core.QuantizedLinear.from_autogptq(L["qweight"], L["qzeros"], L["scales"], None, 128, 4,
                                              g_idx=L["g_idx"] if act_order else None)


@pytest.mark.parametrize("layer,dt", [
    pytest.param(lambda: _ggml("Q4_0", 4096, 1024), np.float32, id="q4_0-f32"),
    pytest.param(lambda: _ggml("Q4_K", 1024, 512), np.float16, id="q4_k-f16"),
    pytest.param(lambda: _gptq(1024, 512, False), np.float32, id="gptq-f32"),
    pytest.param(lambda: _gptq(1024, 512, True), np.float16, id="gptq-act-order-f16")])
def test_two_threads_on_one_stream(gpu, layer, dt):
    import torch
    lin = layer()
    K = lin.Kt
    xs = [torch.from_numpy(synth.activations(M, M, K, dt)).cuda() for M in (77, 130)]
    alone = [lin.forward(x) for x in xs]
    wrong = [torch.zeros((), dtype=torch.int64, device="cuda") for _ in xs]
    errors, start = [], threading.Barrier(len(xs))

    def work(i):
        try:
            start.wait(30)
            for _ in range(100):
                wrong[i] += (lin.forward(xs[i]) != alone[i]).sum()
        except Exception as e:  # reported by the test's own thread
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    torch.cuda.synchronize()
    assert not errors, errors
    assert [int(w) for w in wrong] == [0, 0]

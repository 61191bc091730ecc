"""Output tile stores of the prefill GEMMs: whole 16-byte pieces where M and y
allow them, single elements otherwise.  Row counts around the piece sizes (8
fp16, 4 fp32 values), partial row and token tiles, y one element off its
alignment: every output is the value of the aligned call (the same arithmetic),
that call is within the parity bar of the oracle, and nothing is written outside
y."""
import numpy as np
import pytest
import torch

import jllm
import oracle
import synth
from gpu_util import f16_to_f64, from_dev, print_case, rel_inf, to_dev

pytestmark = pytest.mark.gpu
GUARD = 64


@pytest.mark.parametrize("t", [12, 13, 14])
@pytest.mark.parametrize("M,N", [(136, 3), (132, 65), (130, 64), (129, 33), (7, 2), (256, 129)])
def test_gemm_output_stores(dev, t, M, N):
    print_case("gemm_store", t, M, N)
    K = 512
    g = synth.rng(M * 7 + N + t)
    W, x = synth.weights(g, t, M, K), synth.x_f16(g, (N, K))
    Wd, xd = to_dev(W), to_dev(x)
    if t == 13:
        want = np.stack([oracle.gemv_quant_cpu(W, 13, x[i], M, K) for i in range(N)])
    else:
        npad = (N + 63) // 64 * 64
        want = oracle.mmq(W, t, oracle.quantize_mmq(x, N, K, npad, t == 12), M, N, K, npad)
    for fn, dt in (("jllm_hip_gemm_quant_batched", torch.int16), ("jllm_hip_gemm_quant_batched_f32", torch.float32)):
        res = []
        for off in (0, 1):
            buf = torch.full((GUARD + off + N * M + GUARD,), 77, dtype=dt, device=dev)
            y = buf[GUARD + off:GUARD + off + N * M]
            jllm.call(fn, y, Wd, t, xd, M, N, K)
            h = from_dev(buf)
            assert np.all(h[:GUARD + off] == 77) and np.all(h[GUARD + off + N * M:] == 77)
            res.append(h[GUARD + off:GUARD + off + N * M])
        assert np.array_equal(res[0], res[1])
        if dt == torch.float32:
            assert rel_inf(res[0].reshape(N, M), want) <= 1e-3
        else:
            got = f16_to_f64(res[0].view(np.uint16)).reshape(N, M)
            assert np.all(np.abs(got - want) <= 1e-3 * np.abs(want).max() + np.abs(want) * 2 ** -10)

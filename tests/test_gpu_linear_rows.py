"""GPU parity of the dense linear above the fused rows (csrc/linear_rows.hip) where it can go wrong: rows at the edges of
its tiles (16, 32, 64, 128 rows), one to eight K-slices and the shortest k, shards of 128 and of 256 columns, every
bitrate and codebook, activations at odd addresses, fp32 in and out; against the oracle (fp32 sums, the fp16 input
Hadamards) within the repository's rel-L2 2e-3 after the same rounding to the output type."""
import numpy as np
import pytest
import torch

from oracle import exl3, linear as olin, synth
from test_gpu_linear import _group, _rel, _round

pytestmark = pytest.mark.gpu
TOL = 2e-3


@pytest.mark.parametrize("k,widths,K,cb", [(128, [128, 256], 3, 2), (640, [256, 512], 2, 2), (1152, [384], 4, 2),
                                           (512, [256], 5, 2), (2048, [256, 256], 6, 2), (384, [128], 4, 1),
                                           (768, [256], 6, 0)])
def test_linear_rows_vs_oracle(k, widths, K, cb):
    ck = olin.checkpoint(600 + k + K + cb, k, widths, K, cb)
    g = _group(ck)
    n = sum(widths)
    xf = exl3.bf16_to_f32(synth.activations(k + K, 200, k))
    ref = olin.linear(xf, ck, "small")
    for M in (9, 16, 17, 32, 33, 64, 65, 128, 129, 200):
        print(f"case linear rows k={k} widths={widths} K={K} cb={cb} M={M}", flush=True)
        for dtype in (torch.bfloat16, torch.float32):
            store = torch.zeros(M * k + 3, dtype=dtype, device="cuda")
            x = store[1:1 + M * k].view(M, k)                    # rows at an odd element
            x.copy_(torch.from_numpy(xf[:M]))
            y = g(x)
            torch.cuda.synchronize()
            got = y.float().cpu().numpy()
            want = _round(ref[:M], dtype)
            assert tuple(y.shape) == (M, n) and y.dtype == dtype and np.isfinite(got).all()
            assert _rel(got, want) < TOL, (M, dtype)
            err = np.linalg.norm((got - want).astype(np.float64), axis=1) / np.linalg.norm(want.astype(np.float64), axis=1)
            assert err.max() < 2 * TOL, (M, dtype, int(err.argmax()))

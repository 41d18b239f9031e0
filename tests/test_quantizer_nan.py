"""fp16 weights that are NaNs get index 0 and leave the scale and the other weights of their block alone, whatever their
payload and whichever kernel variant and nearest-entry rule the call takes."""
import numpy as np
import pytest

from helpers import O, to_dev

NANS = np.array([b for b in range(65536) if (b & 0x7fff) > 0x7c00], np.uint16)  # quiet and signalling, both signs


def _codebooks():
    nf4 = O.nf4_codebook()
    close = nf4.copy()
    close[8:10] = close[7] + np.float32(1e-3) * np.arange(1, 3)  # two decision boundaries in one bucket of 1/32
    return {"table": nf4, "search": close, "any": nf4[::-1].copy()}


@pytest.mark.gpu
@pytest.mark.parametrize("rule", ["table", "search", "any"])
@pytest.mark.parametrize("k,block", [(256, 8), (4096, 64), (4096, 256), (2048, None), (4096, None), (8192, None), (16384, None),
                                     (20480, None)])
def test_nan_weights_get_index_zero(rule, k, block):
    import torch

    from tuna_amd import ops

    m, rng = 64, np.random.default_rng(k)
    w = (rng.standard_normal((m, k)) * 0.02).astype(np.float16).view(np.uint16)
    at = rng.random((m, k)) < 0.1
    w[at] = rng.permutation(np.resize(NANS, int(at.sum())))
    w[0, :8], w[1, :] = NANS[:8], NANS[-1]  # blocks, and a row, of nothing else
    code = _codebooks()[rule]
    dw, dc = to_dev(w.view(np.float16), code)
    q, a, _ = ops.quantize(dw, dc, block_size=block)
    torch.cuda.synchronize()
    q_ref, a_ref = O.quantize(w, code, m, k, block_size=block)
    assert np.array_equal(a.cpu().numpy().reshape(a_ref.shape), a_ref)
    assert np.array_equal(q.cpu().numpy().reshape(q_ref.shape), q_ref)

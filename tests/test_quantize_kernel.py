"""The device quantizer (csrc/dequant_kernel.hip) at the edges of its row lengths and quads, bit-exact against the oracle."""
import numpy as np
import pytest

from helpers import O, to_dev

pytestmark = pytest.mark.gpu


# per row: one lane, ragged quads, the ends of the one-, two- and four-quad variants of 8 and 16 waves, two passes;
# more block rows than workgroups; blocks that span a lane's registers, ragged quads
@pytest.mark.parametrize("m,k,bs", [(8, 8, None), (16, 264, None), (8, 2048, None), (24, 2056, None), (16, 4104, None), (8, 8200, None),
                                    (16, 16384, None), (8, 16392, None), (8192, 136, None), (4128, 8200, None), (8, 384, 128),
                                    (4104, 320, 64), (16, 1032, 8), (8, 528, 16), (8, 768, 256), (24, 96, 32), (8, 384, 384)])
def test_edges(m, k, bs):
    import torch

    from tuna_amd import ops

    rng = np.random.default_rng(m + k)
    w = (rng.standard_normal((m, k)) * 0.03).astype(np.float16)
    w[3] = 0
    code = O.nf4_codebook()
    dw, dc = to_dev(w, code)
    q, a, _ = ops.quantize(dw, dc, block_size=bs)
    torch.cuda.synchronize()
    q_ref, a_ref = O.quantize(w.view(np.uint16), code, m, k, block_size=bs)
    assert np.array_equal(a.cpu().numpy(), a_ref)
    assert np.array_equal(q.cpu().numpy(), q_ref)

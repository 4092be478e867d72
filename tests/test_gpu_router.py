"""Router logits on the fp32 matrix cores, bit for bit: selections of the 32
largest logits and their softmax weights against the oracle's, at the edges
of the kernel's tiles (16 and 32 tokens, 16 and 32 experts per workgroup),
one and several K chunks, and both sides of its token threshold."""
import numpy as np
import pytest

import tie_amd
from conftest import bits, synth_layer
from oracle import bind
from tie_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    import torch
    assert torch.cuda.is_available(), "GPU test without a GPU"
    tie_amd.init(0)
    yield
    tie_amd.shutdown()


# (d, E, T): 16 x 16 tiles (one chunk, several, an odd number, 16; E not a
# multiple of 32; E not a multiple of 16: the row kernel), then enough
# experts for 16 x 32 and 32 x 32 tiles, with ragged last tiles
@pytest.mark.parametrize("d,E,T", [(256, 16, 32), (256, 16, 33), (512, 48, 47), (768, 128, 65), (4096, 32, 50),
                                   (512, 24, 70), (256, 128, 257), (256, 1024, 97), (512, 1024, 200),
                                   (256, 512, 391)])
@pytest.mark.parametrize("zipf", [None, 1.2])
def test_logits_bit_exact(d, E, T, zipf):
    import torch
    F, k = 256, min(E, 32)
    layer = synth_layer(211 + E, d, F, E, synth.Q4_K, synth.Q4_K, zipf)
    x = synth.make_input(212 + T, T, d)
    x[0] *= 1e-30   # sums in the denormals
    x[-1] *= 1e30   # and near the largest values (recomputed: out of the f16 range)
    x[T // 2, 3] = np.nan
    logits = bind.mat_mat(x, layer.router, synth.F32, E)
    if layer.bias is not None:
        logits = logits + layer.bias
    lib = bind.oracle()
    ri, rw = np.empty((T, k), np.int32), np.empty((T, k), np.float32)
    for t in range(T):
        lib.orc_find_top_k(logits[t].ctypes.data, E, k, ri[t].ctypes.data, rw[t].ctypes.data)
        lib.orc_softmax(rw[t].ctypes.data, k)
    L = tie_amd.Layer.from_synth(layer)
    out = torch.empty((T, d), device="cuda")
    idx = torch.empty((T, k), dtype=torch.int32, device="cuda")
    w = torch.empty((T, k), device="cuda")
    L.forward(torch.from_numpy(x).cuda(), T, k, out, idx, w, flags=tie_amd.PATH_MFMA)
    torch.cuda.synchronize()
    L.close()
    ok = np.arange(T) != T // 2
    np.testing.assert_array_equal(idx.cpu().numpy()[ok], ri[ok])
    np.testing.assert_array_equal(bits(w.cpu().numpy()[ok]), bits(rw[ok]))
    assert (idx.cpu().numpy()[T // 2] == -1).all()  # all logits NaN: nothing is selected

"""The RMSNorm in front of the block, bit for bit against the oracle: formed
inside the one-launch decode (T = 1, in place and out of place, both forms of
the kernel, one and two float4 per thread, and rows too long for it, which
take the separate kernel), and the separate kernel's chunks (T > 1).  The
host-buffer calls around it, and where the selection is written."""
import numpy as np
import pytest

import tie_amd
from conftest import bits, synth_layer
from oracle import bind
from tie_amd import synth

pytestmark = pytest.mark.gpu
EPS = 1e-6


@pytest.fixture(scope="module", autouse=True)
def device():
    import torch
    assert torch.cuda.is_available(), "GPU test without a GPU"
    tie_amd.init(0)
    yield
    tie_amd.debug_decode_form(-1)
    tie_amd.shutdown()


@pytest.mark.parametrize("T,d,F,E,k", [(1, 256, 256, 8, 2), (1, 2048, 768, 128, 8), (1, 4096, 512, 16, 4),
                                       (1, 8192, 256, 8, 2), (3, 256, 256, 8, 2), (5, 2304, 256, 8, 2),
                                       (2, 4096, 256, 8, 2)])
@pytest.mark.parametrize("form", [-1, 0, 1])
def test_norm_in_front(T, d, F, E, k, form):
    import torch
    if T > 1 and form != -1:
        pytest.skip("the form is the one-token kernel's")
    tie_amd.debug_decode_form(form)
    layer = synth_layer(401 + d, d, F, E, synth.Q4_K, synth.Q6_K, None)
    norm = synth.make_norm_weight(402 + d, d)
    hidden = synth.make_input(403 + d, T, d) * np.float32(3.0)
    ro, ri, rw = bind.qwen3_ffn(layer, hidden, k, norm, EPS)
    L = tie_amd.Layer.from_synth(layer)
    nd = torch.from_numpy(norm).cuda()
    for in_place in (False, True):
        h = torch.from_numpy(hidden).cuda()
        out = h if in_place else torch.empty_like(h)
        idx = torch.empty((T, k), dtype=torch.int32, device="cuda")
        w = torch.empty((T, k), device="cuda")
        L.forward_residual(h, nd, EPS, T, k, out, idx, w)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(idx.cpu().numpy(), ri)
        np.testing.assert_array_equal(bits(w.cpu().numpy()), bits(rw))
        np.testing.assert_array_equal(bits(out.cpu().numpy()), bits(ro))
    L.close()


# host buffers through the pinned staging (at most 256 KiB of x) and past it,
# with and without the norm and the selection, growing and shrinking
@pytest.mark.parametrize("T", [1, 2, 14, 31, 32, 33, 1])
def test_host_staging(T):
    d, F, E, k = 2048, 256, 16, 4
    layer = synth_layer(411, d, F, E, synth.Q4_K, synth.Q6_K, None)
    norm = synth.make_norm_weight(412, d)
    x = synth.make_input(413 + T, T, d)
    tie_amd.lib().tie_hip_set_exact_max_tokens(64)
    try:
        for sel in (True, False):
            out, idx, w = tie_amd.moe_ffn(x, layer, k, with_topk=sel)
            ro, ri, rw = bind.moe_block(layer, x, k)
            np.testing.assert_array_equal(bits(out), bits(ro))
            h, hidx, hw = tie_amd.qwen3_ffn(x, layer, k, norm, EPS, with_topk=sel)
            qo, qi, qw = bind.qwen3_ffn(layer, x, k, norm, EPS)
            np.testing.assert_array_equal(bits(h), bits(qo))
            if sel:
                for a, b in ((idx, ri), (hidx, qi)):
                    np.testing.assert_array_equal(a, b)
                for a, b in ((w, rw), (hw, qw)):
                    np.testing.assert_array_equal(bits(a), bits(b))
    finally:
        tie_amd.lib().tie_hip_set_exact_max_tokens(14)


@pytest.mark.parametrize("T", [1, 6, 40])
@pytest.mark.parametrize("offset", [0, 1])
def test_selection_into_callers_buffers(T, offset):
    """The selection in the caller's buffers, 16-byte aligned and not, and
    nothing beside it."""
    import torch
    d, F, E, k = 512, 256, 16, 4
    layer = synth_layer(421, d, F, E, synth.Q4_K, synth.Q6_K, None)
    x = synth.make_input(422 + T, T, d)
    _, ri, rw = bind.moe_block(layer, x, k)
    L = tie_amd.Layer.from_synth(layer)
    idx = torch.full((T * k + 8,), -7, dtype=torch.int32, device="cuda")
    w = torch.full((T * k + 8,), -7.0, device="cuda")
    L.forward(torch.from_numpy(x).cuda(), T, k, torch.empty((T, d), device="cuda"), idx[offset:], w[offset:])
    torch.cuda.synchronize()
    L.close()
    i, g = idx.cpu().numpy(), w.cpu().numpy()
    np.testing.assert_array_equal(i[offset:offset + T * k].reshape(T, k), ri)
    np.testing.assert_array_equal(bits(g[offset:offset + T * k]).reshape(T, k), bits(rw))
    assert (i[:offset] == -7).all() and (i[offset + T * k:] == -7).all() and (g[offset + T * k:] == -7).all()

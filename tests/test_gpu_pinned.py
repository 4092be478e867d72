"""Without host memory to pin, every call still answers, with the same bits:
one token by the kernels that need no status word, host buffers by copies
from and to the caller's own, and the other calls, which have no use for it,
as ever."""
import numpy as np
import pytest

import tie_amd
from conftest import bits, synth_layer
from oracle import bind
from tie_amd import synth

pytestmark = pytest.mark.gpu
D, F, E, K = 512, 256, 16, 4


@pytest.fixture(scope="module", autouse=True)
def device():
    import torch
    assert torch.cuda.is_available(), "GPU test without a GPU"
    tie_amd.init(0)
    yield
    tie_amd.lib().tie_hip_debug_fail_alloc(0)
    tie_amd.shutdown()


# (tokens, path, allocation of the first call on a stream that fails: its
# workspace is the first, the one-launch kernel's status word the second; 0:
# none)
@pytest.mark.parametrize("T,path,nth", [(1, tie_amd.PATH_EXACT, 2), (1, tie_amd.PATH_EXACT, 0),
                                        (1, tie_amd.PATH_MFMA, 2), (3, tie_amd.PATH_EXACT, 2)])
@pytest.mark.parametrize("residual", [False, True])
def test_first_call_on_a_stream(T, path, nth, residual):
    import torch
    layer = synth_layer(501, D, F, E, synth.Q4_K, synth.Q6_K, None)
    x, norm, eps = synth.make_input(502 + T, T, D), synth.make_norm_weight(503, D), 1e-6
    ref = (bind.qwen3_ffn(layer, x, K, norm, eps) if residual else bind.moe_block(layer, x, K))[0]
    L = tie_amd.Layer.from_synth(layer)
    xd, nd, out = torch.from_numpy(x).cuda(), torch.from_numpy(norm).cuda(), torch.empty((T, D), device="cuda")
    if residual:  # (the norm's table, at the library's first such call)
        L.forward_residual(xd, nd, eps, T, K, out)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    for call in range(3):
        out.fill_(np.nan)
        torch.cuda.synchronize()
        tie_amd.lib().tie_hip_debug_fail_alloc(nth if call == 0 else 0)
        if residual:
            L.forward_residual(xd, nd, eps, T, K, out, flags=path, stream=s.cuda_stream)
        else:
            L.forward(xd, T, K, out, flags=path, stream=s.cuda_stream)
        tie_amd.stream_status(s.cuda_stream)
        got = out.cpu().numpy()
        if path == tie_amd.PATH_EXACT:
            np.testing.assert_array_equal(bits(got), bits(ref))
        else:
            # (test_gpu_mfma.py's bound of the f16 operands, there derived)
            assert np.linalg.norm(got - ref) <= 1e-3 * np.linalg.norm(ref)
    tie_amd.lib().tie_hip_debug_fail_alloc(0)
    tie_amd.stream_release(s.cuda_stream)
    L.close()


@pytest.mark.parametrize("T", [1, 5])
def test_host_buffers(T):
    tie_amd.shutdown()  # no staging from earlier calls
    tie_amd.init(0)
    layer = synth_layer(511, D, F, E, synth.Q4_K, synth.Q6_K, None)
    # the layer, the workspace and the device staging, by a call whose x is
    # too large for the pinned staging
    tie_amd.moe_ffn(synth.make_input(512, 200, D), layer, K)
    x = synth.make_input(513 + T, T, D)
    ro, ri, rw = bind.moe_block(layer, x, K)
    for call in range(2):
        tie_amd.lib().tie_hip_debug_fail_alloc(1 if call == 0 else 0)  # the pinned staging
        out, idx, w = tie_amd.moe_ffn(x, layer, K)
        np.testing.assert_array_equal(bits(out), bits(ro))
        np.testing.assert_array_equal(idx, ri)
        np.testing.assert_array_equal(bits(w), bits(rw))

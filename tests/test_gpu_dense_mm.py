"""Dense products.  Exact ones of 5 and more tokens (the block dots on the fp32
matrix cores), bit for bit against the oracle's rows: quads of tokens and
their remainders, one and several groups, one super-block column and more
than the workgroup's waves, both workgroup sizes (BF16 rows: pairs of tokens
and a single one), and inputs whose products
reach zeros of both signs, denormals and infinities.  Matrix-core ones on
both sides of the K split (by the inputs, 512 and 768, and by the workgroups)
and of each of its tile heights, against a float64 model of their operands."""
import numpy as np
import pytest

import tie_amd
from conftest import bits
from oracle import bind
from test_gpu_mfma import MODEL_RL2, expert_weights, f16, rel_l2
from tie_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    import torch
    assert torch.cuda.is_available(), "GPU test without a GPU"
    tie_amd.init(0)
    yield
    tie_amd.shutdown()


@pytest.mark.parametrize("wtype", [synth.Q4_K, synth.Q6_K, synth.BF16])
@pytest.mark.parametrize("rows,inn,T", [(64, 256, 5), (64, 512, 6), (128, 256, 7), (64, 768, 8), (64, 256, 9),
                                        (64, 512, 11), (64, 2304, 13), (64, 8448, 9), (4096, 256, 34)])
def test_dense_exact_groups(wtype, rows, inn, T):
    import torch
    rng = np.random.default_rng(17 + rows + inn + T + wtype)
    w = synth.expert_tensor(rng, wtype, 1, rows, inn)
    x = synth.make_input(18 + T, T, inn)
    x[1] *= np.float32(1e-36)      # products in the denormals
    x[2, ::3] = np.float32(-0.0)
    x[3] *= np.float32(1e36)       # and past the largest value
    m = tie_amd.Matrix(w, wtype, rows, inn)
    out = torch.empty((T, rows), device="cuda")
    m.mat_mat(torch.from_numpy(x).cuda(), T, out)
    torch.cuda.synchronize()
    got, ref = out.cpu().numpy(), bind.mat_mat(x, w, wtype, rows)
    m.close()
    nan = np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(bits(got)[~nan], bits(ref)[~nan])


@pytest.mark.parametrize("wtype", [synth.Q4_K, synth.Q6_K])
def test_dense_exact_needs_no_scratch(wtype):
    """The quantised exact products take no memory: the first call on a
    stream, larger ones and one captured into a graph, with an allocation
    failure armed all along."""
    import torch
    rows, inn = 64, 512
    w = synth.expert_tensor(np.random.default_rng(41 + wtype), wtype, 1, rows, inn)
    m = tie_amd.Matrix(w, wtype, rows, inn)
    s = torch.cuda.Stream()
    xs = {T: synth.make_input(42 + T, T, inn) for T in (5, 70)}
    dev = {T: (torch.from_numpy(x).cuda(), torch.empty((T, rows), device="cuda")) for T, x in xs.items()}
    torch.cuda.synchronize()
    tie_amd.lib().tie_hip_debug_fail_alloc(1)
    try:
        for T in (5, 70):
            m.mat_mat(dev[T][0], T, dev[T][1], stream=s.cuda_stream)
        s.synchronize()
        for T in (5, 70):
            np.testing.assert_array_equal(bits(dev[T][1].cpu().numpy()), bits(bind.mat_mat(xs[T], w, wtype, rows)))
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            m.mat_mat(dev[70][0], 70, dev[70][1], stream=torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            dev[70][1].fill_(np.nan)
            g.replay()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(bits(dev[70][1].cpu().numpy()), bits(bind.mat_mat(xs[70], w, wtype, rows)))
    finally:
        tie_amd.lib().tie_hip_debug_fail_alloc(0)
    m.close()


# one workgroup per CU or fewer (32-, 64- and 128-row tiles, whole up to 512
# inputs, with their K groups from 768 on), and more
@pytest.mark.parametrize("wtype", [synth.Q4_K, synth.Q6_K])
@pytest.mark.parametrize("rows,inn,T", [(256, 256, 1), (512, 768, 33), (4096, 256, 512), (4096, 256, 1021),
                                        (4096, 512, 2047), (4096, 256, 2049), (4096, 768, 509), (4096, 768, 1021),
                                        (4096, 768, 2048), (4096, 768, 2049)])
def test_dense_mfma_k_groups(wtype, rows, inn, T):
    import torch
    rng = np.random.default_rng(29 + rows + inn + T + wtype)
    w = synth.expert_tensor(rng, wtype, 1, rows, inn)
    x = synth.make_input(30 + T, T, inn)
    m = tie_amd.Matrix(w, wtype, rows, inn)
    out = torch.full((T, rows), np.nan, device="cuda")
    m.mat_mat(torch.from_numpy(x).cuda(), T, out, flags=tie_amd.PATH_MFMA)
    torch.cuda.synchronize()
    m.close()
    ref = f16(x).astype(np.float64) @ expert_weights(w, wtype, 0, rows, inn, True).astype(np.float64).T
    assert rel_l2(out.cpu().numpy(), ref) <= MODEL_RL2

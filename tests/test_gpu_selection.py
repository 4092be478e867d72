"""The selection outputs (topk_idx, topk_w) are outputs only: whatever the
caller passes for them, and whatever other work does to them meanwhile, the
block's output keeps its bits.  One test per kernel that writes them."""
import numpy as np
import pytest

import tie_amd
from conftest import bits, synth_layer
from oracle import bind
from tie_amd import synth

pytestmark = pytest.mark.gpu
Q4, Q6, BF = synth.Q4_K, synth.Q6_K, synth.BF16
EXACT, MFMA = tie_amd.PATH_EXACT, tie_amd.PATH_MFMA


@pytest.fixture(scope="module", autouse=True)
def device():
    import torch
    assert torch.cuda.is_available(), "GPU test without a GPU"
    tie_amd.init(0)
    yield
    tie_amd.shutdown()


# (d, F, E, k, T, path, gate/up, down, no-allocation entry point): one launch;
# two launches with the selection in the first and (E > 128) before them; the
# fp32 combine on the exact path (quantised, BF16, one token) and after the
# matrix cores (BF16); the combine with the recomputation in its launch, and
# (235B's d and F) in one of its own
CASES = [(512, 256, 32, 5, 1, EXACT, Q4, Q6, False), (512, 256, 32, 5, 1, EXACT, Q4, Q6, True),
         (512, 256, 160, 7, 1, EXACT, Q4, Q4, True), (512, 256, 32, 3, 1, EXACT, BF, BF, False),
         (512, 256, 32, 5, 7, EXACT, Q4, Q6, False), (512, 256, 32, 32, 150, EXACT, Q4, Q4, False),
         (512, 256, 16, 3, 41, MFMA, BF, BF, False), (512, 256, 32, 5, 41, MFMA, Q4, Q6, False),
         (512, 256, 32, 7, 301, MFMA, Q4, Q4, False), (4096, 1536, 16, 3, 17, MFMA, Q4, Q6, False)]


def setup(case, n=0):
    import torch
    d, F, E, k, T, path, gu, dn, noalloc = case
    layer = synth_layer(301 + n, d, F, E, gu, dn, None)
    x = synth.make_input(302 + n, T, d)
    if path == MFMA and gu != BF:
        x[T // 2] *= np.float32(1e6)  # recomputed: out of the f16 range
    L = tie_amd.Layer.from_synth(layer)
    call = L.forward_noalloc if noalloc else L.forward

    def run(idx, w, x_dev=None, stream=None):
        out = torch.empty((T, d), device="cuda")
        call(torch.from_numpy(x).cuda() if x_dev is None else x_dev, T, k, out, idx, w, flags=path, stream=stream)
        return out

    return layer, L, x, k, T, run


@pytest.mark.parametrize("case", CASES)
def test_any_buffers(case):
    import torch
    layer, L, x, k, T, run = setup(case)
    _, ri, rw = bind.moe_block(layer, x, k)

    def check(out, idx, w, what):
        torch.cuda.synchronize()
        np.testing.assert_array_equal(bits(out.cpu().numpy()), want, what)
        if idx is not None:
            np.testing.assert_array_equal(idx.cpu().numpy().reshape(T, k), ri, what)
        if w is not None:
            np.testing.assert_array_equal(bits(w.cpu().numpy()).reshape(T, k), bits(rw), what)

    want = run(None, None)
    torch.cuda.synchronize()
    want = bits(want.cpu().numpy())
    buf = torch.full((2 * T * k + 2,), -7, dtype=torch.int32, device="cuda")
    idx, w = buf[1:T * k + 1], buf[T * k + 1:2 * T * k + 1].view(torch.float32)
    check(run(idx, w), idx, w, "apart, 4-byte aligned")
    assert buf[0].item() == -7 and buf[-1].item() == -7
    buf.fill_(-7)
    check(run(idx, None), idx, None, "indices only")
    check(run(None, w), None, w, "weights only")
    check(run(buf, buf), None, buf[:T * k].view(torch.float32), "one buffer for both: the weights last")
    xd = torch.from_numpy(x).cuda()
    over = xd.view(-1)[:T * k].view(torch.int32)
    check(run(over, w, xd), over, w, "indices over x")
    L.close()


@pytest.mark.parametrize("case", CASES[:1] + CASES[3:])
def test_shared_by_two_streams(case):
    import torch
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    lanes = [setup(case, 10 * i) for i in range(2)]
    k, T = lanes[0][3], lanes[0][4]
    xs = [torch.from_numpy(l[2]).cuda() for l in lanes]
    idx = torch.empty((T, k), dtype=torch.int32, device="cuda")
    w = torch.empty((T, k), device="cuda")
    want = [l[5](None, None) for l in lanes]
    torch.cuda.synchronize()
    for rep in range(4):
        got = []
        for _ in range(4):
            for i, l in enumerate(lanes):
                got.append((i, l[5](idx, w, xs[i], streams[i].cuda_stream)))
        torch.cuda.synchronize()
        for i, out in got:
            np.testing.assert_array_equal(bits(out.cpu().numpy()), bits(want[i].cpu().numpy()), "stream %d" % i)
    for l in lanes:
        l[1].close()
    for s in streams:
        tie_amd.stream_release(s.cuda_stream)

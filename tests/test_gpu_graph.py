"""HIP graph capture of the entry points (after one eager call has sized the
scratch, as tc_gemv_reserve documents): every replay, with eager work and
synchronizations between replays, must reproduce the eager results bit for
bit."""
import numpy as np
import pytest

from qdata import IQ4_NL, Q4_K, Q6_K, Q8_0, gaussian, random_blocks

pytestmark = pytest.mark.gpu


def to_dev(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def test_graph_replays_match_eager(tc, dev):
    import torch
    import tc_hip
    rng = np.random.default_rng(21)
    rows, cols, M = 700, 2048, 40
    w4 = to_dev(random_blocks(Q4_K, rng, rows, cols), dev)
    wu = to_dev(random_blocks(Q4_K, rng, rows, cols), dev)
    w8 = to_dev(random_blocks(Q8_0, rng, rows, cols), dev)
    x1 = to_dev(gaussian(rng, (1, cols)), dev)
    xm = to_dev(gaussian(rng, (M, cols)), dev)
    outs = {k: torch.empty(shape, device=dev) for k, shape in
            (("gemv", (1, rows)), ("g", (1, rows)), ("u", (1, rows)), ("q8", (1, rows)), ("gemm", (M, rows)),
             ("gemm8", (M, rows)))}

    def work():
        tc.gemv(Q4_K, w4, x1, rows, cols, out=outs["gemv"])
        tc._check(tc.lib.tc_gemv_dual(Q4_K, tc_hip._ptr(w4), tc_hip._ptr(wu), tc_hip._ptr(x1), tc_hip._ptr(outs["g"]),
                                      tc_hip._ptr(outs["u"]), rows, cols, tc._stream()))
        tc.gemv(Q8_0, w8, x1, rows, cols, out=outs["q8"])
        tc.gemm(Q4_K, w4, xm, rows, cols, out=outs["gemm"])
        tc.gemm(Q8_0, w8, xm, rows, cols, out=outs["gemm8"])

    work()  # sizes the scratch
    torch.cuda.synchronize()
    ref = {k: v.clone() for k, v in outs.items()}
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            work()
    torch.cuda.synchronize()
    for rep in range(3):
        for v in outs.values():
            v.fill_(float("nan"))  # eager work between replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for k in outs:
            assert torch.equal(outs[k], ref[k]), (rep, k)


def test_graph_scratch_outlives_growth(tc, dev):
    """Reserve, capture, then eager calls of at most the reserved size and a
    larger reservation: the replays go on using the buffers they were recorded
    with. The wide decode (prequantized activations), the prefill GEMM
    (activations and partials) and the MoE FFN (intermediates) hold an address."""
    import torch
    rng = np.random.default_rng(22)
    rows, cols, H, FF, E = 40, 18944, 512, 256, 4
    w4, w6, wn = (to_dev(random_blocks(t, rng, rows, cols), dev) for t in (Q4_K, Q6_K, IQ4_NL))
    x1, x8 = to_dev(gaussian(rng, (1, cols)), dev), to_dev(gaussian(rng, (8, cols)), dev)
    experts = [to_dev(random_blocks(Q4_K, rng, E * r, c), dev) for r, c in ((FF, H), (FF, H), (H, FF))]
    xe = to_dev(gaussian(rng, (2, H)), dev)
    ids = to_dev(np.array([[0, 3], [2, 1]], np.int32), dev)
    wts = to_dev(np.array([[0.75, 0.25], [0.5, 0.5]], np.float32), dev)
    outs = {"q6": torch.empty((1, rows), device=dev), "gemm": torch.empty((8, rows), device=dev)}

    def work():
        tc.gemv(Q6_K, w6, x1, rows, cols, out=outs["q6"])
        tc.gemm(Q4_K, w4, x8, rows, cols, out=outs["gemm"])
        outs["moe"] = tc.moe_ffn(xe, ids, wts, *experts, E, H, FF)

    tc._check(tc.lib.tc_gemv_reserve(cols, 8))
    work()
    torch.cuda.synchronize()
    ref = {k: v.clone() for k, v in outs.items()}
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        work()
    for step in range(3):
        if step == 0:
            tc.gemv(Q6_K, w6, x8[:4].contiguous(), rows, cols)  # of at most the reserved size
            tc.gemm(IQ4_NL, wn, x8, rows, cols)
        elif step == 1:
            tc._check(tc.lib.tc_gemv_reserve(4096, 1 << 17))  # larger than any call of this suite: the buffers grow
        junk = [torch.full((1 << 24,), float("nan"), device=dev) for _ in range(8)]
        for v in outs.values():
            v.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for k in outs:
            assert torch.equal(outs[k], ref[k]), (step, k)
        del junk

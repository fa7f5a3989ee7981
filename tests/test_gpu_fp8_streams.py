"""dsv4_gpu_fp8_gemv_n_d on several streams and under capture. Its tiles split
over workgroups (few tiles, rows of 4096 columns on) leave part sums for a
second launch; calls on different streams that overlap must not meet in them,
and a captured call must hold no scratch that a later call could use or free.
Every result has the single-token GEMV's bits, whichever form a call took."""
import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu

# split over 2, 4, 4, 3 workgroups a tile (12288 columns: rows of 192 slots)
SHAPES = [(1536, 7168, 13), (512, 4096, 16), (1024, 16384, 16), (300, 12288, 9)]


def _problem(torch, gpu, seed, rows, cols, nt):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    w = torch.randint(0, 127, (rows, cols), generator=g, device="cuda", dtype=torch.uint8)
    s = torch.randint(119, 123, (-(-rows // 128), -(-cols // 128)), generator=g, device="cuda",
                      dtype=torch.uint8)
    x = torch.randn(nt, cols, generator=g, device="cuda")
    y = torch.empty(nt, rows, device="cuda")
    want = torch.empty(nt, rows, device="cuda")
    for t in range(nt):
        assert gpu.dsv4_gpu_fp8_gemv_d(want[t].data_ptr(), x[t].data_ptr(), w.data_ptr(),
                                       s.data_ptr(), 0, rows, cols, None) == 0
    return dict(w=w, s=s, x=x, y=y, want=want.cpu().numpy(), rows=rows, cols=cols, nt=nt)


def _call(gpu, p, stream):
    assert gpu.dsv4_gpu_fp8_gemv_n_d(p["y"].data_ptr(), p["x"].data_ptr(), p["w"].data_ptr(),
                                     p["s"].data_ptr(), 0, p["rows"], p["cols"], p["nt"],
                                     stream) == 0


@pytest.mark.parametrize("n", [2, 12])
def test_overlapping_streams(gpu, dsv4, n):
    """n streams at once, each with its own x and y (12: more than have a place
    for part sums); 40 calls on each, its shape changing from call to call."""
    import torch
    streams = [torch.cuda.Stream() for _ in range(n)]
    probs = [[_problem(torch, gpu, 10 * i + k, *sh) for k, sh in enumerate(SHAPES)]
             for i in range(n)]
    torch.cuda.synchronize()
    for rep in range(10):
        for i, st in enumerate(streams):
            for p in probs[i]:
                _call(gpu, p, st.cuda_stream)
    torch.cuda.synchronize()
    for i in range(n):
        for p in probs[i]:
            assert common.bits_equal(p["y"].cpu().numpy(), p["want"]), (i, p["rows"], p["cols"])


@pytest.mark.parametrize("k", range(len(SHAPES)))
def test_capture(gpu, dsv4, k):
    """Captured on a stream that has run nothing, replayed on another while
    eager calls run on the first, every replay checked."""
    import torch
    p = _problem(torch, gpu, 77 + k, *SHAPES[k])
    other = _problem(torch, gpu, 99 + k, *SHAPES[k])
    cap, run = torch.cuda.Stream(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=cap):
        _call(gpu, p, cap.cuda_stream)
    for rep in range(4):
        p["y"].zero_()
        other["y"].zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(run):
            graph.replay()
        for _ in range(3):
            _call(gpu, other, cap.cuda_stream)
        torch.cuda.synchronize()
        assert common.bits_equal(p["y"].cpu().numpy(), p["want"]), rep
        assert common.bits_equal(other["y"].cpu().numpy(), other["want"]), rep

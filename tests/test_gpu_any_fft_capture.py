"""The run-time-length transforms inside a captured HIP graph (they replaced library transforms there
too): several replays with new inputs, eager work and synchronisation in between, each equal to the
eager call. Lengths with LDS below and above the size a kernel has to ask for, each kind of plan."""

import math

import pytest
import torch

from test_gpu_any_fft import _rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,G", [((70, 60), (88, 75)), ((400, 30), (500, 37)), ((30, 230), (38, 293)),
                                 ((270, 400), (340, 510)), ((20, 24, 90), (25, 29, 113))])
def test_replays_equal_eager(dev, N, G):
    from mr_recon_amd import ops

    x, smaps = _rand((1, *N), 1, dev), _rand((3, *N), 2, dev)
    kern = _rand(G, 3, dev) / math.prod(G)

    def run():
        g = ops.pad_fft(x, N, G, smaps=smaps)
        keep = g.clone()
        return keep, ops.ifft_crop(g, N, G, 1, smaps=smaps), ops.toeplitz_normal(x[0], N, G, smaps, kern)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()  # tables and kernel attributes, before the capture
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for seed in range(4):
        x.copy_(_rand((1, *N), 10 + seed, dev))
        graph.replay()
        torch.cuda.synchronize()
        for got, want in zip(out, run()):
            assert torch.equal(got, want)
        torch.cuda.synchronize()

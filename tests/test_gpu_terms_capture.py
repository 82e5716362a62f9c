"""The term-by-term H.v needs no workspace: it runs in a stream capture that no
H.v came before on the stream, as the same kernel."""
import numpy as np
import pytest
import torch

import mcpi_amd
from tests.gpu_util import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M", [(6, 9), (3, 14)])
def test_first_call_under_capture(N, M):
    note(f"terms under capture N={N} M={M}")
    mats = mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, 4.0)
    rng = np.random.default_rng(N)
    b = mcpi_amd.Basis(N, M, "full")
    H = mcpi_amd.Hamiltonian(b, *mats, schedule=7)
    C, out = mcpi_amd.DeviceArray(b.nc), mcpi_amd.DeviceArray(b.nc)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        H.apply(C, out, stream=stream.cuda_stream)
    eager = mcpi_amd.Hamiltonian(mcpi_amd.Basis(N, M, "full"), *mats, schedule=7)
    for k in range(3):
        v = rng.standard_normal(b.nc) + 1j * rng.standard_normal(b.nc)
        C.upload(v)
        mcpi_amd.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.numpy(), eager(v)), k

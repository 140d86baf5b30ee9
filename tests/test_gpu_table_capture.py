"""pt_location_table_noalloc under stream capture, in each of its forms: one
launch with one copy of the counters, with several, with more than 64 KB of
LDS, and the radix build.  Replayed with other keys, with eager work between."""
import numpy as np
import pytest

from test_gpu_location_table import closed_form

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K", [(20_000, 545), (131_072, 100), (131_072, 2500), (131_072, 5000), (131_073, 5000)])
def test_captured_tables(n, K):
    import torch
    from pandemicthrust_amd.api import lib
    L = lib()
    rng = np.random.default_rng(n + K)
    keys = torch.zeros(n, dtype=torch.int32, device="cuda")
    people = torch.empty(n, dtype=torch.int32, device="cuda")
    offsets = torch.empty(K + 1, dtype=torch.int32, device="cuda")

    def call(stream):
        return L.pt_location_table_noalloc(keys.data_ptr(), n, K, people.data_ptr(), offsets.data_ptr(), 0,
                                           stream.cuda_stream)

    assert call(torch.cuda.current_stream()) == 0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert call(torch.cuda.current_stream()) == 0
    for k in range(4):
        host = rng.integers(0, K, n, dtype=np.uint32)
        host[: n // 3] = K // 2
        keys.copy_(torch.from_numpy(host.astype(np.int32)))
        people.fill_(-1)
        offsets.fill_(-1)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want_p, want_o = closed_form(host, K)
        assert np.array_equal(offsets.cpu().numpy(), want_o) and np.array_equal(people.cpu().numpy(), want_p), k

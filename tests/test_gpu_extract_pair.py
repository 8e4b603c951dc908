"""A's rows and B's columns extracted in one launch (both of at most 4096
elements): products equal to the oracle's bit for bit at the edges of its
shapes, for operands that allow 16-byte loads and for views that do not."""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


# 256, 1024, 2048 and 4096 (4096 and not 4097, which is not extracted so)
# end a shape; one line, one column, 64 and 65 lines
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 2, 65), (64, 255, 1), (65, 256, 64),
                                   (2, 257, 129), (7, 1024, 5), (66, 1025, 3), (5, 2048, 64),
                                   (65, 2049, 2), (3, 4095, 66), (9, 4096, 4), (4, 4097, 5)])
@pytest.mark.parametrize("view", [False, True])
def test_pair_extraction_edges(ozk, shape, view):
    import torch
    N, K, M = shape
    rng = np.random.RandomState(N + K + M)
    A = rng.randn(N, K) * np.exp(3 * rng.randn(N, 1))
    B = rng.randn(K, M) * np.exp(3 * rng.randn(1, M))

    def device(X):
        if not view:
            return torch.from_numpy(X).to("cuda")
        t = torch.zeros((X.shape[0], X.shape[1] + 3), dtype=torch.float64, device="cuda")
        t[:, 1:1 + X.shape[1]] = torch.from_numpy(X)
        return t[:, 1:1 + X.shape[1]]

    print(f"[case] extraction of both operands {shape} view={view}", flush=True)
    for acc, ref in (("fused", O.matmul_ondevice_a4), ("host", O.matmul_ondevice_a3)):
        C = ozk.matmul(device(A), device(B), pipeline="ondevice", accumulation=acc)
        assert np.array_equal(C.cpu().numpy(), ref(A, B)), acc

"""Products of few tiles: 32-row tiles, and K split over the CUs where the
model of its cost says so; equal to the oracle's bit for bit at the edges."""

import numpy as np
import pytest

import oracle as O
from oracle import pipeline as OP

pytestmark = pytest.mark.gpu


def operands(N, K, M):
    rng = np.random.RandomState(N + K + M)
    return (rng.randn(N, K) * np.exp(2 * rng.randn(N, 1)),
            rng.randn(K, M) * np.exp(2 * rng.randn(1, M)))


# One row or column; both sides of 32 and 64 rows; 256 tiles of 32 rows (the
# last shape that takes them) and more; one stage and a ragged last one.  With K
# split: 4 tiles on BF16 and INT8 planes, 256 tiles in 2 pieces, 16 tiles
# after a round of 64-row ones, and (medium) of 96-row ones.  Long K, where the
# usual tiles come back (64 and 96 rows), and where they do not yet.  128 tiles
# of 96 rows after a round, of the fewest pairs.
@pytest.mark.parametrize("shape,precision", [
    ((1, 1, 1), "high"), ((31, 33, 64), "high"), ((33, 32, 65), "max"), ((65, 300, 63), "medium"),
    ((1024, 70, 512), "high"), ((1024, 70, 512), "max"), ((1024, 70, 512), "medium"),
    ((1025, 70, 512), "high"), ((1025, 70, 512), "medium"),
    ((40, 4096, 60), "high"), ((40, 8200, 60), "high"), ((40, 8200, 60), "medium"),
    ((500, 4090, 510), "high"), ((1056, 4200, 1024), "high"), ((1600, 4200, 1030), "medium"),
    ((384, 24000, 512), "high"), ((384, 24000, 512), "medium"), ((384, 12000, 512), "high"),
    ((1536, 4096, 1536), (1, 1))])
def test_few_tiles_ondevice(ozk, shape, precision):
    N, K, M = shape
    A, B = operands(N, K, M)
    nh, nl = OP.resolve_precision(precision)
    rows = np.unique(np.r_[0:min(N, 34), N // 2:min(N, N // 2 + 4), max(0, N - 34):N])
    for acc, ref in (("fused", O.matmul_ondevice_a4), ("host", O.matmul_ondevice_a3)):
        print(f"[case] few tiles {shape} {precision} {acc}", flush=True)
        C = ozk.matmul(A, B, pipeline="ondevice", accumulation=acc, precision=precision)
        assert np.array_equal(C[rows], ref(A[rows], B, "raise", nh, nl)), acc


@pytest.mark.parametrize("shape,n", [((1, 1, 1), 8), ((33, 65, 70), 8), ((1024, 40, 512), 8),
                                     ((1025, 40, 512), 8), ((70, 1100, 33), 9)])
def test_few_tiles_host(ozk, shape, n):
    N, K, M = shape
    A, B = operands(N, K, M)
    rows = np.unique(np.r_[0:min(N, 34), max(0, N - 34):N])
    print(f"[case] few tiles host {shape} {n} slices", flush=True)
    assert np.array_equal(ozk.matmul(A, B, n_slices=n)[rows],
                          OP.matmul_host_a2(A[rows], B, n_slices=n))
    assert np.array_equal(ozk.matmul_numpy(A, B, n_slices=n)[rows],
                          O.matmul_numpy(A[rows], B, n_slices=n))

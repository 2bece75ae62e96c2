"""Which kernel serves a call, decided on the host (no GPU): the choices that entry points promise
to share.  Shapes are of ordinary models, ragged, and at the edges of the ranges of M."""
import ctypes

import pytest

import mlxr_amd as mx
from mlxr_amd import qgemm

Q4K, Q5K, Q6K, Q80, Q40 = (mx.QuantType.Q4_K, mx.QuantType.Q5_K, mx.QuantType.Q6_K, mx.QuantType.Q8_0,
                           mx.QuantType.Q4_0)
MS = (5, 17, 32, 33, 48, 64, 65, 100, 128, 256, 257, 333, 512, 1024, 2048, 2049)


def _grouped_need(weights, M):
    arr = (qgemm.Item * len(weights))(*[qgemm.Item(int(q), N, K) for q, N, K in weights])
    v = ctypes.c_size_t(0)
    qgemm._check(mx.lib().mlxr_qgemm_grouped_workspace_size(len(weights), arr, M, ctypes.byref(v)))
    return v.value


GROUPS = [
    [(Q4K, 4096, 4096), (Q4K, 1024, 4096), (Q4K, 1024, 4096)],
    [(Q4K, 8192, 8192), (Q4K, 1024, 8192), (Q6K, 1024, 8192)],
    [(Q4K, 14336, 4096)] * 2,
    [(Q4K, 28672, 8192)] * 2,
    [(Q80, 2048, 2048), (Q80, 256, 2048), (Q80, 256, 2048)],
    [(Q4K, 512, 256), (Q4K, 1, 256)],
    [(Q6K, 5632, 2048)] * 2,
    [(Q5K, 100, 768)] * 5,
    [(Q40, 512, 96), (Q40, 65536, 96)],
    [(Q4K, 128256, 4096)],
    [(Q80, 65536, 2048), (Q80, 33, 2048)],
]


@pytest.mark.parametrize("g", range(len(GROUPS)))
def test_grouped_workspace_below_its_size_is_none(g):
    """A grouped call with less workspace than its size (or with any where its size is 0) takes
    the kernels and launches of one without a workspace."""
    for M in MS:
        need = _grouped_need(GROUPS[g], M)
        none = qgemm.test_kernels("grouped", GROUPS[g], M)
        for nbytes in (1, need // 2, need - 1) if need else (1, 1 << 30):
            assert qgemm.test_kernels("grouped", GROUPS[g], M, nbytes) == none, (M, need, nbytes)


@pytest.mark.parametrize("g", range(len(GROUPS)))
def test_grouped_without_workspace_takes_kernels_of_single_calls(g):
    """Without a workspace a grouped call equals separate calls bit for bit (M > 4): every item
    runs on the kernel of its own call, and items of different types or kernels share no launch."""
    for M in MS:
        kernels, launches = qgemm.test_kernels("grouped", GROUPS[g], M)
        assert kernels == qgemm.test_kernels("single", GROUPS[g], M)[0], M
        for i in range(len(kernels)):
            together = [j for j in range(len(kernels)) if launches[j] == launches[i]]
            assert len(together) <= 4
            assert {(kernels[j], GROUPS[g][j][0]) for j in together} == {(kernels[i], GROUPS[g][i][0])}, M


def test_skinny_launch_counts_the_items_of_all_its_weights():
    """The skinny kernel finds an item's slab by a multiplication that is exact for fewer than 2^32 /
    blocks of M items: weights that are within it alone and past it together do not share a
    launch (the quotient of the last items would be wrong, as it is here for two of them)."""
    M, N, K, blocks = 2000, 12_000_000, 32, 63
    mdiv = -(-2**32 // blocks)
    last = lambda n: n * (N // 16) - 1  # the last slab of n weights
    assert ((last(1) * blocks + blocks - 1) * mdiv) >> 32 == last(1)
    assert ((last(2) * blocks + blocks - 1) * mdiv) >> 32 != last(2)
    try:
        qgemm.test_force_skinny(True)
        for nbytes in (0, 1 << 40):
            kernels, launches = qgemm.test_kernels("grouped", [(Q40, N, K)] * 4, M, nbytes)
            assert kernels != [qgemm.KERNEL_SKINNY] * 4 or len(set(launches)) == 4
            assert qgemm.test_kernels("grouped", [(Q40, N // 4, K)] * 4, M, nbytes) == ([qgemm.KERNEL_SKINNY] * 4, [0] * 4)
    finally:
        qgemm.test_force_skinny(False)

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
    """A grouped call with less workspace than its size takes the kernels and launches of one without
    a workspace; a size of 0 asks for none."""
    for M in MS:
        need = _grouped_need(GROUPS[g], M)
        none = qgemm.test_kernels("grouped", GROUPS[g], M)
        for nbytes in (0, 1, need // 2, need - 1) if need else ():
            assert qgemm.test_kernels("grouped_ws", GROUPS[g], M, nbytes) == none, (M, need, nbytes)
        if need == 0:
            assert qgemm.test_kernels("grouped_ws", GROUPS[g], M) == qgemm.test_kernels("grouped_ws", GROUPS[g], M, 1 << 30)


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
        for call in ("grouped", "grouped_ws"):
            kernels, launches = qgemm.test_kernels(call, [(Q40, N, K)] * 4, M)
            assert kernels != [qgemm.KERNEL_SKINNY] * 4 or len(set(launches)) == 4
            assert qgemm.test_kernels(call, [(Q40, N // 4, K)] * 4, M) == ([qgemm.KERNEL_SKINNY] * 4, [0] * 4)
    finally:
        qgemm.test_force_skinny(False)


# (call, weights, M, the kernel; measured on MI355X, us, skinny / tiled with the workspace asked for)
MEASURED = [
    ("single", [(Q6K, 18944, 3584)], 96, "tiled", 57.4, 44.7),
    ("single", [(Q6K, 11008, 4096)], 333, "tiled", 104.9, 72.5),
    ("single", [(Q6K, 2048, 5632)], 512, "tiled", 38.9, 33.4),
    ("single", [(Q4K, 28672, 8192)], 128, "tiled", 147.9, 78.2),
    ("single", [(Q4K, 1024, 4096)], 128, "skinny", 7.2, 11.8),
    ("single", [(Q4K, 4096, 4096)], 64, "skinny", 10.7, 18.1),
    ("single", [(Q4K, 5120, 5120)], 33, "skinny", 18.7, 59.8),
    ("single", [(Q4K, 3072, 8192)], 64, "skinny", 16.9, 26.3),
    ("single", [(Q80, 8192, 8192)], 48, "skinny", 29.2, 36.2),
    ("single", [(Q80, 8192, 8192)], 64, "skinny", 31.1, 35.7),
    ("single", [(Q5K, 5120, 5120)], 64, "skinny", 22.8, 25.3),
    ("single", [(Q4K, 3072, 8192)], 96, "skinny", 23.8, 26.8),
    ("single", [(Q80, 896, 4864)], 333, "skinny", 19.4, 23.0),
    ("single", [(Q80, 6144, 16384)], 96, "tiled", 83.7, 64.2),
    ("single", [(Q4K, 14336, 4096)], 128, "tiled", 48.8, 33.7),
    ("swiglu", [(Q6K, 18944, 3584)], 96, "tiled", 99.9, 69.0),
    ("swiglu", [(Q6K, 28672, 8192)], 33, "tiled", 203.7, 148.1),
    ("swiglu", [(Q4K, 5632, 2048)], 64, "skinny", 16.2, 19.9),
    ("grouped_ws", [(Q6K, 14336, 4096)] * 2, 64, "tiled", 63.3, 51.6),
    ("grouped_ws", [(Q4K, 4096, 4096), (Q4K, 1024, 4096), (Q4K, 1024, 4096)], 64, "skinny", 14.6, 23.0),
]


@pytest.mark.parametrize("call,weights,M,kernel,skinny_us,tiled_us", MEASURED)
def test_kernel_is_the_faster_one(call, weights, M, kernel, skinny_us, tiled_us):
    """With the workspace asked for, the faster of the skinny and the tiled kernel serves the call."""
    assert kernel == ("skinny" if skinny_us < tiled_us else "tiled")
    qt, N, K = weights[0]
    if call == "single":
        need = mx.workspace_size(qt, N, K, M)
    elif call == "swiglu":
        v = ctypes.c_size_t(0)
        qgemm._check(mx.lib().mlxr_qgemm_swiglu_workspace_size(int(qt), N, K, M, mx.BF16, ctypes.byref(v)))
        need = v.value
    else:
        need = _grouped_need(weights, M)
    kernels = qgemm.test_kernels(call, weights, M, need)[0]
    skinny = [k == qgemm.KERNEL_SKINNY for k in kernels]
    assert all(skinny) if kernel == "skinny" else not any(skinny), kernels


def test_skinny_tiles_fill_whole_rounds():
    """5120 rows in two blocks of M: four tiles per wavefront (160 workgroups, one round of the CUs) and
    not two (320, two rounds; Q4_K, K = 13824, 36.9 against 47.4 us)."""
    assert qgemm.test_skinny_layout(Q4K, 5120, 13824, 33)[0] == 4


# (type, N, K, M, bytes of a single call, of the fused SwiGLU)
SIZES = [
    (3, 4096, 4096, 4, 0, 0), (3, 4096, 14336, 4, 131072, 0),
    (4, 1024, 8192, 13, 425984, 425984), (2, 2048, 2048, 8, 262144, 262144),
    (3, 2048, 14336, 32, 1048576, 1048576), (0, 512, 4096, 17, 278528, 557056),
    (10, 896, 4864, 24, 430080, 860160), (4, 128256, 4096, 6, 0, 0),
    (3, 1024, 4096, 33, 1081344, 2162688), (3, 4096, 14336, 33, 7569408, 7569408),
    (2, 256, 2048, 64, 524288, 524288), (3, 14336, 4096, 64, 14680064, 14680064),
    (4, 5632, 2048, 100, 0, 18022400), (3, 5120, 13824, 48, 8847360, 11796480),
    (2, 2048, 5632, 333, 16367616, 21823488), (3, 4096, 4096, 512, 33554432, 33554432),
    (3, 4096, 14336, 1024, 67108864, 67108864), (4, 8192, 28672, 256, 67108864, 67108864),
    (1, 33, 96, 70, 0, 0), (3, 28672, 8192, 2048, 0, 0),
]


@pytest.mark.parametrize("entry", SIZES)
def test_reported_workspace_sizes_stay(entry):
    """The workspace sizes reported decide how callers allocate and which calls
    mlxr_qgemm_run_noalloc takes: they do not follow the choice of kernels."""
    qt, N, K, M, single, swiglu = entry
    v = ctypes.c_size_t(0)
    assert mx.workspace_size(qt, N, K, M) == single
    qgemm._check(mx.lib().mlxr_qgemm_swiglu_workspace_size(qt, N, K, M, mx.BF16, ctypes.byref(v)))
    assert v.value == swiglu

"""Small- and mid-M tiles of the bf16 GEMM (16 x 16 to 128 x 128 on the 16 x 16 x 32 MFMA): every
row equals the row of a 256 x 256-tile call (32 x 32 x 16 MFMA) bit for bit, at sizes on both sides of
each tile's limit, with partial last row tiles, at K values that leave out the deep-stage tiles, and with
a row pitch too wide for 32-bit tile offsets."""

import numpy as np
import pytest
import torch

from yapd_amd import kernels

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
BIG = 16384


def rnd(*shape, std=1.0, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(BF)


# N = 1024: 16 x 16 up to M = 64, 32 x 16 to 128, 32 x 32 to 256, 64 x 32 to 512, 64 x 64 to 1024, 128 x 64 to
# 2048, 128 x 128 to 4096
SIZES = (1, 15, 17, 64, 65, 100, 113, 127, 128, 129, 256, 257, 511, 513, 1000, 1025, 1900, 2049, 3000, 4096)


@pytest.mark.parametrize("epi", ["store", "residual"])
@pytest.mark.parametrize("N,K", [(1024, 1024), (1024, 4096), (1000, 512)])
def test_rows_equal_the_large_tiles(dev, epi, N, K):
    A, W, R = rnd(BIG, K, std=0.5, seed=1), rnd(N, K, std=0.02, seed=2), rnd(BIG, N, seed=3)

    def call(M):
        C = R[:M].clone()
        (kernels.gemm_bf16_residual if epi == "residual" else kernels.gemm_bf16)(A[:M], W, C)
        return C

    ref = call(BIG)
    for M in SIZES:
        assert torch.equal(call(M), ref[:M]), M


@pytest.mark.parametrize("M", [1, 16, 33, 64, 100, 128, 200, 256, 300, 512, 900])
def test_swiglu_rows_equal_the_large_tiles(dev, M):
    A, W = rnd(8192, 1024, seed=4), rnd(8192, 1024, std=0.02, seed=5)
    out = [torch.empty(m, 4096, dtype=BF, device=dev) for m in (8192, M)]
    for o in out:
        kernels.gemm_swiglu(A[: len(o)], W, o)
    assert torch.equal(out[0][:M], out[1])


@pytest.mark.parametrize("rows,bl", [(1, 1), (3, 5), (2, 32), (5, 32), (8, 16), (17, 13), (32, 16), (40, 32)])
@pytest.mark.parametrize("H", [16, 4])
def test_qkv_rows_equal_the_large_tiles(dev, rows, bl, H):
    """Blocks that start at any slot of a page; H = 4: 64-column groups of q, k and v share a tile."""
    D, big = 1024, 16384 // bl
    A, W = rnd(big * bl, D, seed=6), rnd(3 * H * 64, D, std=0.02, seed=7)
    fr = torch.outer(torch.arange(400.0), 10000.0 ** (-torch.arange(0, 64, 2) / 64))
    cos, sin = (torch.cat([f, f], -1).to(BF).float().to(dev) for f in (fr.cos(), fr.sin()))
    rng = np.random.default_rng(8)
    pos0 = torch.from_numpy(rng.integers(0, 300, big).astype(np.int32)).to(dev)
    cols = (300 + bl) // 16 + 1
    table = torch.from_numpy(rng.permutation(big * cols).reshape(big, cols).astype(np.int32)).to(dev)
    got = []
    for n in (big, rows):
        pool = torch.zeros(big * cols, 2, H, 1024, dtype=BF, device=dev)
        q = torch.empty(n * bl, H * 64, dtype=BF, device=dev)
        kernels.gemm_qkv_rope_kv(A[: n * bl], W, cos, sin, pos0[:n], bl, q, pool, table[:n])
        got.append((q[: rows * bl], pool[table[:rows].long()]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("rows,bl", [(1, 7), (2, 32), (9, 16), (30, 16), (70, 32)])
def test_head_rows_equal_the_large_tiles(dev, rows, bl):
    D, V, big = 1024, 8194, 8192 // bl
    hid, ctx, W = rnd(big, bl, D, seed=9), rnd(big, 1, D, seed=10), rnd(V, D, std=0.02, seed=11)
    out = [torch.empty(n, bl, 8200, dtype=BF, device=dev)[..., :V] for n in (big, rows)]
    for o in out:
        kernels.gemm_head_shift(hid[: len(o)], ctx[: len(o)], W, o)
    assert torch.equal(out[0][:rows], out[1])


@pytest.mark.parametrize("K", [64, 128, 192, 320, 1344])
@pytest.mark.parametrize("M", [40, 1000, 3000])
def test_short_and_odd_k(dev, K, M):
    """Products of fp32 sums of K exact bf16 products against fp64, rounded to bf16: half a bf16 ulp
    (2^-9 relative) plus the sums' own error, K * 2^-24 of the sum of magnitudes."""
    A, W = rnd(M, K, seed=12), rnd(1024, K, std=0.02, seed=13)
    C = torch.empty(M, 1024, dtype=BF, device=dev)
    kernels.gemm_bf16(A, W, C)
    ref = A.double() @ W.double().T
    mag = A.double().abs() @ W.double().abs().T
    assert ((C.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * K * 2.0 ** -24).all()


@pytest.mark.parametrize("K", [64, 128, 192, 320, 512, 576, 1088, 1344, 2048])
def test_short_k_rows_equal_the_large_tiles(dev, K):
    """129 to 256 tiles of 128 x 128: three stages of gemm_dl_kernel at short K, gemm_sk_kernel above, whose limit
    depends on the epilogue; one k-tile, as many as the stages hold, and more."""
    A, W, R = rnd(BIG, K, std=0.5, seed=19), rnd(1024, K, std=0.02, seed=20), rnd(BIG, 1024, seed=21)
    for f in (kernels.gemm_bf16, kernels.gemm_bf16_residual):
        got = [R[:M].clone() for M in (BIG, 3001)]
        for C in got:
            f(A[: len(C)], W, C)
        assert torch.equal(got[0][:3001], got[1]), f.__name__
    W = rnd(8192, K, std=0.02, seed=22)
    act = [torch.empty(M, 4096, dtype=BF, device=dev) for M in (8192, 461)]
    for o in act:
        kernels.gemm_swiglu(A[: len(o)], W, o)
    assert torch.equal(act[0][:461], act[1])


@pytest.mark.parametrize("D", [64, 512, 1088])
def test_short_k_qkv_rows_equal_the_large_tiles(dev, D):
    H, bl, big, rows = 8, 32, 1024, 60
    A, W = rnd(big * bl, D, seed=23), rnd(3 * H * 64, D, std=0.02, seed=24)
    fr = torch.outer(torch.arange(400.0), 10000.0 ** (-torch.arange(0, 64, 2) / 64))
    cos, sin = (torch.cat([f, f], -1).to(BF).float().to(dev) for f in (fr.cos(), fr.sin()))
    pos0 = torch.arange(big, dtype=torch.int32, device=dev) % 77
    table = torch.arange(big * 8, dtype=torch.int32, device=dev).view(big, 8)
    got = []
    for n in (big, rows):
        pool = torch.zeros(big * 8, 2, H, 1024, dtype=BF, device=dev)
        q = torch.empty(n * bl, H * 64, dtype=BF, device=dev)
        kernels.gemm_qkv_rope_kv(A[: n * bl], W, cos, sin, pos0[:n], bl, q, pool, table[:n])
        got.append((q[: rows * bl], pool[: rows * 8]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("epi,which", [("store", "A"), ("store", "W"), ("residual", "A"), ("residual", "W"),
                                       ("swiglu", "A"), ("qkv", "A"), ("head", "W")])  # others take packed rows only
def test_wide_row_pitch(dev, epi, which):
    """Rows of A or W further apart than 32-bit offsets in a tile reach: the same values as a packed call."""
    H, rows, bl, K = 4, 3, 43, 128  # 129 rows: two row tiles, the second of one row
    M, N = rows * bl, {"qkv": 3 * H * 64}.get(epi, 256)
    A, W = rnd(M, K, seed=14), rnd(N, K, std=0.02, seed=15)
    n_wide = M if which == "A" else N
    wide = torch.empty(n_wide, (1 << 22) + 8, dtype=BF, device=dev)[:, :K]
    wide.copy_(A if which == "A" else W)
    table = torch.arange(rows * 4, dtype=torch.int32, device=dev).view(rows, 4)
    pos0 = torch.tensor([0, 5, 16], dtype=torch.int32, device=dev)
    cos, sin = rnd(64, 64, seed=27).float(), rnd(64, 64, seed=28).float()
    got = []
    for a, w in ((A, W), (wide, W) if which == "A" else (A, wide)):
        if epi == "qkv":
            C, pool = torch.empty(M, H * 64, dtype=BF, device=dev), torch.zeros(rows * 4, 2, H, 1024, dtype=BF, device=dev)
            kernels.gemm_qkv_rope_kv(a, w, cos, sin, pos0, bl, C, pool, table)
            got.append((C, pool))
        elif epi == "head":
            C = torch.empty(rows, bl, N, dtype=BF, device=dev)
            kernels.gemm_head_shift(a.view(rows, bl, K), rnd(rows, 1, K, seed=29), w, C)
            got.append((C,))
        else:
            C = rnd(M, N // 2 if epi == "swiglu" else N, seed=30)
            {"store": kernels.gemm_bf16, "residual": kernels.gemm_bf16_residual, "swiglu": kernels.gemm_swiglu}[epi](a, w, C)
            got.append((C,))
    for x, y in zip(*got):
        assert torch.equal(x, y)


@pytest.mark.parametrize("D", [512, 1024, 2048])
@pytest.mark.parametrize("add", [False, True])
def test_rmsnorm_rows_equal_those_of_a_large_call(dev, D, add):
    """One row a workgroup up to 512 rows, one row a wave up to 3072, two above: the same sums per row."""
    x, d, w = rnd(4099, D, seed=16), rnd(4099, D, seed=17), rnd(D, seed=18)
    got = []
    for M in (4099, 3073, 3072, 515, 513, 512, 65, 1):
        r, out = x[:M].clone(), torch.empty(M, D, dtype=BF, device=dev)
        kernels.rmsnorm(r, w, 1e-5, out, delta=d[:M] if add else None)
        got.append((r, out))
    for r, out in got[1:]:
        assert torch.equal(out, got[0][1][: len(out)]) and torch.equal(r, got[0][0][: len(r)])


@pytest.mark.parametrize("N", [1, 2, 63, 64, 65, 255, 257])
def test_few_columns_of_many_rows(dev, N):
    """One 256 x 256 tile per CU and no more columns than a last column tile that is split off holds: the bound of
    test_short_and_odd_k."""
    M, K = 65536, 128
    A, W = rnd(M, K, seed=25), rnd(N, K, std=0.1, seed=26)
    C = torch.full((M, N), float("nan"), dtype=BF, device=dev)
    kernels.gemm_bf16(A, W, C)
    ref = A.double() @ W.double().T
    mag = A.double().abs() @ W.double().abs().T
    assert ((C.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * K * 2.0 ** -24).all()


@pytest.mark.parametrize("epi", ["store", "residual", "swiglu"])
@pytest.mark.parametrize("off,pitch", [(0, 1), (1, 0), (2, 2), (4, 4)])
def test_output_rows_anywhere(dev, epi, off, pitch):
    """C from any element on and with any row pitch, on each tile: the values of a packed call, and nothing beside
    them."""
    N, K = 256, 512
    for M in (3, 100, 257, 1000, 2049, 4100, 9000):
        A, W = rnd(M, K, std=0.5, seed=31), rnd(2 * N if epi == "swiglu" else N, K, std=0.05, seed=32)
        R = rnd(M, N, seed=33)
        f = {"store": kernels.gemm_bf16, "residual": kernels.gemm_bf16_residual, "swiglu": kernels.gemm_swiglu}[epi]
        C = R.clone()
        f(A, W, C)
        ld = N + pitch + off
        wide = torch.full((M * ld + 8,), 7.0, dtype=BF, device=dev)
        out = torch.as_strided(wide, (M, N), (ld, 1), off)
        out.copy_(R)
        f(A, W, out)
        assert torch.equal(out, C), M
        out.fill_(7.0)
        assert (wide == 7.0).all(), M

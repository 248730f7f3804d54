"""The four-deep chain tiles (pk_chain4.h), bit for bit: every tile against the
CPU oracle at the edges of its tiles and chunks, and against the K = 1 chain
kernels where operands hold subnormals, infinities, NaN and signed zeros.
The tile never changes a result, so every comparison is exact."""
import numpy as np
import pytest

import pyoracle as po
from pkgpu import Dev, bits_equal, describe_mismatch, pk

SEED = 0x5EED4400
TILES = range(6)
EPI_RELU = 4                                    # PK_GPU_EPI_RELU
BITS = {"f32": 32, "i8": 8, "i4": 4}


@pytest.fixture(scope="module")
def dev():
    return Dev()


def make(kind, M, N, K, tag):
    lda = (K + 3) // 4 * 4                      # rows stay 16-byte aligned at any K
    A = po.normal((M, lda), 0.0, 1.0, po.seed(SEED, f"{tag}.A"))
    C0 = po.normal((M, N), 0.0, 1.0, po.seed(SEED, f"{tag}.C"))
    if kind == "i4":
        return A, po.bytes_((K, N // 2), po.seed(SEED, f"{tag}.P")), \
            po.uniform((K, N // 32) if N % 32 == 0 else (K * (N // 32) + 1,), 0.005, 0.02,
                       po.seed(SEED, f"{tag}.S")), C0
    if kind == "i8":
        return A, po.int8s((K, N), -127, 127, po.seed(SEED, f"{tag}.Q")), 0.01, C0
    return A, po.normal((K, N), 0.0, 0.02, po.seed(SEED, f"{tag}.W")), None, C0


def run(dev, kind, A, W, extra, C0, K, beta=0.0, bias=None, epi=0, cfg=-1, tile=-1):
    M, N = C0.shape
    a, w, c = dev.put(A), dev.put(W), dev.put(C0)
    s = dev.put(extra) if kind == "i4" else None
    b = dev.put(bias) if bias is not None else None
    prev = pk.load().pk_gpu_get_numerics()
    pk.call("pk_gpu_set_numerics", pk.NUMERICS_EXACT)
    pk.call("pk_gpu_force_config", cfg)
    pk.call("pk_gpu_force_chain_tile", tile)
    try:
        tail = (beta, c.data_ptr(), N, b.data_ptr() if b is not None else None, epi, dev.stream())
        if kind == "i4":
            pk.call("pk_gpu_gemm_i4_ex_dev", M, N, K, 1.0, a.data_ptr(), A.shape[1], w.data_ptr(), s.data_ptr(),
                    N // 2, *tail)
        elif kind == "i8":
            pk.call("pk_gpu_gemm_i8_ex_dev", M, N, K, 1.0, a.data_ptr(), A.shape[1], w.data_ptr(), extra, N, *tail)
        else:
            pk.call("pk_gpu_sgemm_ex_dev", M, N, K, 1.0, a.data_ptr(), A.shape[1], w.data_ptr(), N, *tail)
    finally:
        pk.call("pk_gpu_force_chain_tile", -1)
        pk.call("pk_gpu_force_config", -1)
        pk.call("pk_gpu_set_numerics", prev)
    dev.sync()
    return c.cpu().numpy()


def oracle(kind, A, W, extra, C0, K, beta):
    a = np.ascontiguousarray(A[:, :K])
    if kind == "i4":
        return po.sgemm_q4b(a, W, extra, C0.copy(), 1.0, beta)
    if kind == "i8":
        return po.sgemm_qb(a, W, extra, C0.copy(), 1.0, beta)
    return po.sgemm(a, W, C0.copy(), 1.0, beta)


# rows and columns around the tiles' 16..128 by 32 / 64, K around 4, 16, the
# chunks (32, 64, 128) and pairs of them
SHAPES = [(1, 32, 1), (15, 64, 3), (17, 96, 36), (31, 32, 64), (33, 160, 65), (48, 192, 127), (49, 64, 128),
          (64, 96, 130), (65, 128, 256), (127, 64, 259), (129, 96, 300), (130, 320, 512), (97, 64, 1028)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["f32", "i8", "i4"])
@pytest.mark.parametrize("tile", TILES)
def test_chain_tile_bit_exact(dev, tile, kind):
    for i, (M, N, K) in enumerate(SHAPES):
        A, W, extra, C0 = make(kind, M, N, K, f"{kind}.{M}.{N}.{K}")
        beta = (0.0, 1.0, 0.5)[i % 3]
        got = run(dev, kind, A, W, extra, C0, K, beta, tile=tile)
        want = oracle(kind, A, W, extra, C0, K, beta)
        assert bits_equal(got, want), f"tile {tile} {kind} {M}x{N}x{K}: {describe_mismatch(got, want)}"


@pytest.mark.gpu
@pytest.mark.parametrize("N", [16, 40, 72, 200])
@pytest.mark.parametrize("kind", ["f32", "i8", "i4"])
def test_chain_tile_partial_columns(dev, kind, N):
    """Columns that end inside a tile, and (int8) before the edge columns; every
    epilogue, vector output rows (scalar ones: test_chain_tile_scalar_rows)."""
    bias = po.normal((N,), 0.0, 1.0, po.seed(SEED, f"bias.{N}"))
    for tile in TILES:
        for M, K, epi, beta in ((35, 68, pk.EPI_NONE, 0.0), (19, 132, pk.EPI_SWISH, 0.0),
                                (70, 96, pk.EPI_HALF_RESIDUAL, 0.0), (5, 40, pk.EPI_RESIDUAL, 0.0),
                                (33, 64, EPI_RELU, 1.0)):
            A, W, extra, C0 = make(kind, M, N, K, f"pc.{kind}.{M}.{N}.{K}")
            got = run(dev, kind, A, W, extra, C0, K, beta, bias, epi, tile=tile)
            want = run(dev, kind, A, W, extra, C0, K, beta, bias, epi, cfg=13)
            assert bits_equal(got, want), f"tile {tile} {kind} {M}x{N}x{K}: {describe_mismatch(got, want)}"


def padded(a, ld, rng):
    """a's rows `ld` elements apart, the elements between them at random."""
    out = rng.integers(0, 256, (a.shape[0], ld * a.itemsize), dtype=np.uint8).view(a.dtype).reshape(a.shape[0], ld)
    out[:, :a.shape[1]] = a
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("kind,N", [("f32", 33), ("f32", 37), ("f32", 50), ("i4", 34), ("i4", 44), ("i4", 70),
                                    ("i4", 72), ("i8", 34), ("i8", 48)])
def test_chain_tile_scalar_rows(dev, kind, N):
    """Weight rows padded to whole words, with columns that end inside a unit of
    8 (f32: a part of it lies past the last row's end; i4: not for the four-deep
    tiles, whichever is forced) and output rows that allow no vector stores: an
    odd row stride, C and bias off their alignment by one float.  Every tile and
    the K = 1 kernels against the oracle; nothing beside the columns is written."""
    rng = np.random.default_rng(N)
    guard = np.float32(-7.0)
    for tile, cfg in [(t, -1) for t in TILES] + [(-1, 13), (-1, 20)]:
        for i, (M, K, epi, beta, ldc, off) in enumerate((
                (35, 68, pk.EPI_NONE, 0.5, N + 1, 0), (17, 131, pk.EPI_SWISH, 0.0, N + 3, 1),
                (70, 96, pk.EPI_HALF_RESIDUAL, 0.0, N + 4 - N % 4, 1), (5, 40, pk.EPI_RESIDUAL, 0.0, N + 1, 0),
                (129, 64, EPI_RELU, 1.0, N + 4 - N % 4, 0), (33, 33, pk.EPI_NONE, 1.0, N + 5, 1))):
            A, W, extra, C0 = make(kind, M, N, K, f"sr.{kind}.{M}.{N}.{K}")
            bias = po.normal((N,), 0.0, 1.0, po.seed(SEED, f"sr.bias.{N}")) if i % 2 == 0 or epi else None
            ldb = (W.shape[1] + 3) // 4 * 4 + 4 * (i % 2)
            a, w = dev.put(A), dev.put(padded(W, ldb, rng))
            s = dev.put(extra) if kind == "i4" else None
            c = dev.torch.full((off + M * ldc,), float(guard), device=dev.dev)
            cv = c[off:].view(M, ldc)
            cv[:, :N] = dev.put(C0)
            b = dev.torch.zeros(N + 1, device=dev.dev)
            if bias is not None:
                b[off:off + N] = dev.put(bias)
            pk.call("pk_gpu_set_numerics", pk.NUMERICS_EXACT)
            pk.call("pk_gpu_force_config", cfg)
            pk.call("pk_gpu_force_chain_tile", tile)
            try:
                tail = (beta, cv.data_ptr(), ldc, b[off:].data_ptr() if bias is not None else None, epi, dev.stream())
                if kind == "i4":
                    pk.call("pk_gpu_gemm_i4_ex_dev", M, N, K, 1.0, a.data_ptr(), A.shape[1], w.data_ptr(),
                            s.data_ptr(), ldb, *tail)
                elif kind == "i8":
                    pk.call("pk_gpu_gemm_i8_ex_dev", M, N, K, 1.0, a.data_ptr(), A.shape[1], w.data_ptr(), extra, ldb,
                            *tail)
                else:
                    pk.call("pk_gpu_sgemm_ex_dev", M, N, K, 1.0, a.data_ptr(), A.shape[1], w.data_ptr(), ldb, *tail)
            finally:
                pk.call("pk_gpu_force_chain_tile", -1)
                pk.call("pk_gpu_force_config", -1)
                pk.call("pk_gpu_set_numerics", pk.NUMERICS_DEFAULT)
            dev.sync()
            got = c.cpu().numpy()
            want = oracle(kind, A, W, extra, C0, K, beta)
            if bias is not None:
                want = want + bias
            if epi == pk.EPI_SWISH:
                want = po.swish(want)
            elif epi == pk.EPI_HALF_RESIDUAL:                   # fma: the half is exact
                want = np.float32(0.5) * want + C0
            elif epi == pk.EPI_RESIDUAL:
                want = C0 + want
            elif epi == EPI_RELU:
                want = np.where(want > 0, want, np.float32(0.0))
            rows = got[off:].reshape(M, ldc)
            what = f"tile {tile} config {cfg} {kind} {M}x{N}x{K} ldc {ldc}"
            assert (got[:off] == guard).all() and (rows[:, N:] == guard).all(), what
            cols = np.ascontiguousarray(rows[:, :N])
            assert bits_equal(cols, want), f"{what}: {describe_mismatch(cols, want)}"


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["f32", "i8", "i4"])
def test_chain_tile_special_values(dev, kind):
    """Subnormal products, cancellation, infinities, NaN and signed zeros, as
    the K = 1 kernels give them (chains that end in NaN need not agree in its
    payload)."""
    M, N = 37, 64
    rng = np.random.default_rng(7)
    for K in (3, 64, 131, 262):
        A, W, extra, C0 = make(kind, M, N, K, f"sv.{kind}.{K}")
        A *= np.exp2(rng.integers(-145, 40, A.shape)).astype(np.float32)
        A[rng.random(A.shape) < 0.1] = -0.0
        A[3, :] = -0.0
        A[5, 0], A[6, K - 1], A[7, K // 2] = np.inf, -np.inf, np.nan
        C0[:] = -0.0
        if kind == "i4":
            extra = extra * np.exp2(rng.integers(-140, 100, extra.shape)).astype(np.float32)
            extra[0, 0], extra[K - 1, 1] = np.inf, -extra[K - 1, 1]
        if kind == "f32":
            W *= np.exp2(rng.integers(-100, 60, W.shape)).astype(np.float32)
        for tile in TILES:
            got = run(dev, kind, A, W, extra, C0, K, 1.0, tile=tile)
            want = run(dev, kind, A, W, extra, C0, K, 1.0, cfg=13)
            nan = np.isnan(want)
            assert np.array_equal(np.isnan(got), nan)
            assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan]), f"tile {tile} {kind} K {K}"


def test_chain_tile_choice():
    """The choice is defined over the whole range, takes small tiles for few
    outputs and large ones for many, and every tile is taken somewhere."""
    lib = pk.load()
    assert lib.pk_gpu_num_chain_tiles() == len(TILES)
    taken = set()
    for bits in BITS.values():
        for N in (1, 16, 256, 1024, 2048, 3072, 4096):
            for M in list(range(1, 700, 7)) + [1000, 1656, 2000, 3312, 5000, 204800]:
                for K in (256, 1024, 4096):
                    t = lib.pk_gpu_pick_chain_tile(M, N, K, bits)
                    assert t in TILES
                    taken.add(t)
        assert lib.pk_gpu_pick_chain_tile(16, 1024, 1024, bits) == 0
        assert lib.pk_gpu_pick_chain_tile(3312, 4096, 1024, bits) >= 4
    assert taken == set(TILES)
    # rows of tiles beyond the grid's 65535 leave only taller tiles (K = 1 tiles: 128 rows)
    for M, tile_rows in ((16 * 65535 + 1, 17), (64 * 65535 + 1, 65), (8388480, 128)):
        bm = {0: 16, 1: 32, 2: 48, 3: 64, 4: 64, 5: 128}
        for N in (16, 32, 64):
            assert bm[lib.pk_gpu_pick_chain_tile(M, N, 32, 32)] >= tile_rows
    assert lib.pk_gpu_pick_chain_tile(16, 16, 16, 7) == -1 and lib.pk_gpu_pick_chain_tile(0, 16, 16, 8) == -1
    assert lib.pk_gpu_force_chain_tile(len(TILES)) == -1
    assert lib.pk_gpu_force_chain_tile(-1) == 0


def test_chain_tile_choice_short_chains():
    """Many short chains (K well below 1024) take the 64 x 64 tiles, whose rounds'
    ends overlap: on 32 x 32 ones these take 1.2 to 1.8 times the K = 1 kernels'
    time, on 64 x 64 ones 0.85 to 1.05 times."""
    lib = pk.load()
    for bits in BITS.values():
        for M, N, K in ((204800, 1024, 64), (51200, 1024, 64), (102400, 256, 64), (204800, 256, 128),
                        (204800, 256, 256), (51200, 256, 256), (51200, 1024, 256), (25600, 4096, 256)):
            assert lib.pk_gpu_pick_chain_tile(M, N, K, bits) == 4, (M, N, K, bits)
        for M, N, K in ((3200, 256, 256), (400, 256, 256), (1000, 1024, 256)):
            assert lib.pk_gpu_pick_chain_tile(M, N, K, bits) <= 3, (M, N, K, bits)

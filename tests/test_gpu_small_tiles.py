"""GPU: the encode's small tiles (32 to 160 tokens by 64 to 256 features) against its 256x256 tile.

All tilings run the same MFMA chain per output, so features, row counts and candidate lists agree
bit for bit with the 256x256 tile's, which the parity tests pin and check against the oracle. Shapes end
inside a tile, a K-step, a 16-B chunk and a 32-token block; W_enc is feature-contiguous or
d_in-contiguous, with 16-B aligned rows (LDS DMA) or rows of odd length (staged through
registers)."""

import pytest
import torch

from saeflow_amd.kernels import encode_gather, encode_pre, encode_rows, fused_encode

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]
TILES = [(32, 64, 2), (128, 64, 4), (128, 128, 4), (32, 128, 4), (64, 128, 4), (160, 256, 4)]
# (tokens, d_in, d_sae): one of everything; exact tiles; remainders on every axis; a long K loop
SHAPES = [(1, 1, 1), (32, 64, 64), (33, 40, 72), (95, 200, 264), (97, 72, 1000), (128, 128, 128), (129, 16, 136),
          (300, 777, 520), (5, 2304, 4096), (257, 1024, 328)]


def config(tile, dtype):
    tm, tn, nw = tile
    bk = (32 if dtype == torch.float32 else 64) // (2 if (tm, tn) == (128, 128) else 1)
    return {"BLOCK_M": tm, "BLOCK_N": tn, "BLOCK_K": bk, "GROUP_M": 1, "NUM_WAVES": nw, "GROUP_N": 4}


def wide(dtype):
    return {"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": 32 if dtype == torch.float32 else 64}


def make(shape, dtype, layout, nan=False):
    M, K, N = shape
    g = torch.Generator().manual_seed(M * 7 + K * 3 + N)
    W = (torch.randn(K, N, generator=g) / K ** 0.5).to(dtype).cuda()
    if layout == "features":
        pass
    elif layout == "d_in":  # rows padded to 16 B, as an aligned transposed view has them, with anything
        back = torch.full((N, -(-K // 8) * 8), float("nan"), dtype=dtype, device="cuda")
        back[:, :K] = W.T
        W = back.T[:K]
    elif layout == "odd_features":  # rows of odd length
        back = torch.zeros(K, N | 1, dtype=dtype, device="cuda")
        back[:, :N] = W
        W = back[:, :N]
    else:
        back = torch.zeros(N, K | 1, dtype=dtype, device="cuda")
        back[:, :K] = W.T
        W = back[:, :K].T
    x = torch.randn(M, K, generator=g)
    if nan:
        x[M // 2] = float("nan")
    cut = torch.rand(N, generator=g) * 0.5
    vec = dict(b_enc=torch.randn(N, generator=g) * 0.1, b_dec=torch.randn(K, generator=g) * 0.1)
    return x.to(dtype).cuda(), W, {k: v.to(dtype).cuda() for k, v in vec.items()}, cut.to(dtype).cuda()


def aligned(shape, dtype, layout):
    """Whether this W takes the DMA paths (the rows of the 256-feature tiles are not staged otherwise)."""
    M, K, N = shape
    if layout == "features":
        return N % (4 if dtype == torch.float32 else 8) == 0
    return layout == "d_in" and K % (4 if dtype == torch.float32 else 8) == 0


def same(a, b):
    bits = {4: torch.int32, 2: torch.int16}[a.element_size()]
    return torch.equal(a.view(bits), b.view(bits))


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("layout", ["features", "d_in", "odd_features", "odd_d_in"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_small_tiles_equal_the_wide_tile(dtype, layout, tile):
    for shape in SHAPES:
        if tile[1] == 256 and not aligned(shape, dtype, layout):
            x, W, p, _ = make(shape, dtype, layout)
            with pytest.raises(ValueError, match="16-B aligned rows"):
                fused_encode(x, W, p["b_enc"], p["b_dec"], config=config(tile, dtype))
            continue
        x, W, p, cut = make(shape, dtype, layout, nan=shape[0] > 100)
        M = shape[0]
        for act, out_dtype in (("jumprelu", None), ("relu", torch.float32)):
            counts = [torch.zeros(M, dtype=torch.int32, device="cuda") for _ in range(2)]
            got, want = (fused_encode(x, W, p["b_enc"], p["b_dec"], cut, act, out_dtype=out_dtype, row_nnz=n, config=c)
                         for n, c in zip(counts, (config(tile, dtype), wide(dtype))))
            assert same(got, want), (shape, act)
            assert torch.equal(*counts), (shape, act)
        got, want = (encode_pre(x, W, p["b_enc"], p["b_dec"], config=c) for c in (config(tile, dtype), wide(dtype)))
        assert same(got, want), shape


@pytest.mark.parametrize("d_in", [1001, 1002, 1004, 1006, 70, 9])
@pytest.mark.parametrize("dtype", DTYPES)
def test_padding_behind_d_in_stays_out_of_the_features(dtype, d_in):
    """A d_in-contiguous W_enc with 16-B aligned rows that end inside a chunk, NaN behind them: the
    features are those of the dense weight on every path."""
    M, N = 130, 300
    x, W, p, cut = make((M, d_in, N), dtype, "features")
    padded = make((M, d_in, N), dtype, "d_in")[1]
    assert torch.equal(padded, W) and padded.stride(0) == 1 and padded.stride(1) % 8 == 0
    want = fused_encode(x, W, p["b_enc"], p["b_dec"], cut, "jumprelu", config=wide(dtype))
    assert not want.isnan().any()
    bk = wide(dtype)["BLOCK_K"]
    for c in (None, wide(dtype), {**wide(dtype), "NUM_WAVES": 4}, config(TILES[0], dtype),
              {"BLOCK_M": 256, "BLOCK_N": 128, "BLOCK_K": bk // 2}):
        assert same(fused_encode(x, padded, p["b_enc"], p["b_dec"], cut, "jumprelu", config=c), want), c
    rows, n = torch.arange(M, dtype=torch.int32, device="cuda"), torch.full((1,), M, dtype=torch.int32, device="cuda")
    assert same(encode_gather(x, padded, p["b_enc"], p["b_dec"], rows, n, cut, "jumprelu", out_rows=M), want)
    for c in (None, wide(dtype)):
        cnt, idx, val = encode_rows(x, padded, p["b_enc"], p["b_dec"], cut, "jumprelu", cap=N, config=c)
        live = torch.arange(N, device="cuda")[None] < cnt[:, None]
        f = torch.zeros(M, N + 1, dtype=dtype, device="cuda")
        f.scatter_(1, torch.where(live, idx, N).long(), val)
        assert same(f[:, :N].contiguous(), want), c


def test_rows_of_w_enc_megabytes_apart():
    """A view of d_in 8 into rows of 4 MB and more, NaN behind it: a tile's 256 features span over 1 GiB, the
    offset that stands for out of range in the DMA path."""
    M, K, N, pitch = 40, 8, 300, (1 << 21) + (1 << 15)
    back = torch.full((N, pitch), float("nan"), dtype=torch.bfloat16, device="cuda")
    x, W, p, _ = make((M, K, N), torch.bfloat16, "features")
    back[:, :K] = W.T
    want = fused_encode(x, W, p["b_enc"], p["b_dec"], config=wide(torch.bfloat16))
    for c in (None, wide(torch.bfloat16), config((32, 64, 2), torch.bfloat16)):
        assert same(fused_encode(x, back[:, :K].T, p["b_enc"], p["b_dec"], config=c), want), c


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("layout", ["features", "odd_features"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_small_tile_row_candidates_equal_the_wide_tiles(dtype, layout, tile):
    for shape in SHAPES:
        if tile[1] == 256 and not aligned(shape, dtype, layout):
            continue
        x, W, p, cut = make(shape, dtype, layout, nan=shape[0] > 100)
        for act, floor in (("jumprelu", None), ("relu", torch.rand(shape[0], device="cuda")),
                           ("relu", torch.full((shape[0],), -1.0, device="cuda"))):
            cap = shape[2] // 3 if floor is None else shape[2]  # some lists overflow
            lists = []
            for c in (config(tile, dtype), wide(dtype)):
                cnt, idx, val = encode_rows(x, W, p["b_enc"], p["b_dec"], cut, act, cap=cap, row_floor=floor, config=c)
                col = torch.arange(cap, device="cuda")[None]
                dead = col >= cnt[:, None]
                order = idx.masked_fill(dead, 1 << 30).sort(dim=1).indices
                bits = val.view({4: torch.int32, 2: torch.int16}[val.element_size()]).to(torch.int64).masked_fill(dead, 0)
                lists.append((cnt, idx.masked_fill(dead, 0).gather(1, order), bits.gather(1, order), cnt > cap))
            (c0, i0, b0, o0), (c1, i1, b1, _) = lists
            assert torch.equal(c0, c1), (shape, act)
            ok = ~o0[:, None]  # an overflowed list holds any cap of the kept values
            assert torch.equal(i0 * ok, i1 * ok) and torch.equal(b0 * ok, b1 * ok), (shape, act)


def test_small_tiles_refuse_a_doubly_strided_weight():
    x, W, p, _ = make((40, 64, 128), torch.bfloat16, "features")
    W = W.repeat_interleave(2, 0).repeat_interleave(2, 1)[::2, ::2]
    with pytest.raises(ValueError, match="contiguous along one axis"):
        fused_encode(x, W, p["b_enc"], p["b_dec"], config=config(TILES[0], torch.bfloat16))
    assert same(fused_encode(x, W, p["b_enc"], p["b_dec"]), fused_encode(x, W.contiguous(), p["b_enc"], p["b_dec"]))


def test_small_tiles_write_a_strided_output_row_in_place():
    """Output rows that are no 16-B multiple take the element stores: the padding stays as it was."""
    from saeflow_amd import _lib
    lib = _lib.load()
    M, K, N = 70, 96, 203
    x, W, p, _ = make((M, K, N), torch.bfloat16, "odd_features")
    want = fused_encode(x, W, p["b_enc"], p["b_dec"], config=wide(torch.bfloat16))
    out = torch.full((M, N + 6), 7.0, dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    _lib.check(lib.sf_encode(_lib.ptr(x), K, 1, 1, _lib.ptr(W), W.stride(0), 1, 1, _lib.ptr(p["b_enc"]), 1,
                             _lib.ptr(p["b_dec"]), 1, None, 0, _lib.ptr(out), N + 6, 1, 1, None, M, N, K, 0, None,
                             _lib.ptr(ws), ws.numel(), _lib.stream(x.device)))
    assert same(out[:, :N].contiguous(), want) and bool((out[:, N:] == 7.0).all())


def test_a_tuned_small_tile_is_reported_and_reproduced_by_its_config():
    """best_config() after a timed call names what the call keeps, for W_enc rows off 16 B (the small
    tiles stage those at several times the rate of the others) and on 16 B, which are tuned apart
    although shape and strides agree."""
    from saeflow_amd.kernels import best_config
    from saeflow_amd.kernels import encode as kenc
    M, K, N, dtype = 1024, 2304, 16384, torch.bfloat16
    assert 2 * M * N * K >= kenc.AUTOTUNE_MIN_FLOPS
    x, big, p, _ = make((M, K, N + 8), dtype, "features")
    be = p["b_enc"][:N]
    saved = dict(kenc._tuned)
    kenc._tuned.clear()
    try:
        f = fused_encode(x, big[:, :N], be, p["b_dec"])
        assert best_config() in kenc._candidates(dtype) or best_config()["BLOCK_M"] < 256
        g = fused_encode(x, big[:, 1:N + 1], be, p["b_dec"])
        picked = best_config()
        assert len(kenc._tuned) == 2 and picked["BLOCK_M"] < 256
        assert picked == kenc._default_tiling(M, N, K, big[:, 1:N + 1])
        assert same(fused_encode(x, big[:, 1:N + 1], be, p["b_dec"], config=picked), g)
        fused_encode(x, big[:, :N], be, p["b_dec"])
        assert best_config() == next(iter(kenc._tuned.values()))  # a shape tuned before keeps its own pick
        assert same(f, fused_encode(x, big[:, :N].contiguous(), be, p["b_dec"], config=wide(dtype)))
    finally:
        kenc._tuned.clear()
        kenc._tuned.update(saved)

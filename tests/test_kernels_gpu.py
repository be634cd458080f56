"""Parity of every HIP kernel, called through the C ABI, with the CPU oracle.

Same seeded inputs on both sides; bf16 outputs within rtol 1e-2 / atol 1e-2 of the
oracle's (f32 accumulation, one rounding), exact for the data movers and the draw.
"""

import math

import numpy as np
import pytest
import torch

from iron_amd import _lib, kernels as K
from iron_amd.bf16 import from_torch, round_bf16, to_torch
from oracle import ops

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-2, 1e-2


def bf(rng, *shape, scale=1.0):
    return round_bf16(rng.standard_normal(shape, dtype=np.float32) * np.float32(scale))


def dev(x, cuda):
    return to_torch(x).to(cuda)


def out_like(shape, cuda, fill=None):
    t = torch.empty(shape, dtype=torch.bfloat16, device=cuda)
    if fill is not None:
        t.fill_(fill)
    return t


def word(v, cuda):
    return torch.tensor([v], dtype=torch.int32, device=cuda)


def close(got, want, rtol=RTOL, atol=ATOL, frac=0.0):
    got = from_torch(got).reshape(np.shape(want)) if isinstance(got, torch.Tensor) else got
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    bad = ~(err <= atol + rtol * np.abs(want))
    assert bad.mean() <= frac, (
        f"{bad.sum()}/{bad.size} outside rtol {rtol} atol {atol}; max err {np.nanmax(err):.5f} "
        f"at {np.unravel_index(np.nanargmax(err), err.shape)}"
    )


# ------------------------------------------------------------------------ GEMV
@pytest.mark.parametrize("Kdim,N", [(2048, 2048), (2048, 512), (2048, 8192), (8192, 2048), (2048, 128256)])
def test_gemv_decode_sweep(cuda, Kdim, N):
    rng = np.random.default_rng(42)
    W, x = bf(rng, N, Kdim, scale=0.02), bf(rng, Kdim)
    y = out_like((N,), cuda)
    K.gemv(dev(W, cuda), dev(x, cuda), y, M=N, K=Kdim)
    close(y, ops.gemv(W, x))


@pytest.mark.parametrize("rpw,ks", [(1, 1), (1, 2), (1, 4), (2, 1), (2, 2), (2, 4), (4, 1), (4, 2), (4, 4), (8, 1)])
def test_gemv_every_launch_shape_and_ragged_rows(cuda, rpw, ks):
    rng = np.random.default_rng(1)
    M, Kdim = 77, 1096  # rows not a multiple of any block, K not a multiple of 512
    W, x = bf(rng, M, Kdim), bf(rng, Kdim)
    y = out_like((M,), cuda)
    K.gemv(dev(W, cuda), dev(x, cuda), y, M=M, K=Kdim, rows_per_wave=rpw, k_split=ks)
    close(y, ops.gemv(W, x), rtol=1e-2, atol=3e-2)


def test_gemv_batches_repeat_and_bound(cuda):
    rng = np.random.default_rng(2)
    # Llama decode's scores shape: 32 heads over 8 groups (gemv.py:51).
    W, x = bf(rng, 8, 256, 64), bf(rng, 32, 64)
    y = out_like((32, 256), cuda)
    K.gemv(dev(W, cuda), dev(x, cuda), y, M=256, K=64, batches=32, repeat=4)
    close(y, ops.gemv(W, x, repeat=4))
    # A bound on the rows: rows past it are left as they were.
    W, x = bf(rng, 300, 128), bf(rng, 128)
    y = out_like((300,), cuda, fill=7.0)
    K.gemv(dev(W, cuda), dev(x, cuda), y, M=300, K=128, valid=word(123, cuda))
    got = from_torch(y)
    close(got[:123], ops.gemv(W, x)[:123])
    assert np.all(got[123:] == 7.0)


# ------------------------------------------------------------------------ GEMM
@pytest.mark.parametrize("M,Kdim,N", [(5, 648, 8), (33, 264, 72), (97, 192, 136), (130, 1096, 600), (1003, 584, 640), (70, 520, 24)])
def test_gemm_turned_over_small_tiles(cuda, M, Kdim, N):
    """B (K,N) into C (N,M), less than a round of tiles of 32 and of 64 rows: edges of both, ragged K, nothing beyond C."""
    rng = np.random.default_rng(M + N)
    A, B = bf(rng, M, Kdim), bf(rng, Kdim, N, scale=0.05)
    C = out_like((N * M + 64,), cuda, fill=3.0)
    K.gemm(dev(A, cuda), dev(B, cuda), C[: N * M].view(N, M), M=M, N=N, K=Kdim, c_col_maj=True)
    got = from_torch(C)
    assert np.all(np.abs(got[: N * M].reshape(N, M).T - ops.gemm(A, B)) <= ops.gemm_bound(A, B)) and np.all(got[N * M :] == 3.0)


@pytest.mark.parametrize("b_col_maj", [False, True])
@pytest.mark.parametrize("c_col_maj", [False, True])
def test_gemm_layouts(cuda, b_col_maj, c_col_maj):
    rng = np.random.default_rng(3)
    M, Kdim, N = 384, 512, 640
    A, B = bf(rng, M, Kdim), bf(rng, (N if b_col_maj else Kdim), (Kdim if b_col_maj else N), scale=0.05)
    C = out_like((N, M) if c_col_maj else (M, N), cuda)
    K.gemm(dev(A, cuda), dev(B, cuda), C, M=M, N=N, K=Kdim, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    want = ops.gemm(A, B, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    close(C, want)
    # And by the reference's own bound: 2 units of 2^-8 |A|@|B| (gemm.py:704-735).
    bound = ops.gemm_bound(A, B, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    assert np.all(np.abs(from_torch(C) - want) <= bound)


def test_native_calls_refuse_what_the_long_way_refuses_and_follow_the_stream(cuda):
    """What the one-call shortcut is not for -- another dtype, strides, count, a refused size -- raises as the long way does; a call inside a
    stream's block runs on that stream, behind what was queued there."""
    x = torch.zeros(64, 64, dtype=torch.bfloat16, device=cuda)
    for bad, error in ((x.float(), TypeError), (x.t()[:, :32], ValueError), (x[:32], ValueError), (torch.zeros(64, 64, dtype=torch.bfloat16), TypeError)):
        with pytest.raises(error):
            K.gemm(x, bad, x.clone(), M=64, N=64, K=64)
        with pytest.raises(error):
            K.mha_prefill(x, bad, x, x.clone(), heads=1, kv_heads=1, d=64, seq=64, kv_len=64)
    with pytest.raises(_lib.IronHipError, match="iron_gemm_bf16 refused.*multiple of 8"):
        K.gemm(x.view(-1)[: 64 * 63], x.view(-1)[: 64 * 63], x.clone(), M=64, N=64, K=63)
    with pytest.raises(_lib.IronHipError, match="refused"):
        K.gemv(x.view(-1)[: 64 * 63], x.view(-1)[:63], x.view(-1)[:64].clone(), M=64, K=63)
    big, one, side = torch.randn(4096, 4096, device=cuda), torch.ones(64, 64, dtype=torch.bfloat16, device=cuda), torch.cuda.Stream()
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(8):
            big = big @ big * 1e-3
        late = one + big[0, 0].to(torch.bfloat16) * 0
        K.gemm(late, one, y, M=64, N=64, K=64)
        out = y.clone()
    side.synchronize()
    assert bool((out == 64).all())


def test_the_native_calls_and_the_long_way_are_the_same_launches(cuda, monkeypatch):
    """A product alone, one whose tiles are shared, a matrix-vector product and prompt attention, with the native calls and without: the same bits."""
    rng = np.random.default_rng(17)
    x = {n: dev(bf(rng, n), cuda) for n in (64 * 8192, 192 * 384, 384 * 64, 8192, 300 * 4 * 64)}

    def run():
        outs = [out_like((64, 64), cuda, fill=5.0), out_like((192, 64), cuda, fill=5.0), out_like((64,), cuda, fill=5.0), out_like((300 * 4 * 64,), cuda, fill=5.0)]
        K.gemm(x[64 * 8192], x[64 * 8192], outs[0], M=64, N=64, K=8192, b_col_maj=True)
        K.gemm(x[192 * 384], x[384 * 64], outs[1], M=192, N=64, K=384)
        K.gemv(x[64 * 8192], x[8192], outs[2], M=64, K=8192)
        K.mha_prefill(*(x[300 * 4 * 64],) * 3, outs[3], heads=4, kv_heads=4, d=64, seq=300, kv_len=300)
        return outs

    assert _lib.native().__name__ == "iron_amd._calls"
    native = run()
    monkeypatch.setattr(K, "native", lambda: _lib._LongWay)
    assert all(torch.equal(a, b) and not bool((a == 5).all()) for a, b in zip(native, run()))


@pytest.mark.parametrize("b_col_maj", [False, True])
@pytest.mark.parametrize("c_col_maj", [False, True])
@pytest.mark.parametrize("M,Kdim,N", [
    (64, 64, 128), (65, 72, 136), (40, 120, 200), (129, 136, 248), (191, 1000, 264), (333, 72, 1000),   # 64 and 128 tiles
    (2049, 200, 1160), (3500, 72, 3400), (3584, 248, 3584), (3329, 128, 3592), (16384, 72, 40),          # ... and 256 ones
])
def test_gemm_at_the_edges_of_tiles_and_stages(cuda, M, Kdim, N, b_col_maj, c_col_maj):
    """A K that ends inside a stage (one piece over it, one piece short, alone in its second stage), edges
    that move the last tile back, one row or column group more than a tile, in every layout.  The
    operands lie between NaNs: a piece read from outside them would show in the sums."""
    rng = np.random.default_rng(M + N + Kdim)
    A, B = bf(rng, M, Kdim), bf(rng, (N if b_col_maj else Kdim), (Kdim if b_col_maj else N), scale=0.05)

    def between_nans(x):
        room = 64 * max(x.shape)
        buf = torch.full((x.size + 2 * room,), float("nan"), dtype=torch.bfloat16, device=cuda)
        inside = buf[room:room + x.size].view(*x.shape)
        inside.copy_(dev(x, cuda))
        return inside

    C = out_like((N, M) if c_col_maj else (M, N), cuda, fill=float("nan"))
    K.gemm(between_nans(A), between_nans(B), C, M=M, N=N, K=Kdim, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    want = ops.gemm(A, B, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    # The bound the layouts are held to above: 2 units of 2^-8 |A|@|B|.
    assert np.all(np.abs(from_torch(C) - want) <= ops.gemm_bound(A, B, b_col_maj=b_col_maj, c_col_maj=c_col_maj))


@pytest.mark.parametrize("M,Kdim,N,b_col_maj,c_col_maj", [
    (64, 200, 16384, False, False), (33, 264, 16264, False, False), (16384, 192, 64, False, True), (16321, 264, 40, False, False), (16384, 200, 32, True, False),
    (31, 1096, 16383, True, True)])
def test_gemm_small_tiles_of_one_whole_round(cuda, M, Kdim, N, b_col_maj, c_col_maj):
    """As many small tiles as there are CUs, a row or a column of tiles long: 128 tiles of 128 x 128 would be half empty."""
    assert K.lib().iron_gemm_tile(0, M, N, Kdim, b_col_maj, c_col_maj, 0) >> 16 in (32, 64)
    test_gemm_at_the_edges_of_tiles_and_stages(cuda, M, Kdim, N, b_col_maj, c_col_maj)


# tiles 14 x 24 and 17 x 21 of 128 x 128 (19 x 16 without a band left over), 17 x 24 of 256 x 256, 24 x 16 and 29 x 13 of 64 x 64
@pytest.mark.parametrize("M,Kdim,N,b_col_maj,c_col_maj", [
    (1700, 136, 3000, False, True), (2050, 72, 2600, False, True), (2400, 64, 2048, False, True), (4100, 64, 6000, True, False), (1536, 192, 1000, True, False),
    (1850, 136, 780, True, False)])
def test_gemm_of_more_than_a_round_of_tiles_by_columns(cuda, M, Kdim, N, b_col_maj, c_col_maj):
    """Twelve rows of tiles and more, and more of them than a round: an XCD's tiles go by bands of columns, each tile computed and none left out."""
    code = K.lib().iron_gemm_tile(0, M, N, Kdim, b_col_maj, c_col_maj, 0)
    rows, cols = -(-M // (code >> 16)), -(-N // (code & 65535))
    assert rows >= 12 and rows * cols > 288
    test_gemm_at_the_edges_of_tiles_and_stages(cuda, M, Kdim, N, b_col_maj, c_col_maj)


@pytest.mark.parametrize("M,Kdim,N,b_col_maj,c_col_maj", [
    (3329, 128, 3593, True, False), (3329, 192, 3592, False, False),                                   # 256 x 256 tiles
    (192, 136, 48000, True, False), (3840, 264, 2819, True, False), (1290, 200, 8200, False, False),   # 192 x 256
    (160, 200, 40963, True, False), (1025, 64, 7169, True, False), (1025, 72, 7176, False, False),     # 160 x 256
    (641, 264, 8067, True, False), (777, 64, 6915, True, False), (641, 136, 5384, False, False),       # 128 x 256
    (128, 328, 33000, True, False), (641, 64, 5377, True, False), (3585, 200, 1025, True, True),       # 128 x 192
])
def test_gemm_large_tiles_of_every_size(cuda, M, Kdim, N, b_col_maj, c_col_maj):
    """Each size of tile a launch without a row bound may take, down to one tile row, one stage of K and a K that ends inside
    one, the last tiles moved back to the edges; the operands lie between NaNs.  B (N,K): the bits of the launch under a bound, whose
    tiles are of other sizes."""
    rng = np.random.default_rng(M + N + Kdim)
    A, B = bf(rng, M, Kdim), bf(rng, (N if b_col_maj else Kdim), (Kdim if b_col_maj else N), scale=0.05)

    def between_nans(x):
        buf = torch.full((x.size + 256 * x.shape[1],), float("nan"), dtype=torch.bfloat16, device=cuda)
        inside = buf[128 * x.shape[1]:128 * x.shape[1] + x.size].view(*x.shape)
        inside.copy_(dev(x, cuda))
        return inside

    dA, dB, buf = between_nans(A), between_nans(B), out_like((M * N + 64,), cuda, fill=3.0)
    C = buf[: M * N].view(*((N, M) if c_col_maj else (M, N)))
    K.gemm(dA, dB, C, M=M, N=N, K=Kdim, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    kw = dict(b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    assert np.all(np.abs(from_torch(C) - ops.gemm(A, B, **kw)) <= ops.gemm_bound(A, B, **kw))
    assert bool((buf[M * N:] == 3).all())
    if b_col_maj and not c_col_maj:
        bounded = torch.empty_like(C)
        K.gemm(dA, dB, bounded, M=M, N=N, K=Kdim, b_col_maj=True, valid=word(M, cuda))
        assert torch.equal(bounded, C)


@pytest.mark.parametrize("M,Kdim,N,b_col_maj,c_col_maj", [
    (64, 8192, 64, True, False), (24, 6200, 200, True, False), (63, 8184, 136, True, True), (67, 3640, 872, True, False), (872, 3640, 67, True, True),   # all tiles shared, B (N,K)
    (1, 4096, 400, False, False), (130, 2504, 72, False, False), (257, 4000, 264, False, False),   # ... and (K,N)
    (123, 2856, 200, False, True), (2049, 2504, 2056, True, False), (2049, 2504, 2056, False, False),   # (N,M); the last round's tiles
])
def test_gemm_whose_tiles_are_shared(cuda, M, Kdim, N, b_col_maj, c_col_maj):
    """Products whose tiles' K is dealt over several blocks, over a workspace of NaNs: against the oracle by the
    layouts' bound, and the same bits from a recorded graph's replays, whatever ran in between."""
    assert K._gemm_workspace(M, N, Kdim, b_col_maj, c_col_maj) > 0
    rng = np.random.default_rng(M + N + Kdim)
    A, B = bf(rng, M, Kdim), bf(rng, (N if b_col_maj else Kdim), (Kdim if b_col_maj else N), scale=0.05)
    dA, dB = dev(A, cuda), dev(B, cuda)
    kw = dict(M=M, N=N, K=Kdim, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    torch.full((32 << 20,), 255, dtype=torch.uint8, device=cuda)   # what the allocator hands out next is bf16 and float32 NaN
    C = out_like((N, M) if c_col_maj else (M, N), cuda, fill=float("nan"))
    K.gemm(dA, dB, C, **kw)
    want = ops.gemm(A, B, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    assert np.all(np.abs(from_torch(C) - want) <= ops.gemm_bound(A, B, b_col_maj=b_col_maj, c_col_maj=c_col_maj))
    again = torch.zeros_like(C)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        K.gemm(dA, dB, again, **kw)
        K.gemm(dA, dB, again, **kw)
    for _ in range(3):
        again.fill_(7.0)
        K.gemm(dA, dB, torch.empty_like(C), **kw)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(again, C)


def test_gemm_that_shares_no_tiles_is_refused_a_workspace(cuda):
    """Whole rounds, or too short a K: no workspace, and the shared entry point refuses before any launch."""
    for M, N, Kdim, b, c in ((2048, 2048, 2048, 0, 0), (1024, 1024, 1024, 1, 0), (64, 64, 56, 1, 0), (64, 64, 12, 1, 0), (16, 4096, 8192, 1, 0)):
        assert K.lib().iron_gemm_workspace_bytes(M, N, Kdim, b, c) == 0
    t = out_like((1024 * 1024,), cuda, fill=0.0)
    assert K.lib().iron_gemm_shared_bf16(t.data_ptr(), t.data_ptr(), t.data_ptr(), 1024, 1024, 1024, 1, 0, t.data_ptr(), 0) == 1


# Few rows by long stages, as (N,M) output too; 600 and more by tiles of 96.
@pytest.mark.parametrize("M,N,Kdim,b_col_maj,c_col_maj", [(25, 364, 5632, 1, 0), (2199, 31, 8000, 1, 1), (8603, 615, 6464, 1, 0), (617, 8242, 4480, 1, 1)])
def test_gemm_that_another_form_made_cheaper_than_shared_tiles_takes_a_workspace_all_the_same(cuda, M, N, Kdim, b_col_maj, c_col_maj):
    """A caller with a workspace of its own size is not refused what shared its tiles before those forms came: it is made by them, and the workspace left alone."""
    assert K.lib().iron_gemm_workspace_bytes(M, N, Kdim, b_col_maj, c_col_maj) == 0
    rng = np.random.default_rng(M)
    A, B, ws = dev(bf(rng, M, Kdim), cuda), dev(bf(rng, N, Kdim, scale=0.05), cuda), out_like((8,), cuda, fill=5.0)
    C = out_like((N, M) if c_col_maj else (M, N), cuda, fill=float("nan"))
    assert K.lib().iron_gemm_shared_bf16(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, Kdim, b_col_maj, c_col_maj, ws.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    want = torch.empty_like(C)
    K.gemm(A, B, want, M=M, N=N, K=Kdim, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    assert torch.equal(C, want) and bool((ws == 5).all())


@pytest.mark.parametrize("b_col_maj", [True, False])
@pytest.mark.parametrize("n", [4096, 8192])
def test_gemm_large_squares_on_sampled_rows(cuda, n, b_col_maj):
    """The 256 x 256-tile kernel at the benchmark's large squares, B as (N, K) and as (K, N): a sample
    of rows (tile edges and random ones) of the product against float64 dot products, and nothing
    left unwritten."""
    rng = np.random.default_rng(n)
    A, B = bf(rng, n, n, scale=0.02), bf(rng, n, n, scale=0.02)   # B is (N, K) or (K, N) as the flag says
    C = out_like((n, n), cuda, fill=float("nan"))
    K.gemm(dev(A, cuda), dev(B, cuda), C, M=n, N=n, K=n, b_col_maj=b_col_maj)
    got = from_torch(C)
    assert not np.isnan(got).any()
    rows = sorted({0, 1, 127, 128, 255, 256, 257, n // 2 - 1, n // 2, n - 256, n - 1, *rng.integers(0, n, 21).tolist()})
    Bd = B.astype(np.float64)
    want = round_bf16((A[rows].astype(np.float64) @ (Bd.T if b_col_maj else Bd)).astype(np.float32))
    close(got[rows], want, rtol=1e-2, atol=1e-3)


@pytest.mark.parametrize("M,Kdim,N", [(2048, 192, 6144), (4096, 64, 3072), (3072, 1152, 4096)])
def test_gemm_large_tiles_with_b_as_stored_by_default(cuda, M, Kdim, N):
    """B (K, N) through the 256 x 256 tiles and the 192 x 256 ones: one stage, three, and
    eighteen of them, every element against the oracle."""
    rng = np.random.default_rng(M + N + Kdim)
    A, B = bf(rng, M, Kdim), bf(rng, Kdim, N)
    C = out_like((M, N), cuda, fill=float("nan"))
    K.gemm(dev(A, cuda), dev(B, cuda), C, M=M, N=N, K=Kdim)
    close(C, ops.gemm(A, B))


def test_gemm_headline_shape(cuda):
    rng = np.random.default_rng(4)
    A, B = bf(rng, 2048, 2048, scale=0.02), bf(rng, 2048, 2048, scale=0.02)
    C = out_like((2048, 2048), cuda)
    K.gemm(dev(A, cuda), dev(B, cuda), C, M=2048, N=2048, K=2048)
    close(C, ops.gemm(A, B), rtol=1e-2, atol=1e-3)
    Bt = np.ascontiguousarray(B.T)
    K.gemm(dev(A, cuda), dev(Bt, cuda), C, M=2048, N=2048, K=2048, b_col_maj=True)
    close(C, ops.gemm(A, B), rtol=1e-2, atol=1e-3)


@pytest.mark.parametrize("M,Kdim,N", [(100, 136, 72), (32, 1152, 2048), (1, 64, 8), (130, 8, 264), (2048, 2048, 512), (192, 8192, 128)])
@pytest.mark.parametrize("b_col_maj", [False, True])
def test_gemm_ragged_shapes(cuda, M, Kdim, N, b_col_maj):
    rng = np.random.default_rng(5)
    A, B = bf(rng, M, Kdim), bf(rng, (N if b_col_maj else Kdim), (Kdim if b_col_maj else N), scale=0.1)
    C = out_like((M, N), cuda)
    K.gemm(dev(A, cuda), dev(B, cuda), C, M=M, N=N, K=Kdim, b_col_maj=b_col_maj)
    close(C, ops.gemm(A, B, b_col_maj=b_col_maj), rtol=1e-2, atol=2e-2)


@pytest.mark.parametrize("M,Kdim,N,rows", [(2048, 512, 8192, None), (2048, 64, 6144, None), (4096, 192, 4096, 1000), (4096, 192, 4096, 3000), (2048, 128, 2048, 512), (2048, 128, 2048, 1500), (2048, 192, 512, 700),
                                           (128, 64, 128, None), (256, 128, 192, None)])
def test_gemm_weight_layout_fast_paths(cuda, M, Kdim, N, rows):
    """B (N,K): tiles from 64 x 64 to 256 x 256, down to a single k stage, with a row bound that cuts
    through a tile."""
    rng = np.random.default_rng(55)
    A, B = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.1)
    want = ops.gemm(A, B, b_col_maj=True)
    if rows is not None:
        A[rows:] = np.nan
    C = out_like((M, N), cuda, fill=5.0)
    K.gemm(dev(A, cuda), dev(B, cuda), C, M=M, N=N, K=Kdim, b_col_maj=True,
           valid=None if rows is None else word(rows, cuda))
    got = from_torch(C)
    lim = M if rows is None else rows
    close(got[:lim], want[:lim], rtol=1e-2, atol=2e-2)
    assert np.all(got[lim:] == 5.0)


# (the first eight: tiles of 32 or 64 columns by 32 and by 64 rows, a single round of them and one tile, K of three stages and more, whole and ragged)
@pytest.mark.parametrize("M,Kdim,N", [(97, 192, 65), (65, 200, 2042), (510, 1096, 333), (1000, 576, 509), (33, 4160, 2000), (129, 2344, 1364), (1000, 584, 640), (70, 264, 24),
                                       (130, 128, 264), (200, 192, 136), (1000, 256, 1000), (65, 64, 65), (2047, 320, 2050), (333, 128, 384)])
@pytest.mark.parametrize("b_col_maj", [False, True])
def test_gemm_direct_to_lds_tiles_at_ragged_edges(cuda, M, Kdim, N, b_col_maj):
    """K a multiple of 64 takes the direct-to-LDS tiles whatever M and N are: rows and columns past
    the edge are clamped on the way in and never stored, and nothing beyond C is touched."""
    if not b_col_maj:
        N = (N + 7) // 8 * 8   # B as (K,N) is loaded 16 bytes along N
    rng = np.random.default_rng(M * 7 + N)
    A, B = bf(rng, M, Kdim), bf(rng, (N if b_col_maj else Kdim), (Kdim if b_col_maj else N), scale=0.1)
    guard = 64
    C = out_like((M * N + guard,), cuda, fill=3.0)
    K.gemm(dev(A, cuda), dev(B, cuda), C[: M * N].view(M, N), M=M, N=N, K=Kdim, b_col_maj=b_col_maj)
    got = from_torch(C)
    close(got[: M * N].reshape(M, N), ops.gemm(A, B, b_col_maj=b_col_maj), rtol=1e-2, atol=2e-2)
    assert np.all(got[M * N:] == 3.0)


@pytest.mark.parametrize("M,Kdim,N,rows", [
    # 64 x 64 tiles, eight stages (no more tiles than CUs): fewer k-stages than the pipeline is deep, an odd count; 64 x 32 ones, many
    (512, 64, 2048, None), (512, 192, 2048, None), (512, 576, 2048, None), (448, 1024, 1024, None),
    # 64 x 64 tiles, four stages (more tiles than CUs, too few for 128 x 128 ones): one stage, odd; under a bound 128 x 64 ones, even
    (1024, 64, 1536, None), (1024, 320, 1536, None), (1024, 512, 1536, 1000),
    # a row bound under which the blocks of one launch pick 64 x 64 and 128 x 64 tiles, short and odd in k
    (2048, 64, 2048, 512), (2048, 192, 2048, 300), (2048, 576, 2048, 896), (2048, 576, 2048, 897)])
@pytest.mark.parametrize("residual", [False, True])
def test_gemm_small_tiles_at_every_depth(cuda, M, Kdim, N, rows, residual):
    """The whole-stage-ahead pipelines of the 64 x 64 tiles where they start and end: K of one stage,
    fewer stages than are in flight, odd and even counts, with and without the residual epilogue."""
    rng = np.random.default_rng(M + Kdim + N)
    A, B, R = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.1), bf(rng, M, N)
    want = ops.gemm(A, B, b_col_maj=True)
    if residual:
        want = round_bf16(np.float32(0.5) * want + R)
    lim = M if rows is None else rows
    if rows is not None:
        A[rows:] = np.nan
    C = out_like((M, N), cuda, fill=5.0)
    bound = None if rows is None else word(rows, cuda)
    if residual:
        K.gemm_residual(dev(A, cuda), dev(B, cuda), dev(R, cuda), C, M=M, N=N, K=Kdim, residual_scale=0.5, valid=bound)
    else:
        K.gemm(dev(A, cuda), dev(B, cuda), C, M=M, N=N, K=Kdim, b_col_maj=True, valid=bound)
    got = from_torch(C)
    close(got[:lim], want[:lim], rtol=1e-2, atol=2e-2)
    assert np.all(got[lim:] == 5.0)


@pytest.mark.parametrize("cols", [2049, 2050, 2052, 2054, 2055, 2060])
@pytest.mark.parametrize("form", ["plain", "turned", "(N,M)", "residual", "pair"])
def test_gemm_rows_that_are_no_whole_pieces(cuda, cols, form):
    """Output rows of every remainder of eight elements, through the 128 x 128 tiles' stores: the columns at a row's end, and
    nothing past the output's."""
    M, Kdim = 1200, 264 if form in ("plain", "turned", "(N,M)") else 256
    rng = np.random.default_rng(cols)
    if form == "(N,M)":   # rows of M elements, B (K,N)
        A, B = bf(rng, cols, Kdim), bf(rng, Kdim, M, scale=0.05)
        want, near = ops.gemm(A, B, c_col_maj=True), ops.gemm_bound(A, B, c_col_maj=True)
    elif form == "turned":
        A, B = bf(rng, cols, Kdim), bf(rng, M, Kdim, scale=0.05)
        want, near = ops.gemm(A, B, b_col_maj=True, c_col_maj=True), ops.gemm_bound(A, B, b_col_maj=True, c_col_maj=True)
    else:
        A, B = bf(rng, M, Kdim), bf(rng, cols, Kdim, scale=0.05)
        want, near = ops.gemm(A, B, b_col_maj=True), ops.gemm_bound(A, B, b_col_maj=True)
    dA, dB, buf = dev(A, cuda), dev(B, cuda), out_like((M * cols + 64,), cuda, fill=3.0)
    C = buf[: M * cols].view(M, cols)
    if form in ("plain", "turned", "(N,M)"):
        m, n = (M, cols) if form == "plain" else (cols, M)
        K.gemm(dA, dB, C, M=m, N=n, K=Kdim, b_col_maj=form != "(N,M)", c_col_maj=form != "plain")
    elif form == "residual":
        R = bf(rng, M, cols)
        K.gemm_residual(dA, dB, dev(R, cuda), C, M=M, N=cols, K=Kdim, residual_scale=0.5)
        near = near + 2.0**-8 * np.abs(0.5 * want + R)   # the sum's own rounding
        want = np.float32(0.5) * want + R
    else:
        B2, G = bf(rng, cols, Kdim, scale=0.05), out_like((M * cols + 64,), cuda, fill=3.0)
        K.gemm_gated_pair(dA, dB, dev(B2, cuda), G[: M * cols].view(M, cols), C, M=M, N=cols, K=Kdim, activation="relu")
        assert np.all(np.abs(from_torch(G[: M * cols].view(M, cols)) - want) <= near) and bool((G[M * cols:] == 3).all())
        gate, up = np.maximum(want, 0), ops.gemm(A, B2, b_col_maj=True)
        near = near * np.abs(up) + gate * ops.gemm_bound(A, B2, b_col_maj=True) + 2.0**-7 * np.abs(gate * up) + near * ops.gemm_bound(A, B2, b_col_maj=True)
        want = gate * up
    assert np.all(np.abs(from_torch(C) - want) <= near)
    assert bool((buf[M * cols:] == 3).all())


@pytest.mark.parametrize("cols", [1, 2, 3, 5, 6, 7, 8])
@pytest.mark.parametrize("M,Kdim,N,b_col_maj,c_col_maj", [
    (8, 2048, 1032, True, False), (30, 4096, 808, True, False),     # strips, a tile a block
    (5, 1024, 16384, True, False), (16, 2048, 4096, True, False), (8, 3584, 2600, True, False), (5, 8200, 2600, True, False), (13, 2056, 6152, True, False),   # ... several, also over a long K
    (40, 264, 72, True, False), (9, 64, 8200, True, False), (7, 2056, 2600, True, False), (38, 2200, 8, True, False),   # few rows otherwise, 16 columns a block and 32
    (200, 200, 328, True, False), (24, 6200, 200, True, False),     # 64 x 64 tiles, shared tiles
    (136, 40, 200, True, False), (200, 40, 136, False, True),       # the general kernel, C as (M,N) and (N,M)
])
def test_gemm_rows_of_every_alignment(cuda, M, Kdim, N, b_col_maj, c_col_maj, cols):
    """Rows of every remainder of eight elements through every other kernel's stores: each begins where it begins, the columns
    at its end, and nothing past the output's."""
    M, N = (M + cols, N) if c_col_maj else (M, N + cols)
    rng = np.random.default_rng(M + N)
    A, B = bf(rng, M, Kdim), bf(rng, (N if b_col_maj else Kdim), (Kdim if b_col_maj else N), scale=0.05)
    buf = out_like((M * N + 64,), cuda, fill=3.0)
    C = buf[: M * N].view(*((N, M) if c_col_maj else (M, N)))
    K.gemm(dev(A, cuda), dev(B, cuda), C, M=M, N=N, K=Kdim, b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    kw = dict(b_col_maj=b_col_maj, c_col_maj=c_col_maj)
    assert np.all(np.abs(from_torch(C) - ops.gemm(A, B, **kw)) <= ops.gemm_bound(A, B, **kw))
    assert bool((buf[M * N:] == 3).all())


@pytest.mark.parametrize("M,Kdim,N,form", [(8190, 136, 140, "plain"), (348, 168, 464, "(N,M)"), (12, 176, 1000, "(N,M)"), (1004, 64, 264, "(N,M)"), (131, 64, 8212, "residual"),
                                           (131, 64, 8236, "bounded")])
def test_gemm_rows_of_whole_pieces_and_a_half_of_one_round(cuda, M, Kdim, N, form):
    """Output rows of four elements more than whole pieces, from 128 x 128 tiles that are one round: each leaves by halves, its last one alone, nothing past
    the output's end and no row past the bound."""
    c_col_maj, rows = form == "(N,M)", M - 2 if form in ("residual", "bounded") else M
    code = K.lib().iron_gemm_tile({"residual": 2, "bounded": 1}.get(form, 0), M, N, Kdim, not c_col_maj, c_col_maj, rows if rows < M else 0)
    assert code == 128 << 16 | 128 and (M if c_col_maj else N) % 8 == 4
    rng = np.random.default_rng(M + N)
    A, B, R = bf(rng, M, Kdim), bf(rng, *((Kdim, N) if c_col_maj else (N, Kdim)), scale=0.05), bf(rng, M, N)
    kw = dict(b_col_maj=not c_col_maj, c_col_maj=c_col_maj)
    want, near = ops.gemm(A, B, **kw), ops.gemm_bound(A, B, **kw)
    buf = out_like((M * N + 64,), cuda, fill=3.0)
    C = buf[: M * N].view(*((N, M) if c_col_maj else (M, N)))
    bound = word(rows, cuda) if rows < M else None
    if form == "residual":
        K.gemm_residual(dev(A, cuda), dev(B, cuda), dev(R, cuda), C, M=M, N=N, K=Kdim, residual_scale=0.5, valid=bound)
        near = near + 2.0**-8 * np.abs(0.5 * want + R)   # the sum's own rounding
        want = np.float32(0.5) * want + R
    else:
        K.gemm(dev(A, cuda), dev(B, cuda), C, M=M, N=N, K=Kdim, valid=bound, **kw)
    got = from_torch(C)
    live = slice(None) if c_col_maj else slice(rows)
    assert np.all(np.abs(got[live] - want[live]) <= near[live])
    assert bool((buf[M * N:] == 3).all()) and (c_col_maj or np.all(got[rows:] == 3))


@pytest.mark.parametrize("M,Kdim,N,b_col_maj,bounds", [
    (2000, 136, 8195, True, (130, 257, 513, 641, 769, 1025, 1281, 1537, 1999)),   # 128 x 128 to 256 x 256 by the bound, the last tiles moved back
    (2048, 200, 8192, True, (1, 128, 129, 1024, 1025, 2047)),    # 64 x 64 to 256 x 256 by the bound
    (1500, 328, 2056, True, (63, 895, 896, 897, 1500)),          # 64 and 128 ones, ragged
    (2048, 1032, 2056, True, (1, 32, 33, 65, 128, 129, 200, 257, 400)), (300, 584, 200, True, (31, 64, 97, 299)),   # 32-column ones and 64 x 64, ragged
    (256, 136, 320, True, (0, 100, 200)), (40, 1000, 4168, True, (17, 40)), (33, 4096, 520, True, (1, 32)),   # 64 x 64, 64 x 32 and 32 x 32 ones whatever the bound
    (2048, 328, 2056, False, (1, 129, 1999)), (300, 200, 136, False, (299,)), (40, 264, 72, False, (17,)),    # (K,N): the last column tile moved back
    (64, 72, 128, False, (5,)), (2, 192, 4104, False, (1,))])
def test_gemm_under_a_bound_at_the_edges_of_tiles_and_stages(cuda, M, Kdim, N, b_col_maj, bounds):
    """A bound on the rows with a K that ends inside a stage or columns inside a tile: rows past the bound are NaN on the way in and
    come out untouched, the operands lie between NaNs."""
    rng = np.random.default_rng(M + N + Kdim)
    A, B = bf(rng, M, Kdim), bf(rng, (N if b_col_maj else Kdim), (Kdim if b_col_maj else N), scale=0.05)
    want, near = ops.gemm(A, B, b_col_maj=b_col_maj), ops.gemm_bound(A, B, b_col_maj=b_col_maj)

    def between_nans(x):
        room = 64 * max(x.shape)
        buf = torch.full((x.size + 2 * room,), float("nan"), dtype=torch.bfloat16, device=cuda)
        inside = buf[room:room + x.size].view(*x.shape)
        inside.copy_(dev(x, cuda))
        return inside

    dB = between_nans(B)
    for rows in bounds:
        live = A.copy()
        live[rows:] = np.nan
        C = out_like((M, N), cuda, fill=7.0)
        K.gemm(between_nans(live), dB, C, M=M, N=N, K=Kdim, b_col_maj=b_col_maj, valid=word(rows, cuda))
        got = from_torch(C)
        assert np.all(np.abs(got[:rows] - want[:rows]) <= near[:rows]), rows
        assert np.all(got[rows:] == 7.0), rows


# Each form that a launch under a bound may take (K decides the price, so the sizes are each form's own), with a last row and column of tiles
# that are no whole ones, which the larger forms move back over their neighbours'.
ROWS_FORMS = {(32, 32): (75, 512, 80), (64, 32): (67, 512, 2808), (64, 64): (74, 64, 80), (128, 64): (132, 64, 8080), (128, 128): (131, 64, 8232),
              (160, 128): (389, 64, 8200), (160, 256): (771, 64, 8256), (192, 128): (482, 64, 8200), (192, 256): (965, 64, 9224), (256, 128): (579, 64, 8208),
              (256, 256): (1156, 64, 9224)}
TAIL_FORMS = {(32, 32): (73, 512, 72), (64, 32): (67, 512, 2736), (64, 64): (68, 64, 72), (128, 64): (131, 64, 8088), (128, 128): (131, 64, 8208),
              (160, 128): (387, 64, 8240), (160, 256): (774, 64, 9424), (192, 128): (481, 64, 8208), (192, 256): (966, 192, 9352), (256, 128): (579, 64, 8216),
              (256, 256): (1413, 512, 8216)}
PAIR_FORMS = [((64, 32), (81, 64, 80)), ((128, 64), (134, 64, 2752)), ((128, 128), (67, 64, 8320)), ((128, 128), (68, 64, 8232)), ((128, 128), (131, 64, 8320)), ((128, 128), (131, 2048, 8320)), ((160, 64), (259, 64, 5504)),
              ((160, 128), (387, 64, 8320)), ((192, 64), (323, 64, 5504)), ((192, 128), (481, 64, 8320)), ((224, 128), (579, 64, 8320)), ((256, 128), (674, 64, 8320))]


@pytest.mark.parametrize("kind,tile,size", [*((k, *f) for k in ("plain", "residual", "gated") for f in (ROWS_FORMS if k == "plain" else TAIL_FORMS).items()),
                                            *(("pair", *f) for f in PAIR_FORMS)])
def test_every_form_of_a_launch_under_a_bound(cuda, kind, tile, size):
    """Each size of tile, named by the launch's own choice, under a bound a few rows short of its last tile's end: against the oracle, rows
    past the bound untouched; with a second operand also in place, where a tile moved back reads what its neighbour has
    perhaps stored already, three times over the same bits."""
    M, Kdim, N = size
    rows = M - 2
    code = K.lib().iron_gemm_tile({"plain": 1, "residual": 2, "gated": 2, "pair": 3}[kind], M, N, Kdim, 1, 0, rows)
    assert (code >> 16, code & 65535) == tile
    rng = np.random.default_rng(M + N)
    A, B, B2, R = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.05), bf(rng, N, Kdim, scale=0.05), bf(rng, M, N)
    want, near = ops.gemm(A, B, b_col_maj=True), ops.gemm_bound(A, B, b_col_maj=True)
    A[rows:] = np.nan
    dA, dB, dR, bound = dev(A, cuda), dev(B, cuda), dev(R, cuda), word(rows, cuda)
    kw = dict(M=M, N=N, K=Kdim, valid=bound)
    C, G = out_like((M, N), cuda, fill=7.0), out_like((M, N), cuda, fill=7.0)
    if kind == "plain":
        K.gemm(dA, dB, C, b_col_maj=True, **kw)
        product = C
    elif kind == "pair":
        K.gemm_gated_pair(dA, dB, dev(B2, cuda), G, C, activation="relu", **kw)
        product = G
    else:
        product = out_like((M, N), cuda, fill=7.0)
        K.gemm(dA, dB, product, b_col_maj=True, **kw)
    assert np.all(np.abs(from_torch(product)[:rows] - want[:rows]) <= near[:rows]) and bool((product[rows:] == 7).all())
    if kind == "pair":
        up = out_like((M, N), cuda, fill=7.0)
        K.gemm_gated(dA, dev(B2, cuda), G, up, activation="relu", **kw)
        assert torch.equal(C[:rows], up[:rows]) and bool((C[rows:] == 7).all())
    elif kind != "plain":
        def run(to, R_):
            if kind == "residual":
                K.gemm_residual(dA, dB, R_, to, residual_scale=0.5, **kw)
            else:
                K.gemm_gated(dA, dB, R_, to, activation="relu", **kw)
            return to

        run(C, dR)
        p = from_torch(product)[:rows]   # the product as the separate launch rounds it
        link = round_bf16(np.float32(0.5) * p + R[:rows]) if kind == "residual" else ops.mul(np.maximum(R[:rows], 0), p)
        assert np.array_equal(from_torch(C)[:rows], link) and bool((C[rows:] == 7).all())
        for _ in range(3):
            held = dR.clone()
            assert torch.equal(run(held, held)[:rows], C[:rows]) and torch.equal(held[rows:], dR[rows:])


# Tiles of 96 x 128 and 224 x 256 without a bound, which begin past K = 512: the last ones moved back, a K that is no whole number of stages, rows that straddle lines.
@pytest.mark.parametrize("tile,M,Kdim,N,col", [((96, 128), 902, 520, 2059, True), ((96, 128), 1798, 520, 1032, True), ((224, 256), 1413, 520, 8200, True), ((224, 256), 1350, 520, 8200, False)])
def test_tiles_of_96_and_224_rows_without_a_bound(cuda, tile, M, Kdim, N, col):
    code = K.lib().iron_gemm_tile(0, M, N, Kdim, col, 0, 0)
    assert (code >> 16, code & 65535) == tile
    rng = np.random.default_rng(M + N)
    A, B = bf(rng, M, Kdim), bf(rng, *((N, Kdim) if col else (Kdim, N)), scale=0.05)
    C, bounded = out_like((M, N), cuda, fill=7.0), out_like((M, N), cuda, fill=7.0)
    kw = dict(M=M, N=N, K=Kdim, b_col_maj=col)
    K.gemm(dev(A, cuda), dev(B, cuda), C, **kw)
    K.gemm(dev(A, cuda), dev(B, cuda), bounded, valid=word(M, cuda), **kw)
    assert torch.equal(C, bounded)   # the same chain of products whatever the tile
    sample = np.unique(np.concatenate([[0, 95, 96, 223, 224, M - 97, M - 1], rng.integers(0, M, 40)]))
    close(from_torch(C)[sample], ops.gemm(A[sample], B, b_col_maj=col), rtol=1e-2, atol=1e-2)


# ... and tiles of 96 and 224 rows, which begin past K = 512; the last ones moved back.
@pytest.mark.parametrize("kind,tile,size", [*((k, *f) for k in ("plain", "residual", "gated") for f in (((96, 128), (131, 576, 8208)), ((224, 128), (579, 576, 9224)),
                                                                                                      ((224, 256), (1155, 576, 9224) if k == "plain" else (579, 1088, 16392)))),
                                            ("pair", (96, 64), (131, 576, 2752)), ("pair", (224, 64), (387, 576, 5504))])
def test_tiles_of_96_and_224_rows_under_a_bound(cuda, kind, tile, size):
    test_every_form_of_a_launch_under_a_bound(cuda, kind, tile, size)


@pytest.mark.parametrize("M,Kdim,N,form", [(*s, f) for s in ((2048, 2048, 2048), (2048, 1024, 8192), (1500, 320, 4160))
                                           for f in ("plain", "residual", "gated", "pair")] +
                         [(2048, 200, 8192, "plain"), (2048, 128, 5632, "pair"), (2000, 192, 888, "pair")])
def test_a_row_s_products_are_the_same_bits_under_every_bound(cuda, M, Kdim, N, form):
    """A bound on the rows chooses the tile (from 32 x 32 to 256 x 256), and with it nothing about a row's sums: what a row
    becomes does not depend on how many others there are."""
    rng = np.random.default_rng(M + N)
    A, B, B2, R = (dev(bf(rng, *s, scale=x), cuda) for s, x in (((M, Kdim), 1.0), ((N, Kdim), 0.05), ((N, Kdim), 0.05), ((M, N), 1.0)))
    kw = dict(M=M, N=N, K=Kdim)

    def run(rows):
        C, G = out_like((M, N), cuda, fill=7.0), out_like((M, N), cuda, fill=7.0)
        if form == "plain":
            K.gemm(A, B, C, b_col_maj=True, valid=word(rows, cuda), **kw)
        elif form == "residual":
            K.gemm_residual(A, B, R, C, residual_scale=0.5, valid=word(rows, cuda), **kw)
        elif form == "gated":
            K.gemm_gated(A, B, R, C, activation="silu", valid=word(rows, cuda), **kw)
        else:
            K.gemm_gated_pair(A, B, B2, G, C, activation="silu", valid=word(rows, cuda), **kw)
        return C, G

    whole = run(M)
    for rows in (5, 32, 33, 64, 65, 128, 129, 256, 257, 384, 385, 513, 896, 897, 1025, 1281):
        for got, want in zip(run(rows), whole):
            assert torch.equal(got[:rows], want[:rows]), rows
            assert (got[rows:] == 7).all(), rows


# One row of tiles, whose stages are 256 columns of K: one stage (a pair's; of the others two, shorter ones go by tiles of 64 x 64), fewer than the ring holds, more; one
# tile of eight columns, some, one a CU (and a tile more, which the others take); rows on either side of sixteen and of the tile's.
@pytest.mark.parametrize("Kdim", [256, 512, 768, 2304])
@pytest.mark.parametrize("N", [8, 200, 2048, 2056])
@pytest.mark.parametrize("form", ["plain", "residual", "gated", "pair"])
def test_few_rows_over_long_stages_are_the_same_bits_as_among_many(cuda, Kdim, N, form):
    rng = np.random.default_rng(Kdim + N)
    M = 600
    N = N if form == "plain" else max(64, 32 * -(-N // 32) if form == "pair" else N)   # (the fewest columns that a second operand is taken with)
    A, B, B2, R = (bf(rng, *s, scale=x) for s, x in (((M, Kdim), 1.0), ((N, Kdim), 0.05), ((N, Kdim), 0.05), ((M, N), 1.0)))
    dB, dB2, dR, kw = dev(B, cuda), dev(B2, cuda), dev(R, cuda), dict(M=M, N=N, K=Kdim)
    by_long_stages = form == "pair" or (Kdim >= 512 and N <= 2048)
    for rows in (1, 32, 33, M):   # (1 << 15: by long stages)
        code = K.lib().iron_gemm_tile({"plain": 1, "residual": 2, "gated": 2, "pair": 3}[form], M, N, Kdim, 1, 0, rows)
        assert code >> 15 & 1 == (by_long_stages and rows <= 32) and (rows > 32 or not by_long_stages or code & 32767 == (32 if form == "pair" else 8))

    def run(rows):
        C, G = out_like((M, N), cuda, fill=7.0), out_like((M, N), cuda, fill=7.0)
        held = A.copy()
        held[rows:] = np.nan
        dA, bound = dev(held, cuda), word(rows, cuda)
        if form == "plain":
            K.gemm(dA, dB, C, b_col_maj=True, valid=bound, **kw)
        elif form == "residual":
            K.gemm_residual(dA, dB, dR, C, residual_scale=0.5, valid=bound, **kw)
        elif form == "gated":
            K.gemm_gated(dA, dB, dR, C, activation="silu", valid=bound, **kw)
        else:
            K.gemm_gated_pair(dA, dB, dB2, G, C, activation="silu", valid=bound, **kw)
        return C, G

    whole = run(M)
    if form in ("plain", "pair"):
        close(whole[form == "pair"][:33], ops.gemm(A[:33], B, b_col_maj=True), rtol=1e-2, atol=1e-2)
    for rows in (1, 8, 16, 17, 31, 32):
        for got, want in zip(run(rows), whole):
            assert torch.equal(got[:rows], want[:rows]), rows
            assert (got[rows:] == 7).all(), rows


# Without a bound: eight, sixteen, thirty-two and sixty-four rows of B a block, the last block's cut; one stage, a last one of eight columns and of all but eight, more than the ring holds.
@pytest.mark.parametrize("M", [17, 31, 32])
@pytest.mark.parametrize("Kdim,N", [(1088, 256), (1032, 2047), (1272, 2049), (2304, 300), (2040, 1001), (1032, 4095), (1088, 4097), (1344, 8189), (320, 8200), (256, 16383)])
@pytest.mark.parametrize("turned", [False, True])
def test_few_rows_over_long_stages_without_a_bound(cuda, M, Kdim, N, turned):
    """Against the oracle; turned: the (N,M) output of B and A, the same product."""
    code = K.lib().iron_gemm_tile(0, *((N, M) if turned else (M, N)), Kdim, 1, turned, 0)
    assert code == 32 << 16 | 1 << 15 | (8 if N <= 2048 else 16 if N <= 4096 else 32 if N <= 8192 else 64)
    rng = np.random.default_rng(M + N)
    A, B = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.05)
    C = out_like((M + 1, N), cuda, fill=7.0)
    if turned:
        K.gemm(dev(B, cuda), dev(A, cuda), C[:M], M=N, N=M, K=Kdim, b_col_maj=True, c_col_maj=True)
    else:
        K.gemm(dev(A, cuda), dev(B, cuda), C[:M], M=M, N=N, K=Kdim, b_col_maj=True)
    close(from_torch(C)[:M], ops.gemm(A, B, b_col_maj=True), rtol=1e-2, atol=1e-2)
    assert (C[M] == 7).all()


@pytest.mark.parametrize("E", [256, 1280])
@pytest.mark.parametrize("H,G", [(32, 8), (48, 8), (56, 8), (4, 2)])   # the most heads whose tiles are one round, and more
def test_few_rows_projections_are_the_same_bits_as_among_many(cuda, E, H, G):
    rng = np.random.default_rng(E + H)
    rows, D = 1024, 64
    x, Wq, Wk, Wv = bf(rng, rows, E), bf(rng, H * D, E, scale=0.05), bf(rng, G * D, E, scale=0.05), bf(rng, G * D, E, scale=0.05)
    fixed = [dev(a, cuda) for a in (Wq, Wk, Wv, round_bf16(ops.rope_angles(D, rows, 500000.0)))]

    def run(bound):
        held = x.copy()
        held[bound:] = np.nan
        outs = [out_like((rows, n), cuda, fill=7.0) for n in (H * D, G * D, G * D)]
        K.prefill_qkv(dev(held, cuda), *fixed, *outs, rows=rows, hidden=E, heads=H, kv_heads=G, d=D, valid=word(bound, cuda))
        return outs

    many = run(100)   # tiles of 64 columns of K
    for bound in (1, 16, 17, 32, 33, 63, 64):
        for got, want in zip(run(bound), many):
            assert torch.equal(got[:bound], want[:bound]), bound
            assert (got[bound:] == 7).all(), bound


@pytest.mark.parametrize("rows,bound,H,G", [(2048, None, 32, 8), (256, 150, 16, 4), (128, None, 2, 2),
                                            # bounds on either side of where the 192-wide tiles take over
                                            (2048, 1280, 32, 8), (2048, 1281, 32, 8), (2048, 1999, 32, 8),
                                            (2048, 2048, 32, 8), (2048, 70, 32, 8),
                                            # ... and of 64-row tiles' half and whole heads
                                            (2048, 1, 32, 8), (2048, 129, 32, 8), (2048, 320, 32, 8), (2048, 321, 32, 8), (256, 31, 16, 4), (130, None, 4, 2),
                                            # heads that do not come in threes keep the 128-wide tiles
                                            (2048, None, 32, 4), (1024, None, 8, 2), (4096, 3000, 16, 4)])
def test_prefill_qkv_equals_three_projections_then_rope(cuda, rows, bound, H, G):
    """The fused launch against the oracle's separate steps: project and round, rotate and round."""
    rng = np.random.default_rng(91)
    E, D = 512, 64
    x = bf(rng, rows, E)
    Wq, Wk, Wv = bf(rng, H * D, E, scale=0.05), bf(rng, G * D, E, scale=0.05), bf(rng, G * D, E, scale=0.05)
    table = round_bf16(ops.rope_angles(D, rows + 5, 500000.0))[5:]
    lim = rows if bound is None else bound
    q, k, v = (ops.gemm(x, W, b_col_maj=True) for W in (Wq, Wk, Wv))
    want_q = ops.rope(q.reshape(rows * H, D), table).reshape(rows, H * D)
    want_k = ops.rope(k.reshape(rows * G, D), table).reshape(rows, G * D)
    if bound is not None:
        x[bound:] = np.nan
    outs = [out_like((rows, n), cuda, fill=7.0) for n in (H * D, G * D, G * D)]
    K.prefill_qkv(dev(x, cuda), dev(Wq, cuda), dev(Wk, cuda), dev(Wv, cuda), dev(table, cuda), *outs, rows=rows,
                  hidden=E, heads=H, kv_heads=G, d=D, valid=None if bound is None else word(bound, cuda))
    for got, want in zip(outs, (want_q, want_k, v)):
        got = from_torch(got)
        close(got[:lim], want[:lim], rtol=1e-2, atol=1e-2)
        assert np.all(got[lim:] == 7.0)


@pytest.mark.parametrize("E", [64, 192, 320, 576])
@pytest.mark.parametrize("rows,bound", [(512, None), (2048, 600), (2048, 100), (2048, 300), (300, None)])
def test_prefill_qkv_one_head_tiles_at_short_hidden(cuda, E, rows, bound):
    """The one-head tiles a short chunk takes (whole-stage-ahead pipeline, five stages) with fewer
    k-stages than are in flight and an odd count of them; the 64-row tiles of few rows likewise."""
    rng = np.random.default_rng(E + rows)
    H, G, D = 32, 8, 64
    x = bf(rng, rows, E)
    Wq, Wk, Wv = bf(rng, H * D, E, scale=0.05), bf(rng, G * D, E, scale=0.05), bf(rng, G * D, E, scale=0.05)
    table = round_bf16(ops.rope_angles(D, rows, 500000.0))
    lim = rows if bound is None else bound
    q, k, v = (ops.gemm(x, W, b_col_maj=True) for W in (Wq, Wk, Wv))
    want_q = ops.rope(q.reshape(rows * H, D), table).reshape(rows, H * D)
    want_k = ops.rope(k.reshape(rows * G, D), table).reshape(rows, G * D)
    if bound is not None:
        x[bound:] = np.nan
    outs = [out_like((rows, n), cuda, fill=7.0) for n in (H * D, G * D, G * D)]
    K.prefill_qkv(dev(x, cuda), dev(Wq, cuda), dev(Wk, cuda), dev(Wv, cuda), dev(table, cuda), *outs, rows=rows,
                  hidden=E, heads=H, kv_heads=G, d=D, valid=None if bound is None else word(bound, cuda))
    for got, want in zip(outs, (want_q, want_k, v)):
        got = from_torch(got)
        close(got[:lim], want[:lim], rtol=1e-2, atol=1e-2)
        assert np.all(got[lim:] == 7.0)


@pytest.mark.parametrize("rows,bound,start,L,H,G", [(256, 150, 300, 1024, 16, 4), (2048, 512, 0, 2048, 32, 8),
                                                    (2048, 1500, 548, 2048, 32, 8), (128, None, 128, 256, 2, 2),
                                                    (256, 64, 960, 1024, 6, 2)])
def test_prefill_qkv_writes_k_and_v_into_the_cache_rows(cuda, rows, bound, start, L, H, G):
    """k and v land in rows start .. start + bound of the caches, bit for bit what the launch with
    outputs of its own writes; every other cache row is left as it was."""
    rng = np.random.default_rng(92)
    E, D = 512, 64
    x = bf(rng, rows, E)
    Wq, Wk, Wv = bf(rng, H * D, E, scale=0.05), bf(rng, G * D, E, scale=0.05), bf(rng, G * D, E, scale=0.05)
    table = round_bf16(ops.rope_angles(D, rows, 500000.0))
    lim = rows if bound is None else bound
    if bound is not None:
        x[bound:] = np.nan
    valid = None if bound is None else word(bound, cuda)
    args = [dev(a, cuda) for a in (x, Wq, Wk, Wv, table)]
    outs = [out_like((rows, n), cuda, fill=7.0) for n in (H * D, G * D, G * D)]
    K.prefill_qkv(*args, *outs, rows=rows, hidden=E, heads=H, kv_heads=G, d=D, valid=valid)
    q = out_like((rows, H * D), cuda, fill=7.0)
    keys, values = (out_like((L, G * D), cuda, fill=3.0) for _ in range(2))
    K.prefill_qkv_cache(*args, q, keys, values, rows=rows, hidden=E, heads=H, kv_heads=G, d=D, cache_rows=L,
                        start=word(start, cuda), valid=valid)
    assert torch.equal(q, outs[0])
    for cache, own in ((keys, outs[1]), (values, outs[2])):
        assert torch.equal(cache[start : start + lim], own[:lim])
        assert bool((cache[:start] == 3.0).all()) and bool((cache[start + lim :] == 3.0).all())
    # A first row whose rows would end past the cache is held inside it.
    K.prefill_qkv_cache(*args, q, keys, values, rows=rows, hidden=E, heads=H, kv_heads=G, d=D, cache_rows=L,
                        start=word(L, cuda), valid=valid)
    assert torch.equal(keys[L - lim :], outs[1][:lim])


@pytest.mark.parametrize("M,Kdim,N,rows,scale", [(2048, 512, 2048, None, 1.0), (2048, 256, 2048, 512, 1.0),
                                                 (2048, 256, 2048, 1500, 0.22), (256, 128, 512, 100, 1.0),
                                                 (128, 64, 64, None, -0.5), (4096, 192, 1024, 3000, 1.0),
                                                 # tiles of 128, 160, 192 and 256 rows by 128 and 256 columns, the last moved back over its neighbour
                                                 *[(2000, 128, 8200, rows, 1.0) for rows in (200, 641, 769, 1025, 1281, 1537, 2000, None)]])
def test_gemm_residual_epilogue(cuda, M, Kdim, N, rows, scale):
    """A projection over many rows with its residual in the epilogue: the product rounded as the
    separate step would store it, then one fused multiply-add with the residual (the sum, or AXPY)."""
    rng = np.random.default_rng(M + N)
    A, B, R = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.05), bf(rng, M, N)
    lim = M if rows is None else rows
    want = ops.axpy(scale, ops.gemm(A, B, b_col_maj=True), R)
    if scale == 1.0:
        assert np.array_equal(want, ops.add(ops.gemm(A, B, b_col_maj=True), R))
    if rows is not None:
        A[rows:] = np.nan
    C = out_like((M, N), cuda, fill=7.0)
    K.gemm_residual(dev(A, cuda), dev(B, cuda), dev(R, cuda), C, M=M, N=N, K=Kdim, residual_scale=scale,
                    valid=None if rows is None else word(rows, cuda))
    got = from_torch(C)
    close(got[:lim], want[:lim], rtol=1e-2, atol=1e-2)
    assert np.all(got[lim:] == 7.0)
    # in place: the residual stream is its own output
    Rd = dev(R, cuda)
    K.gemm_residual(dev(np.nan_to_num(A), cuda), dev(B, cuda), Rd, Rd, M=M, N=N, K=Kdim, residual_scale=scale,
                    valid=None if rows is None else word(rows, cuda))
    close(from_torch(Rd)[:lim], want[:lim], rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("M,Kdim,N,rows,scale", [
    (2048, 8192, 2048, 512, 1.0),     # a prompt chunk's down projection: K dealt four ways, a slice an XCD pair
    (2048, 4096, 2048, 1024, 1.0),    # two ways
    (2048, 4096, 2048, 1281, 0.22),   # whole K: the first launch is the plain residual product's
    (512, 4096, 2048, None, 1.0),
    (256, 4096, 128, 130, 1.0),       # one tile column, a tile row the bound cuts
    (384, 4096, 384, 300, -0.5),      # pairs that do not fill whole XCD rounds
    (256, 4096, 4096, 77, 1.0),       # two pieces of a row a thread
    (128, 4608, 8192, None, 1.0)])    # four
def test_gemm_residual_then_rmsnorm_with_k_dealt_over_blocks(cuda, M, Kdim, N, rows, scale):
    """A residual product of few rows over a long K and the norm of its rows as two launches: the
    product's K dealt over several blocks a tile (float32 sums through a workspace holding garbage),
    the rows finished and normed by the second.  C against the oracle's product and sum; Y is the
    norm kernel's of that C bit for bit, and within tolerance of the oracle's norm of it; rows past
    the bound are not touched; in place on the residual stream."""
    rng = np.random.default_rng(M + N + Kdim)
    lim = M if rows is None else rows
    A, B, R, gain = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.02), bf(rng, M, N), bf(rng, N)
    product = ops.gemm(A[:lim], B, b_col_maj=True)
    want = ops.axpy(scale, product, R[:lim])
    # The product is rounded before the sum: where the float32 sums differ in their last bits it may
    # round to the neighbouring bf16 (2^-7 of it at most), whatever the sum then cancels to.
    ulp = np.abs(scale * product) * 2.0 ** -7

    def near(got, want):
        err = np.abs(got.astype(np.float64) - want.astype(np.float64))
        bad = ~(err <= 1e-2 + 1e-2 * np.abs(want) + ulp)
        assert not bad.any(), f"{bad.sum()}/{bad.size} outside the tolerance; max err {err.max():.5f}"

    if rows is not None:
        A[rows:] = np.nan
    valid = None if rows is None else word(rows, cuda)
    need = K.gemm_residual_norm_workspace_bytes(M, N, Kdim)
    assert need > 0
    ws = torch.full((need // 4,), float("nan"), dtype=torch.float32, device=cuda)
    Ad, Bd, Rd, gd = dev(A, cuda), dev(B, cuda), dev(R, cuda), dev(gain, cuda)
    C, Y = out_like((M, N), cuda, fill=7.0), out_like((M, N), cuda, fill=7.0)
    K.gemm_residual_norm(Ad, Bd, Rd, gd, C, Y, ws, M=M, N=N, K=Kdim, eps=1e-6, residual_scale=scale, valid=valid)
    got = from_torch(C)
    near(got[:lim], want)
    assert np.all(got[lim:] == 7.0) and bool((Y[lim:] == 7.0).all())
    normed = out_like((M, N), cuda, fill=7.0)
    K.rmsnorm(C, gd, normed, rows=M, cols=N, eps=1e-6, valid=valid)
    assert torch.equal(Y[:lim], normed[:lim])
    close(from_torch(Y)[:lim], ops.rms_norm(got[:lim], gain, epsilon=1e-6), rtol=1e-2, atol=1e-2)
    # again over the workspace the first call left, in place on the residual stream: the same bits
    Y2 = out_like((M, N), cuda, fill=7.0)
    K.gemm_residual_norm(Ad, Bd, Rd, gd, Rd, Y2, ws, M=M, N=N, K=Kdim, eps=1e-6, residual_scale=scale, valid=valid)
    assert torch.equal(Rd[:lim], C[:lim]) and torch.equal(Y2[:lim], Y[:lim])
    assert np.array_equal(from_torch(Rd)[lim:], R[lim:])


# Sixteen slices: a 1B prompt's few rows and the most there are for it; K no power of two; tile columns that the tiles of sixteen do
# not fill, two tile rows; a row of four pieces a thread.  Eight, of a K that sixteen cut too short or not whole.
@pytest.mark.parametrize("M,Kdim,N,rows,slices", [(2048, 8192, 2048, 29, 16), (2048, 8192, 2048, 128, 16), (256, 14336, 384, 130, 16), (128, 9216, 1024, None, 16),
                                                  (256, 8192, 1024, 256, 8), (256, 5632, 256, 200, 8), (128, 4608, 4096, 77, 8), (256, 4096, 2048, 200, 4)])
def test_gemm_residual_then_rmsnorm_with_k_dealt_over_many_blocks(cuda, M, Kdim, N, rows, slices):
    test_gemm_residual_then_rmsnorm_with_k_dealt_over_blocks(cuda, M, Kdim, N, rows, 1.0)
    # ... and as many slices of sums as the rows and K call for: the workspace holds them one behind the other.
    A, B, R = (torch.ones(s, dtype=torch.bfloat16, device=cuda) for s in ((M, Kdim), (N, Kdim), (M, N)))
    ws = torch.full((K.gemm_residual_norm_workspace_bytes(M, N, Kdim) // 4,), float("nan"), dtype=torch.float32, device=cuda)
    K.gemm_residual_norm(A, B, R, R[0], torch.empty_like(R), torch.empty_like(R), ws, M=M, N=N, K=Kdim, eps=1e-6,
                         valid=None if rows is None else word(rows, cuda))
    sums = ws[~ws.isnan()]
    assert (sums == Kdim // slices).all() and sums.numel() == slices * (rows or M) * N


# Three, five, six and seven slices, whose stages do not come out even: rows on either side of a count, a K of 64 and of 72 stages, a bound inside a tile.
@pytest.mark.parametrize("M,Kdim,N,rows,slices", [(1024, 4096, 2048, 640, 3), (1024, 4096, 2048, 641, 2), (384, 4608, 2048, 300, 5), (128, 4096, 5120, 77, 6), (512, 4096, 1152, 500, 7),
                                                  (512, 4608, 1024, 512, 4)])
def test_gemm_residual_then_rmsnorm_with_k_dealt_unevenly(cuda, M, Kdim, N, rows, slices):
    test_gemm_residual_then_rmsnorm_with_k_dealt_over_blocks(cuda, M, Kdim, N, rows, 1.0)
    A, B, R = (torch.ones(s, dtype=torch.bfloat16, device=cuda) for s in ((M, Kdim), (N, Kdim), (M, N)))
    ws = torch.full((K.gemm_residual_norm_workspace_bytes(M, N, Kdim) // 4,), float("nan"), dtype=torch.float32, device=cuda)
    K.gemm_residual_norm(A, B, R, R[0], torch.empty_like(R), torch.empty_like(R), ws, M=M, N=N, K=Kdim, eps=1e-6, valid=word(rows, cuda))
    sums, stages = ws[~ws.isnan()], Kdim // 64
    assert sums.numel() == slices * rows * N and int(sums.double().sum()) == Kdim * rows * N
    assert set(sums.unique().tolist()) <= {64.0 * (stages // slices), 64.0 * -(-stages // slices)}


# Whole K by tiles of 96 rows while they are one round: the last one moved back, the most rows there are, and one more.
@pytest.mark.parametrize("M,rows", [(1500, 1473), (2048, 1536), (2048, 1537)])
def test_gemm_residual_then_rmsnorm_by_tiles_of_96_rows(cuda, M, rows):
    test_gemm_residual_then_rmsnorm_with_k_dealt_over_blocks(cuda, M, 4096, 2048, rows, 1.0)


def test_gemm_residual_then_rmsnorm_refuses_other_shapes(cuda):
    """Shapes whose K is too short to deal, or whose rows the second launch cannot hold, report no
    workspace and are refused with a reason before any launch."""
    for M, N, Kdim in ((64, 2048, 8192), (512, 2048, 2048), (512, 2000, 8192), (512, 16384, 8192), (512, 2048, 8192 + 64)):
        assert K.gemm_residual_norm_workspace_bytes(M, N, Kdim) == 0
    t, w = out_like((512 * 2048,), cuda, fill=0.0), out_like((2048 * 2048,), cuda, fill=0.0)
    with pytest.raises(Exception, match="iron_gemm_residual_norm_bf16 refused"):
        K.gemm_residual_norm(t, w, t, t[:2048], t, out_like((512 * 2048,), cuda), torch.empty(16, device=cuda),
                             M=512, N=2048, K=2048, eps=1e-6)


@pytest.mark.parametrize("M,Kdim,N,rows,activation", [
    (2048, 2048, 8192, 512, "silu"), (2048, 256, 8192, None, "silu"), (2048, 256, 2048, 1500, "silu"),
    (256, 128, 512, 100, "silu"), (128, 64, 64, None, "silu"), (4096, 192, 1024, 3000, "silu"), (200, 128, 136, None, "silu"),
    (2048, 256, 8192, 512, "gelu_tanh"), (256, 128, 512, 100, "gelu_tanh"), (200, 128, 136, None, "gelu_tanh")])
def test_gemm_gated_epilogue(cuda, M, Kdim, N, rows, activation):
    """A gated feed-forward's second projection over many rows with the activated gate (SiLU, or
    GELU by its tanh form) in its epilogue.  The chain rounds twice (the product, then the gated
    product), so it is checked link by link: the product of the separate launch against the oracle's
    GEMM, the fused launch against the oracle's activation and ElementwiseMul of that product, and
    bit for bit against this library's own separate launches.  The first case is Llama-3.2-1B's
    prompt chunk."""
    rng = np.random.default_rng(M + N + 1)
    A, B, G = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.05), bf(rng, M, N, scale=2.0)
    lim = M if rows is None else rows
    product = ops.gemm(A[:lim], B, b_col_maj=True)
    if rows is not None:
        A[rows:] = np.nan
    bound = None if rows is None else word(rows, cuda)
    flat_bound = None if rows is None else word(rows * N, cuda)
    # the separate launches: the product, then the activation and the multiplication
    U, Y = out_like((M, N), cuda, fill=7.0), out_like((M, N), cuda, fill=7.0)
    K.gemm(dev(A, cuda), dev(B, cuda), U, M=M, N=N, K=Kdim, b_col_maj=True, valid=bound)
    if activation == "silu":
        K.silu_mul(dev(G, cuda).reshape(-1), U.reshape(-1), Y.reshape(-1), n=M * N, valid=flat_bound)
        activated = ops.silu(G[:lim])
    else:
        act = out_like((M, N), cuda, fill=7.0)
        K.unary(dev(G, cuda).reshape(-1), act.reshape(-1), "gelu_tanh", n=M * N, valid=flat_bound)
        K.mul(act.reshape(-1), U.reshape(-1), Y.reshape(-1), n=M * N, valid=flat_bound)
        activated = ops.gelu(G[:lim], approximate="tanh")
    close(U[:lim], product, rtol=1e-2, atol=1e-2)
    C = out_like((M, N), cuda, fill=7.0)
    K.gemm_gated(dev(A, cuda), dev(B, cuda), dev(G, cuda), C, M=M, N=N, K=Kdim, activation=activation, valid=bound)
    got = from_torch(C)
    close(got[:lim], ops.mul(activated, from_torch(U)[:lim]), rtol=1e-2, atol=1e-2)
    assert np.all(got[lim:] == 7.0)
    assert torch.equal(Y[:lim], C[:lim])
    # in place: the gate's product is its own output
    Gd = dev(G, cuda)
    K.gemm_gated(dev(np.nan_to_num(A), cuda), dev(B, cuda), Gd, Gd, M=M, N=N, K=Kdim, activation=activation, valid=bound)
    assert torch.equal(Gd[:lim], C[:lim])


@pytest.mark.parametrize("M,Kdim,N,rows", [(2048, 2048, 8192, 512), (2048, 2048, 8192, 1281), (2048, 2048, 8192, 100),
                                           (256, 512, 1024, None), (192, 128, 320, 70),
                                           # 256-row tiles: one stage, two, the last tile moved back, a bound inside it
                                           (2048, 64, 4096, None), (1300, 128, 4096, None), (1301, 192, 4096, 1100),
                                           (257, 64, 16512, 257), (1300, 128, 4100, None),
                                           # every form by the bound: 64 x 32 (of each), 128 x 64, 160 x 64, 192 x 64, 128 x 128, 160, 192, 224, 256 x 128
                                           *[(2000, 128, 8192, rows) for rows in (1, 64, 65, 256, 257, 320, 321, 449, 513, 641, 769, 1600, 1793, 2000)],
                                           (1999, 192, 4160, 1100), (4500, 64, 1088, 3000), (160, 64, 2048, 159)])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_gemm_gated_pair_is_the_two_launches_bit_for_bit(cuda, M, Kdim, N, rows, activation):
    """Both first projections of a gated feed-forward in one launch: the gate's product and the gated
    output against the two launches they replace (the gate's GEMM, then the gated GEMM) bit for bit --
    under row bounds that pick every size of tile, and none whole -- and the gate's
    product against the oracle's GEMM; rows past the bound are left as they were.  The first case is
    Llama-3.2-1B's prompt chunk."""
    rng = np.random.default_rng(M + N + 3)
    A, Bg, Bu = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.05), bf(rng, N, Kdim, scale=0.05)
    lim = M if rows is None else rows
    if rows is not None:
        A[rows:] = np.nan
    bound = None if rows is None else word(rows, cuda)
    dA, dBg, dBu = dev(A, cuda), dev(Bg, cuda), dev(Bu, cuda)
    G2, C2 = out_like((M, N), cuda, fill=7.0), out_like((M, N), cuda, fill=7.0)
    K.gemm(dA, dBg, G2, M=M, N=N, K=Kdim, b_col_maj=True, valid=bound)
    K.gemm_gated(dA, dBu, G2, C2, M=M, N=N, K=Kdim, activation=activation, valid=bound)
    G1, C1 = out_like((M, N), cuda, fill=7.0), out_like((M, N), cuda, fill=7.0)
    K.gemm_gated_pair(dA, dBg, dBu, G1, C1, M=M, N=N, K=Kdim, activation=activation, valid=bound)
    close(G1[:lim], ops.gemm(A[:lim], Bg, b_col_maj=True), rtol=1e-2, atol=1e-2)
    assert torch.equal(G1[:lim], G2[:lim]) and torch.equal(C1[:lim], C2[:lim])
    assert np.all(from_torch(C1)[lim:] == 7.0) and np.all(from_torch(G1)[lim:] == 7.0)


# few rows; 64 x 32, edged, 128 x 64, 128 x 128 by both bodies and 256 x 128 tiles; a bound inside a tile
@pytest.mark.parametrize("M,Kdim,N,rows", [(40, 128, 320, None), (192, 128, 320, 70), (1300, 128, 4100, None), (2000, 128, 8192, 200), (1024, 512, 4096, None),
                                           (1024, 2048, 4096, 1000), (2048, 128, 8192, 1999)])
def test_gemm_gated_product_is_the_pair_without_the_gate_s_own(cuda, M, Kdim, N, rows):
    rng = np.random.default_rng(M + N)
    A, Bg, Bu = (dev(bf(rng, *shape, scale=0.1), cuda) for shape in ((M, Kdim), (N, Kdim), (N, Kdim)))
    G, want, got = (out_like((M, N), cuda, fill=7.0) for _ in range(3))
    kw = dict(M=M, N=N, K=Kdim, activation="silu", valid=None if rows is None else word(rows, cuda))
    K.gemm_gated_pair(A, Bg, Bu, G, want, **kw)
    K.gemm_gated_product(A, Bg, Bu, got, **kw)
    assert torch.equal(got, want)


@pytest.mark.parametrize("bound", [None, 512, 1281])
@pytest.mark.parametrize("cache", [False, True])
def test_prefill_qkv_at_the_decoder_s_width(cuda, bound, cache):
    """The fused pre-attention launch at Llama-3.2-1B's own sizes: a 2048-row chunk of hidden 2048,
    32 query and 8 KV heads, whole and under the bounds a prompt leaves (512 rows: the one-head
    tiles; 1281: the 192-wide ones), against the oracle's three GEMMs, then RoPE."""
    rng = np.random.default_rng(93)
    rows, E, H, G, D, L, start = 2048, 2048, 32, 8, 64, 4096, 777
    x = bf(rng, rows, E)
    Wq, Wk, Wv = bf(rng, H * D, E, scale=0.02), bf(rng, G * D, E, scale=0.02), bf(rng, G * D, E, scale=0.02)
    table = round_bf16(ops.rope_angles(D, rows, 500000.0))
    lim = rows if bound is None else bound
    q, k, v = (ops.gemm(x[:lim], W, b_col_maj=True) for W in (Wq, Wk, Wv))
    want_q = ops.rope(q.reshape(lim * H, D), table[:lim]).reshape(lim, H * D)
    want_k = ops.rope(k.reshape(lim * G, D), table[:lim]).reshape(lim, G * D)
    if bound is not None:
        x[bound:] = np.nan
    valid = None if bound is None else word(bound, cuda)
    args = [dev(a, cuda) for a in (x, Wq, Wk, Wv, table)]
    q_out = out_like((rows, H * D), cuda, fill=7.0)
    if cache:
        keys, values = (out_like((L, G * D), cuda, fill=3.0) for _ in range(2))
        K.prefill_qkv_cache(*args, q_out, keys, values, rows=rows, hidden=E, heads=H, kv_heads=G, d=D,
                            cache_rows=L, start=word(start, cuda), valid=valid)
        k_got, v_got = from_torch(keys), from_torch(values)
        for got in (k_got, v_got):
            assert np.all(got[:start] == 3.0) and np.all(got[start + lim :] == 3.0)
        k_got, v_got = k_got[start : start + lim], v_got[start : start + lim]
    else:
        k_out, v_out = (out_like((rows, G * D), cuda, fill=7.0) for _ in range(2))
        K.prefill_qkv(*args, q_out, k_out, v_out, rows=rows, hidden=E, heads=H, kv_heads=G, d=D, valid=valid)
        k_got, v_got = from_torch(k_out), from_torch(v_out)
        assert np.all(k_got[lim:] == 7.0) and np.all(v_got[lim:] == 7.0)
        k_got, v_got = k_got[:lim], v_got[:lim]
    q_got = from_torch(q_out)
    assert np.all(q_got[lim:] == 7.0)
    close(q_got[:lim], want_q)
    close(k_got, want_k)
    close(v_got, v)


@pytest.mark.parametrize("M,Kdim,N", [(2048, 2048, 8192), (2048, 8192, 2048), (2048, 2048, 2048), (2048, 2048, 512)])
@pytest.mark.parametrize("rows", [512, 1281])
def test_prompt_chunk_projections_under_a_row_bound(cuda, M, Kdim, N, rows):
    """The launches a bounded prompt chunk takes at Llama-3.2-1B's widths (blocks choosing their tile
    by the bound, the ranges of the bound served by two launches): the plain product and the one
    with its residual, at the full depth of K, poison past the bound, nothing written past it."""
    rng = np.random.default_rng(M + Kdim + N + rows)
    A, B, R = bf(rng, M, Kdim), bf(rng, N, Kdim, scale=0.02), bf(rng, M, N)
    want = ops.gemm(A[:rows], B, b_col_maj=True)
    A[rows:] = np.nan
    C = out_like((M, N), cuda, fill=5.0)
    K.gemm(dev(A, cuda), dev(B, cuda), C, M=M, N=N, K=Kdim, b_col_maj=True, valid=word(rows, cuda))
    got = from_torch(C)
    close(got[:rows], want)
    assert np.all(got[rows:] == 5.0)
    Rd = dev(R, cuda)
    K.gemm_residual(dev(A, cuda), dev(B, cuda), Rd, Rd, M=M, N=N, K=Kdim, residual_scale=1.0, valid=word(rows, cuda))
    got = from_torch(Rd)
    # The product is rounded to bf16 before the sum, as the separate step stores it: where float32
    # sums in another order round it the other way, the sum moves by the PRODUCT's last place,
    # however small the sum itself comes out.
    total = ops.add(want, R[:rows])
    assert np.all(np.abs(got[:rows] - total) <= ATOL + RTOL * np.abs(total) + 2.0**-7 * np.abs(want))
    assert np.array_equal(got[rows:], R[rows:])


@pytest.mark.parametrize("b_col_maj", [False, True])
def test_gemm_bounded_rows_and_k_do_not_read_the_poison(cuda, b_col_maj):
    """NaN past the bounds must not reach the output (test_gemm_bounded_k.py)."""
    rng = np.random.default_rng(6)
    M, Kdim, N, rows, kv = 256, 512, 128, 150, 332
    A, B = bf(rng, M, Kdim), bf(rng, Kdim, N, scale=0.1)
    want = ops.gemm(A, B, valid_k=kv)
    A[:, kv:], B[kv:], A[rows:] = np.nan, np.nan, np.nan
    Bs = np.ascontiguousarray(B.T) if b_col_maj else B
    C = out_like((M, N), cuda, fill=5.0)
    K.gemm(dev(A, cuda), dev(Bs, cuda), C, M=M, N=N, K=Kdim, b_col_maj=b_col_maj,
           valid=word(rows, cuda), valid_k=word(kv, cuda))
    got = from_torch(C)
    close(got[:rows], want[:rows], rtol=1e-2, atol=2e-2)
    assert np.all(got[rows:] == 5.0)


@pytest.mark.parametrize("rows,cols", [(1, 2048), (8, 512), (2048, 512), (64, 5120), (7, 12288)])
@pytest.mark.parametrize("multiply", [False, True])
def test_row_broadcast_exact(cuda, rows, cols, multiply):
    rng = np.random.default_rng(70)
    x, row = bf(rng, rows, cols), bf(rng, cols)
    y = out_like((rows, cols), cuda, fill=3.0)
    bound = max(1, rows - 3)
    K.row_broadcast(dev(x, cuda), dev(row, cuda), y, rows=rows, cols=cols, multiply=multiply, valid=word(bound, cuda))
    want = (ops.mul if multiply else ops.add)(x, np.broadcast_to(row, x.shape))
    got = from_torch(y)
    assert np.array_equal(got[:bound], want[:bound])
    assert np.all(got[bound:] == 3.0)


# --------------------------------------------------------------------- rowwise
@pytest.mark.parametrize("rows,cols", [(1, 2048), (2048, 2048), (7, 64), (3, 8192), (2, 16640)])
@pytest.mark.parametrize("weighted", [False, True])
def test_rmsnorm(cuda, rows, cols, weighted):
    rng = np.random.default_rng(7)
    x = bf(rng, rows, cols)
    w = round_bf16(rng.uniform(0.9, 1.1, cols)) if weighted else None
    y = out_like((rows, cols), cuda)
    K.rmsnorm(dev(x, cuda), None if w is None else dev(w, cuda), y, rows=rows, cols=cols, eps=1e-5)
    close(y, ops.rms_norm(x, w, epsilon=1e-5))


def test_rmsnorm_bound(cuda):
    rng = np.random.default_rng(8)
    x = bf(rng, 16, 256)
    y = out_like((16, 256), cuda, fill=3.0)
    K.rmsnorm(dev(x, cuda), None, y, rows=16, cols=256, eps=1e-5, valid=word(5, cuda))
    got = from_torch(y)
    close(got[:5], ops.rms_norm(x[:5]))
    assert np.all(got[5:] == 3.0)


@pytest.mark.parametrize("rows,row,cols,angle_rows,halves", [(64, 128, 32, 2, True), (32, 64, 32, 1, True), (96, 256, 64, 96, True),
                                                             (40, 80, 16, 5, False), (2048 * 8, 64, 32, 2048, True)])
def test_rope_over_the_first_columns_of_each_row(cuda, rows, row, cols, angle_rows, halves):
    """Partial rotary: the first ``cols`` columns of a ``row``-wide row turn exactly as a row of that
    width would, the rest come through bit for bit; rows past a bound are left alone."""
    rng = np.random.default_rng(rows + row)
    x = bf(rng, rows, row)
    table = round_bf16(ops.rope_angles(cols, angle_rows + 3, 10000.0))[3:]
    bound = rows - rows // 3
    y = out_like((rows, row), cuda, fill=9.0)
    K.rope(dev(x, cuda), dev(table, cuda), y, rows=rows, cols=cols, angle_rows=angle_rows, two_halves=halves,
           valid=word(bound, cuda), row_cols=row)
    got = from_torch(y)
    want = ops.rope(x[:, :cols], table, two_halves=halves)
    close(got[:bound, :cols], want[:bound])
    assert np.array_equal(got[:bound, cols:], x[:bound, cols:]) and np.all(got[bound:] == 9.0)
    # ... and the turned columns are the bits the whole-row launch gives a row of that width
    narrow = out_like((rows, cols), cuda)
    K.rope(dev(np.ascontiguousarray(x[:, :cols]), cuda), dev(table, cuda), narrow, rows=rows, cols=cols,
           angle_rows=angle_rows, two_halves=halves)
    assert np.array_equal(got[:bound, :cols], from_torch(narrow)[:bound])


@pytest.mark.parametrize("rows,cols,weighted,bound", [(1, 2048, True, None), (64, 512, True, 40), (7, 8192, False, None)])
def test_rmsnorm_with_its_residual(cuda, rows, cols, weighted, bound):
    """The normed rows added to a residual in the norm's own pass: bit for bit the norm launch
    followed by the sum (each rounds where the other does), in place too; rows past a bound keep theirs."""
    rng = np.random.default_rng(9)
    x, r = bf(rng, rows, cols), bf(rng, rows, cols)
    w = dev(round_bf16(rng.uniform(0.9, 1.1, cols)), cuda) if weighted else None
    valid = None if bound is None else word(bound, cuda)
    lim = rows if bound is None else bound
    normed, summed = out_like((rows, cols), cuda), out_like((rows, cols), cuda, fill=3.0)
    K.rmsnorm(dev(x, cuda), w, normed, rows=rows, cols=cols, eps=1e-6)
    K.add(dev(r, cuda).reshape(-1), normed.reshape(-1), summed.reshape(-1), n=rows * cols,
          valid=None if bound is None else word(bound * cols, cuda))
    once = out_like((rows, cols), cuda, fill=3.0)
    K.rmsnorm(dev(x, cuda), w, once, rows=rows, cols=cols, eps=1e-6, valid=valid, residual=dev(r, cuda))
    assert torch.equal(once, summed)
    close(from_torch(once)[:lim], ops.add(r, ops.rms_norm(x, None if w is None else from_torch(w), epsilon=1e-6))[:lim])
    stream = dev(r, cuda)
    K.rmsnorm(dev(x, cuda), w, stream, rows=rows, cols=cols, eps=1e-6, valid=valid, residual=stream)
    assert torch.equal(stream[:lim], summed[:lim]) and np.array_equal(from_torch(stream)[lim:], r[lim:])


def angle_table(rng, angle_rows, cols):
    theta = rng.uniform(-np.pi, np.pi, (angle_rows, cols // 2))
    table = np.empty((angle_rows, cols), np.float32)
    table[:, ::2], table[:, 1::2] = np.cos(theta), np.sin(theta)
    return round_bf16(table)


@pytest.mark.parametrize("rows,cols,angle_rows", [(8, 32, 2), (1024, 32, 1), (13, 32, 13), (12, 32, 4),
                                                  (32, 64, 1), (8, 64, 1), (2048 * 32, 64, 2048),
                                                  (32, 512, 8), (64, 128, 16)])
@pytest.mark.parametrize("two_halves", [True, False])
def test_rope(cuda, rows, cols, angle_rows, two_halves):
    rng = np.random.default_rng(0)
    x, ang = bf(rng, rows, cols), angle_table(rng, angle_rows, cols)
    y = out_like((rows, cols), cuda)
    K.rope(dev(x, cuda), dev(ang, cuda), y, rows=rows, cols=cols, angle_rows=angle_rows, two_halves=two_halves)
    want = ops.rope(x, ang, two_halves=two_halves)
    got = from_torch(y)
    close(got, want)
    # Same f32 formula, one rounding: all but fused-multiply-add ties agree bit for bit.
    assert (got != want).mean() < 0.02


def test_rope_bound(cuda):
    rng = np.random.default_rng(1)
    x, ang = bf(rng, 64 * 4, 64), angle_table(rng, 64, 64)
    y = out_like((256, 64), cuda, fill=9.0)
    K.rope(dev(x, cuda), dev(ang, cuda), y, rows=256, cols=64, angle_rows=64, valid=word(40, cuda))
    got = from_torch(y)
    close(got[:40], ops.rope(x, ang)[:40])
    assert np.all(got[40:] == 9.0)


@pytest.mark.parametrize("n", [8192, 2048, 1003, 5, 2048 * 8192])
def test_elementwise(cuda, n):
    rng = np.random.default_rng(9)
    a, b = bf(rng, n, scale=3), bf(rng, n, scale=3)
    da, db = dev(a, cuda), dev(b, cuda)
    y = out_like((n,), cuda)
    K.add(da, db, y)
    assert np.array_equal(from_torch(y), ops.add(a, b))  # bit-exact (test_elementwise.py:125-132)
    K.mul(da, db, y)
    assert np.array_equal(from_torch(y), ops.mul(a, b))
    K.silu(da, y)
    close(y, ops.silu(a))
    K.silu_mul(da, db, y)
    close(y, ops.mul(ops.silu(a), b), atol=2e-2)


def test_elementwise_bound(cuda):
    rng = np.random.default_rng(10)
    a, b = bf(rng, 4096), bf(rng, 4096)
    y = out_like((4096,), cuda, fill=2.0)
    K.add(dev(a, cuda), dev(b, cuda), y, valid=word(1001, cuda))
    got = from_torch(y)
    assert np.array_equal(got[:1001], ops.add(a, b)[:1001]) and np.all(got[1001:] == 2.0)


# ------------------------------------------------------------------- attention
def run_prefill(cuda, Q, Kc, Vc, *, H, G, d, seq, seq_len, kv_len, causal=True, window=None,
                interleaved=True, valid=None, kv_valid=None, scale=None):
    O = out_like(Q.shape, cuda, fill=float("nan"))
    K.mha_prefill(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=d, seq=seq,
                  seq_len=seq_len, kv_len=kv_len, scale=scale, causal=causal, window=window,
                  q_interleaved=interleaved, kv_interleaved=interleaved,
                  valid=None if valid is None else word(valid, cuda),
                  kv_valid=None if kv_valid is None else word(kv_valid, cuda))
    want = ops.mha(Q, Kc, Vc, num_heads=H, num_KV_heads=G, seq_len=seq_len, kv_len=kv_len, d=d,
                   causal=causal, window=window, scale=scale, heads_interleaved=interleaved,
                   kv_interleaved=interleaved, valid=valid, kv_valid=kv_valid)
    return from_torch(O), want


def test_mha_prefill_longest_shape_on_sampled_queries(cuda):
    """S = 8192 (the longest of the benchmark's shapes): the whole output would take the oracle
    minutes, so every head of a sample of queries -- tile edges, both ends, random rows -- is
    checked against the oracle's attention of that one query over its keys."""
    rng = np.random.default_rng(12)
    S, H, G, d = 8192, 32, 8, 64
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, S, G, d), bf(rng, S, G, d)
    O = out_like(Q.shape, cuda, fill=float("nan"))
    K.mha_prefill(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=d, seq=S, seq_len=S,
                  kv_len=S, scale=0.125, causal=True, q_interleaved=True, kv_interleaved=True)
    got = from_torch(O)
    assert not np.isnan(got).any()
    rows = sorted({0, 1, 63, 64, 127, 128, 129, 4095, 4096, 8063, 8064, 8191, *rng.integers(0, S, 12).tolist()})
    for r in rows:
        # The query at position r attends keys 0..r: the one-query form of the same operator.
        want = ops.mha(Q[r : r + 1], Kc[: r + 1], Vc[: r + 1], num_heads=H, num_KV_heads=G, seq_len=1, kv_len=r + 1,
                       d=d, causal=True, scale=0.125, heads_interleaved=True, kv_interleaved=True)
        close(got[r : r + 1], want)


@pytest.mark.parametrize("H,G,S,window,causal", [(4, 2, 65, None, True), (4, 1, 200, 40, True), (2, 2, 1, None, True), (8, 2, 130, None, False),
                                                 (12, 4, 700, 300, True)])
def test_mha_prefill_128_wide_heads_of_short_prompts(cuda, H, G, S, window, causal):
    """d = 128 in blocks of 64 queries: one query past a block, a block of one, and masks, against the oracle."""
    rng = np.random.default_rng(S + H)
    Q, Kc, Vc = bf(rng, S, H, 128), bf(rng, S, G, 128), bf(rng, S, G, 128)
    O = out_like(Q.shape, cuda, fill=float("nan"))
    K.mha_prefill(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=128, seq=S, kv_len=S, causal=causal, window=window,
                  q_interleaved=True, kv_interleaved=True)
    got = from_torch(O)
    for r in sorted({0, S - 1, min(63, S - 1), min(64, S - 1), *rng.integers(0, S, 8).tolist()}):
        last = r + 1 if causal else S
        first = max(0, r - window) if window is not None else 0
        want = ops.mha(Q[r : r + 1], Kc[first:last], Vc[first:last], num_heads=H, num_KV_heads=G, seq_len=1, kv_len=last - first, d=128,
                       causal=False, scale=128**-0.5, heads_interleaved=True, kv_interleaved=True)
        close(got[r : r + 1], want)


@pytest.mark.parametrize("H,G,d,S,rows,L,keys,window,causal", [
    (32, 8, 64, 2048, 40, 4096, 3001, None, True),     # a turn behind a history: two groups of queries, keys that end inside a tile
    (32, 8, 64, 2048, 1, 2048, 512, None, True), (32, 8, 64, 2048, 512, 2048, 1024, None, True),   # the fewest and the most of each
    (32, 8, 64, 2048, 300, 2048, 1700, 600, True), (16, 4, 64, 128, 33, 4096, 2000, None, False),
    (12, 4, 64, 65, 65, 900, 900, 700, False), (8, 2, 128, 2048, 96, 4096, 1333, None, True),
    (32, 8, 128, 40, 40, 3000, 3000, None, True), (4, 4, 128, 256, 129, 1024, 1024, 500, True),
])
def test_mha_prefill_of_few_rows_over_many_keys(cuda, H, G, d, S, rows, L, keys, window, causal):
    """Few live queries: 32 a block, the keys dealt over its waves.  Every head of a sample of rows against the
    oracle's attention of that one query over the keys its mask leaves it; rows past the bound are zero, and NaN past
    either bound reaches nothing."""
    rng = np.random.default_rng(rows + keys)
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, L, G, d), bf(rng, L, G, d)
    Q[rows:], Kc[keys:], Vc[keys:] = np.nan, np.nan, np.nan
    O = out_like(Q.shape, cuda, fill=float("nan"))
    bounds = {} if (rows, keys) == (S, L) else dict(valid=word(rows, cuda), kv_valid=word(keys, cuda))
    K.mha_prefill(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=d, seq=S, kv_len=L, causal=causal,
                  window=window, q_interleaved=True, kv_interleaved=True, **bounds)
    got = from_torch(O)
    assert np.all(got[rows:] == 0)
    masked = causal or window is not None
    for r in sorted({0, rows - 1, min(31, rows - 1), min(32, rows - 1), *rng.integers(0, rows, 6).tolist()}):
        at = keys - rows + r   # the query's position
        last = at + 1 if causal else (min(keys, at + window + 1) if window is not None else keys)
        first = max(0, at - window) if window is not None else 0
        if not masked:
            first, last = 0, keys
        n = last - first
        want = ops.mha(Q[r : r + 1], Kc[first:last], Vc[first:last], num_heads=H, num_KV_heads=G, seq_len=1, kv_len=n, d=d,
                       causal=False, scale=d**-0.5, heads_interleaved=True, kv_interleaved=True)
        close(got[r : r + 1], want)


# Queries of 4, 3, 1 and 8 heads a KV head: one, a block of 128 (row, head) pairs and one row more, one and one that a block's edge cuts; one slice, two, as many
# as there are CUs, two blocks a CU (600 over 7000); slices that see no tile of the first queries'; windows, no mask; both layouts' strides in Q.
@pytest.mark.parametrize("H,G,d,S,rows,L,keys,window,causal", [
    (32, 8, 64, 256, 1, 4096, 3001, None, True), (32, 8, 64, 256, 32, 4096, 2560, None, True), (32, 8, 64, 256, 33, 4096, 4000, None, True),
    (24, 8, 64, 200, 43, 3000, 2999, None, True), (12, 4, 128, 130, 129, 4000, 3900, None, True), (8, 8, 128, 64, 64, 2600, 2600, None, True),
    (8, 1, 64, 64, 17, 2600, 2561, None, False), (32, 8, 64, 2048, 600, 7168, 7000, None, True), (4, 1, 64, 800, 800, 800, 800, None, True),
    (16, 4, 64, 100, 40, 4096, 4096, 1500, True), (6, 2, 64, 300, 70, 3000, 2700, 700, False), (4, 4, 64, 33, 33, 65, 65, None, True),
    (32, 8, 128, 256, 40, 9000, 8999, None, True)])
@pytest.mark.parametrize("interleaved", [True, False])
def test_mha_prefill_dealt_over_blocks(cuda, H, G, d, S, rows, L, keys, window, causal, interleaved):
    """The keys dealt over blocks and the parts' sums by way of a workspace of NaNs: every head of a sample of rows against the oracle's attention
    of that one query over the keys its mask leaves it; rows past the bound are zero, NaN past either bound reaches nothing, and the same bits again."""
    rng = np.random.default_rng(rows + keys)
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, L, G, d), bf(rng, L, G, d)
    Q[rows:], Kc[keys:], Vc[keys:] = np.nan, np.nan, np.nan
    own = (lambda x: x) if interleaved else (lambda x: np.ascontiguousarray(x.swapaxes(0, 1)))
    ws = torch.full_like(K.mha_prefill_dealt_workspace(H, G, d, cuda), float("nan"))
    outs = []
    for _ in range(2):
        O = out_like(own(Q).shape, cuda, fill=float("nan"))
        K.mha_prefill_dealt(dev(own(Q), cuda), dev(own(Kc), cuda), dev(own(Vc), cuda), O, ws, heads=H, kv_heads=G, d=d, seq=S, kv_len=L, causal=causal, window=window,
                            q_interleaved=interleaved, kv_interleaved=interleaved, valid=word(rows, cuda), kv_valid=word(keys, cuda))
        outs.append(O)
    assert torch.equal(*outs)
    got = own(from_torch(outs[0]).reshape(own(Q).shape))
    assert np.all(got[rows:] == 0)
    for r in sorted({0, rows - 1, min(31, rows - 1), min(32, rows - 1), *rng.integers(0, rows, 5).tolist()}):
        at = (keys - rows if causal or window is not None else 0) + r   # the query's position
        last = at + 1 if causal else (min(keys, at + window + 1) if window is not None else keys)
        first = max(0, at - window) if window is not None else 0
        want = ops.mha(Q[r : r + 1], Kc[first:last], Vc[first:last], num_heads=H, num_KV_heads=G, seq_len=1, kv_len=last - first, d=d,
                       causal=False, scale=d**-0.5, heads_interleaved=True, kv_interleaved=True)
        close(got[r : r + 1], want)


def test_mha_prefill_dealt_refuses_other_widths_and_small_workspaces(cuda):
    t = out_like((64 * 256,), cuda, fill=0.0)
    assert K.lib().iron_mha_prefill_dealt_workspace_bytes(4, 4, 256) == 0
    with pytest.raises(ValueError, match="workspace holds"):
        K.mha_prefill_dealt(t[: 64 * 64], t[: 64 * 64], t[: 64 * 64], t[: 64 * 64], torch.empty(16, device=cuda), heads=1, kv_heads=1, d=64, seq=64, kv_len=64)
    with pytest.raises(Exception, match="iron_mha_prefill_dealt_bf16 refused"):
        K.mha_prefill_dealt(t, t, t, t, torch.empty(16, device=cuda), heads=1, kv_heads=1, d=256, seq=64, kv_len=64)


# 128-wide heads, more queries than a block of 64 has: all of a launch's in the few-row form, with four waves a block and with eight; one
# more than that form takes; a second round of blocks that only a causal mask over the queries' own keys allows, and one it does not.
@pytest.mark.parametrize("H,G,S,rows,L,keys,window,causal", [
    (32, 8, 256, 256, 1000, 1000, None, True), (32, 8, 256, 230, 2500, 2100, None, True), (32, 8, 200, 200, 1600, 1600, None, False),
    (32, 8, 257, 257, 1600, 1600, None, True), (32, 8, 300, 270, 2000, 400, None, True),
    (32, 8, 700, 700, 700, 700, None, True), (32, 8, 640, 640, 1700, 1700, None, True), (8, 2, 2200, 2200, 2200, 2200, 1500, True),
    # more blocks than two a CU, keys dealt over two halves: one key, one tile, two, three of them, a window, no mask, rows past the bounds
    (576, 64, 1, 1, 1, 1, None, True), (576, 64, 64, 64, 64, 64, None, False), (576, 64, 65, 65, 65, 65, None, True),
    (256, 64, 300, 300, 300, 300, None, True), (288, 32, 129, 129, 190, 190, None, False), (288, 32, 129, 129, 700, 700, 200, True),
    (288, 32, 200, 131, 500, 400, None, True)])
def test_mha_prefill_128_wide_heads_at_the_lines_between_the_forms(cuda, H, G, S, rows, L, keys, window, causal):
    test_mha_prefill_of_few_rows_over_many_keys(cuda, H, G, 128, S, rows, L, keys, window, causal)


@pytest.mark.parametrize("H,G,S", [(32, 8, 2305), (16, 4, 5000), (32, 32, 4096)])   # 608, 640 and 1024 blocks of 128 queries
def test_mha_prefill_128_wide_heads_keep_a_reference_for_each_half_of_the_tiles(cuda, H, G, S):
    """Every query sees one key of the first tile at a score of 0 and a value of 0, one of the second at a score of its own and a value of
    1, and others out of sight of both.  With a reference for the even tiles and one for the odd, both weights are exactly 1 in the products and the
    sums join in float32, so the answer w / (1 + w) is off by its own rounding alone (half a step of bf16, 2^-8 of its power of
    two) and float32's; with one reference w itself is rounded to bf16 first, half a step more."""
    rng = np.random.default_rng(S)
    Q, Kc, Vc = np.zeros((S, H, 128), np.float32), np.zeros((S, G, 128), np.float32), np.zeros((S, G, 128), np.float32)
    Q[..., 0] = round_bf16(rng.uniform(0.1, 3.0, (S, H)).astype(np.float32))
    Q[..., 1] = 1.0
    Kc[..., 1] = -300.0
    Kc[5, :, 1] = 0.0
    Kc[70, :, 0], Kc[70, :, 1] = -1.0, 0.0
    Vc[70] = 1.0
    O = out_like(Q.shape, cuda, fill=float("nan"))
    K.mha_prefill(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=128, seq=S, kv_len=S, scale=1.0, causal=True,
                  q_interleaved=True, kv_interleaved=True)
    w = np.exp(-Q[71:, :, 0].astype(np.float64))
    want = w / (1 + w)
    err = np.abs(from_torch(O)[71:].astype(np.float64) - want[..., None])
    step = 2.0 ** (np.floor(np.log2(want)) - 7)
    assert np.all(err <= (0.5 * step + 2.0**-18 * want)[..., None]), f"{(err > (0.5 * step + 2.0**-18 * want)[..., None]).mean():.3f} are off by more"


# 600 and 832 blocks of 128 queries, four waves each (and one query past a block); windows of 1024 and 513 keys, 528 and 1020 blocks.
@pytest.mark.parametrize("H,G,S,window", [(40, 8, 1900, None), (32, 8, 3201, None), (16, 4, 4170, 1023), (60, 4, 2100, 512)])
def test_mha_prefill_128_wide_heads_first_tiles_weights_in_two_terms(cuda, H, G, S, window):
    """As above by one reference a query: the two weights lie in the first two tiles, whose weights keep what bf16 leaves of them, so the answer is off by its own
    rounding (half a step) and by the 2^-18 of a weight that two terms leave."""
    rng = np.random.default_rng(S)
    Q, Kc, Vc = np.zeros((S, H, 128), np.float32), np.zeros((S, G, 128), np.float32), np.zeros((S, G, 128), np.float32)
    Q[..., 0] = round_bf16(rng.uniform(0.1, 3.0, (S, H)).astype(np.float32))
    Q[..., 1] = 1.0
    Kc[..., 1] = -300.0
    Kc[5, :, 1] = 0.0
    Kc[70, :, 0], Kc[70, :, 1] = -1.0, 0.0
    Vc[70] = 1.0
    O = out_like(Q.shape, cuda, fill=float("nan"))
    K.mha_prefill(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=128, seq=S, kv_len=S, scale=1.0, causal=True, window=window,
                  q_interleaved=True, kv_interleaved=True)
    got, last = from_torch(O).astype(np.float64), S if window is None else window + 6   # (past them the first key is out of sight)
    w = np.exp(-Q[71:last, :, 0].astype(np.float64))
    want = w / (1 + w)
    step = 2.0 ** (np.floor(np.log2(want)) - 7)
    assert np.all(np.abs(got[71:last] - want[..., None]) <= (0.5 * step + 2.0**-17 * want)[..., None])
    assert not np.isnan(got).any() and np.all(got[:70] == 0) and (window is None or np.all(got[71 + window:] == 0))


# Launches of more than 1024 blocks, four waves each, which read a tile's keys ahead and refill their place at the next step: one key, one tile and one
# key more, two tiles, three and four (the first refill, the last step's reads past the end), a window, no mask, rows past the bounds.
@pytest.mark.parametrize("H,G,S,rows,L,keys,window,causal", [
    (1088, 64, 1, 1, 1, 1, None, True), (1088, 64, 64, 64, 64, 64, None, False), (1088, 64, 65, 65, 65, 65, None, True),
    (1088, 32, 128, 128, 128, 128, None, True), (1088, 32, 97, 97, 192, 192, None, False), (1088, 32, 100, 100, 250, 250, None, True),
    (544, 32, 300, 300, 300, 300, 100, True), (544, 32, 200, 131, 450, 400, None, True)])
def test_mha_prefill_128_wide_heads_whose_keys_are_read_a_tile_ahead(cuda, H, G, S, rows, L, keys, window, causal):
    test_mha_prefill_of_few_rows_over_many_keys(cuda, H, G, 128, S, rows, L, keys, window, causal)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("interleaved", [True, False])
def test_mha_prefill_of_few_rows_in_both_layouts_and_a_window_of_a_buffer(cuda, d, interleaved):
    """The few-row form over keys stored head by head or row by row, and over a run of a longer buffer's rows: the same bits."""
    rng = np.random.default_rng(d)
    H, G, S, L, first, rows, keys = 8, 2, 512, 1024, 37, 45, 800
    Q, Kc, Vc = (torch.from_numpy(x).to(cuda).bfloat16() for x in (bf(rng, S, H, d), bf(rng, L, G, d), bf(rng, L, G, d)))
    kw = dict(heads=H, kv_heads=G, d=d, seq=S, kv_len=L, valid=word(rows, cuda), kv_valid=word(keys, cuda))
    plain, other = torch.empty_like(Q), torch.empty_like(Q)
    K.mha_prefill(Q, Kc, Vc, plain, q_interleaved=True, kv_interleaved=True, **kw)
    want = ops.mha(from_torch(Q)[44:45], from_torch(Kc)[:keys], from_torch(Vc)[:keys], num_heads=H, num_KV_heads=G, seq_len=1, kv_len=keys, d=d,
                   causal=False, scale=d**-0.5, heads_interleaved=True, kv_interleaved=True)
    close(from_torch(plain)[44:45], want)
    if interleaved:
        held = [torch.full((L + 100, G, d), float("nan"), dtype=torch.bfloat16, device=cuda) for _ in range(2)]
        for buf, x in zip(held, (Kc, Vc)):
            buf[first : first + L] = x
        K.mha_prefill(Q, *held, other, q_interleaved=True, kv_interleaved=True, kv_first=word(first, cuda), kv_rows=L + 100, **kw)
    else:
        by_head = torch.empty(H, S, d, dtype=torch.bfloat16, device=cuda)
        K.mha_prefill(Q.transpose(0, 1).contiguous(), Kc.transpose(0, 1).contiguous(), Vc.transpose(0, 1).contiguous(), by_head,
                      q_interleaved=False, kv_interleaved=False, **kw)
        other = by_head.transpose(0, 1)
    assert torch.equal(plain, other)


@pytest.mark.parametrize("rows", [512, 1500])
def test_mha_prefill_bounded_chunk_at_the_decoder_s_width(cuda, rows):
    """A 2048-row prompt chunk of 32 heads under row and key bounds read on the device (512 rows
    as the benchmark's prompt leaves, and 1500): every head of a sample of rows against the oracle's
    one-query attention over the keys before it; the rows past the bound are zero, and NaN there
    reaches nothing."""
    rng = np.random.default_rng(rows)
    S, H, G, d = 2048, 32, 8, 64
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, S, G, d), bf(rng, S, G, d)
    Q[rows:], Kc[rows:], Vc[rows:] = np.nan, np.nan, np.nan
    O = out_like(Q.shape, cuda, fill=float("nan"))
    K.mha_prefill(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=d, seq=S, seq_len=S,
                  kv_len=S, scale=0.125, causal=True, q_interleaved=True, kv_interleaved=True,
                  valid=word(rows, cuda), kv_valid=word(rows, cuda))
    got = from_torch(O)
    assert np.all(got[rows:] == 0)
    assert not np.isnan(got[:rows]).any()
    for r in sorted({0, 1, 31, 32, 63, 64, 65, 127, 128, 129, rows - 65, rows - 64, rows - 1, *rng.integers(0, rows, 10).tolist()}):
        want = ops.mha(Q[r : r + 1], Kc[: r + 1], Vc[: r + 1], num_heads=H, num_KV_heads=G, seq_len=1, kv_len=r + 1,
                       d=d, causal=True, scale=0.125, heads_interleaved=True, kv_interleaved=True)
        close(got[r : r + 1], want)


@pytest.mark.parametrize("S", [512, 2048])
def test_mha_prefill_llama_shape(cuda, S):
    rng = np.random.default_rng(11)
    H, G, d = 32, 8, 64
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, S, G, d), bf(rng, S, G, d)
    got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=S, seq_len=S, kv_len=S, scale=0.125)
    close(got, want)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("shape", ["huge_range", "rising", "falling", "constant", "far_below_zero", "far_above_zero"])
def test_mha_prefill_scores_that_move_the_softmax_reference(cuda, d, shape):
    """The exponentials are taken against a reference that follows the maxima lazily, and a tile is
    first tried without taking its maximum at all: scores spread over hundreds of doublings, scores
    that rise or fall along the keys by far more than float32's exponent range holds, equal scores,
    and scores all far below or far above zero (where a reference of zero would under- or overflow)
    against the oracle's softmax, causal and not, over many tiles."""
    rng = np.random.default_rng(len(shape) + d)
    H, G, S = 4, 2, 1100
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, S, G, d), bf(rng, S, G, d)
    ramp = np.linspace(0.0, 1.0, S, dtype=np.float32)[:, None, None]
    scale = None
    if shape == "huge_range":
        Q, Kc = round_bf16(Q * 6), round_bf16(Kc * 6)            # scaled scores of a few hundred either way
    elif shape in ("rising", "falling"):
        # one direction of the head carries a score that climbs (or drops) by ~1500 along the keys
        Q[..., 0] = 8.0
        Kc[..., 0] = round_bf16((ramp if shape == "rising" else 1 - ramp) * 190.0)[..., 0]
        scale = 1.0
    elif shape == "constant":
        Q[:], Kc[:] = 0.0, 0.0
    else:
        Q[..., 0] = 16.0
        Kc[..., 0] = -40.0 if shape == "far_below_zero" else 40.0   # every score near -640 / +640 before the scale
        scale = 1.0
    for causal in (True, False):
        got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=S, seq_len=S, kv_len=S, causal=causal, scale=scale)
        assert not np.isnan(got).any()
        close(got, want)


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("causal,window", [(True, None), (True, 100), (False, 70), (False, None)])
def test_mha_prefill_masks_and_layouts(cuda, causal, window, interleaved):
    rng = np.random.default_rng(12)
    H, G, d, S, L = 8, 2, 64, 192, 448
    qs = (S, H, d) if interleaved else (H, S, d)
    ks = (L, G, d) if interleaved else (G, L, d)
    Q, Kc, Vc = bf(rng, *qs), bf(rng, *ks), bf(rng, *ks)
    got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=S, seq_len=S, kv_len=L, causal=causal,
                            window=window, interleaved=interleaved)
    close(got, want)


def test_mha_prefill_chunk_over_cache_bounded(cuda):
    """A prompt chunk: `valid` of 256 rows at the end of `kv_valid` keys of a longer cache; NaN
    past the bounds must not reach the output and padding rows are exactly zero
    (test_mha_bounded_rows.py:98-102,197-225)."""
    rng = np.random.default_rng(13)
    H, G, d, C, L = 8, 2, 64, 256, 1024
    rows, kv = 150, 600
    Q, Kc, Vc = bf(rng, C, H, d), bf(rng, L, G, d), bf(rng, L, G, d)
    Q[rows:], Kc[kv:], Vc[kv:] = np.nan, np.nan, np.nan
    got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=C, seq_len=C, kv_len=L, valid=rows, kv_valid=kv)
    assert np.all(got[rows:] == 0)
    close(got[:rows], want[:rows])


def test_mha_prefill_d128_and_ragged_seq(cuda):
    rng = np.random.default_rng(14)
    H, G, d, S = 6, 2, 128, 200
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, S, G, d), bf(rng, S, G, d)
    got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=S, seq_len=S, kv_len=S)
    close(got, want)


def test_mha_prefill_d256_ragged_windowed_and_bounded(cuda):
    """256-wide heads (a global layer's of a toy Gemma 4): a ragged causal sequence, a window, and a
    prompt chunk bounded by device words at the end of a longer cache, unscaled as Gemma attends."""
    rng = np.random.default_rng(21)
    H, G, d, S = 4, 1, 256, 200
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, S, G, d), bf(rng, S, G, d)
    for window in (None, 37):
        got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=S, seq_len=S, kv_len=S, window=window)
        close(got, want)
    C, L, rows, kv = 64, 512, 40, 300
    Q, Kc, Vc = bf(rng, C, H, d) * 0.25, bf(rng, L, G, d) * 0.25, bf(rng, L, G, d)
    Q[rows:], Kc[kv:], Vc[kv:] = np.nan, np.nan, np.nan
    got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=C, seq_len=C, kv_len=L, valid=rows, kv_valid=kv,
                            scale=1.0)
    assert np.all(got[rows:] == 0)
    close(got[:rows], want[:rows])


@pytest.mark.parametrize("d,H,G,S,window", [(512, 32, 8, 2048, None), (256, 32, 8, 2048, 300), (256, 32, 4, 4096, None),
                                             (512, 16, 16, 1100, None)])
def test_mha_prefill_wide_heads_at_every_block_shape_on_sampled_queries(cuda, d, H, G, S, window):
    """256- and 512-wide heads where the launch has blocks enough for its larger shapes (128-query
    blocks of eight waves; at 256 two query groups a wave from a thousand blocks on): the whole
    output would take the oracle minutes, so every head of a sample of queries -- tile and block
    edges, both ends, random rows -- is checked against the oracle's attention of that one query."""
    rng = np.random.default_rng(d + S)
    Q, Kc, Vc = bf(rng, S, H, d) * 0.25, bf(rng, S, G, d) * 0.25, bf(rng, S, G, d)
    O = out_like(Q.shape, cuda, fill=float("nan"))
    K.mha_prefill(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=d, seq=S, seq_len=S,
                  kv_len=S, scale=1.0, causal=True, window=window, q_interleaved=True, kv_interleaved=True)
    got = from_torch(O)
    assert not np.isnan(got).any()
    for r in sorted({0, 1, 15, 16, 31, 32, 33, 63, 64, 127, 128, 129, 255, 256, S - 129, S - 128, S - 1,
                     *rng.integers(0, S, 8).tolist()}):
        lo = 0 if window is None else max(0, r - window)
        want = ops.mha(Q[r : r + 1], Kc[lo : r + 1], Vc[lo : r + 1], num_heads=H, num_KV_heads=G, seq_len=1,
                       kv_len=r + 1 - lo, d=d, causal=True, scale=1.0, heads_interleaved=True, kv_interleaved=True)
        close(got[r : r + 1], want)


@pytest.mark.parametrize("interleaved", [True, False])
def test_mha_prefill_512_wide_heads_over_many_tiles(cuda, interleaved):
    """512-wide heads past a block's 64 queries and a tile's 32 keys: several heads a KV head, a ragged
    causal sequence, a window that drops whole tiles, no mask at all, a chunk at the end of a longer
    cache under bounds on both sides, and an unscaled product."""
    rng = np.random.default_rng(24)
    H, G, d, S = 4, 2, 512, 333
    Q, Kc, Vc = bf(rng, S, H, d) * 0.25, bf(rng, S, G, d) * 0.25, bf(rng, S, G, d)
    if not interleaved:
        Q, Kc, Vc = (np.ascontiguousarray(a.transpose(1, 0, 2)) for a in (Q, Kc, Vc))
    for causal, window in ((True, None), (True, 70), (False, 45), (False, None)):
        got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=S, seq_len=S, kv_len=S, causal=causal,
                                window=window, interleaved=interleaved)
        close(got, want)
    C, L, rows, kv = 192, 700, 130, 611
    Q, Kc, Vc = bf(rng, C, H, d) * 0.25, bf(rng, L, G, d) * 0.25, bf(rng, L, G, d)
    Q[rows:], Kc[kv:], Vc[kv:] = np.nan, np.nan, np.nan
    if not interleaved:
        Q, Kc, Vc = (np.ascontiguousarray(a.transpose(1, 0, 2)) for a in (Q, Kc, Vc))
    got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=C, seq_len=C, kv_len=L, valid=rows, kv_valid=kv,
                            scale=1.0, interleaved=interleaved)
    if interleaved:
        assert np.all(got[rows:] == 0)
        close(got[:rows], want[:rows])
    else:
        assert np.all(got[:, rows:] == 0)
        close(got[:, :rows], want[:, :rows])


@pytest.mark.parametrize("d,H,G", [(64, 8, 2), (128, 4, 1), (256, 4, 1), (512, 4, 1)])
def test_mha_over_a_window_of_a_longer_buffer(cuda, d, H, G):
    """Keys that are a run of rows of a longer buffer, from a row a device word names (a ring cache's
    window): the launch that is handed those rows as tensors of their own, bit for bit; the buffer's
    other rows (NaN here) reach nothing, and a word past the end is held inside the buffer."""
    rng = np.random.default_rng(23)
    rows, L, S = 300, 96, 64
    Kb, Vb = bf(rng, rows, G, d) * 0.25, bf(rng, rows, G, d)
    Q = bf(rng, S, H, d) * 0.25
    ws = K.mha_decode_workspace(H, d, cuda)
    for first, kv_valid in ((0, 96), (37, 80), (204, 96), (1000, 70)):
        held = max(0, min(first, rows - L))
        Kw, Vw = Kb[held : held + L].copy(), Vb[held : held + L].copy()
        Kp, Vp = np.full_like(Kb, np.nan), np.full_like(Vb, np.nan)
        Kp[held : held + kv_valid], Vp[held : held + kv_valid] = Kb[held : held + kv_valid], Vb[held : held + kv_valid]
        for window in (None, 20):
            own = out_like((S, H, d), cuda)
            K.mha_prefill(dev(Q, cuda), dev(Kw, cuda), dev(Vw, cuda), own, heads=H, kv_heads=G, d=d, seq=S, kv_len=L,
                          scale=1.0, window=window, q_interleaved=True, kv_interleaved=True, kv_valid=word(kv_valid, cuda))
            at = out_like((S, H, d), cuda, fill=float("nan"))
            K.mha_prefill(dev(Q, cuda), dev(Kp, cuda), dev(Vp, cuda), at, heads=H, kv_heads=G, d=d, seq=S, kv_len=L,
                          scale=1.0, window=window, q_interleaved=True, kv_interleaved=True, kv_valid=word(kv_valid, cuda),
                          kv_first=word(first, cuda), kv_rows=rows)
            assert torch.equal(own, at), (first, kv_valid, window)
            own1, at1 = out_like((1, H, d), cuda), out_like((1, H, d), cuda, fill=float("nan"))
            K.mha_decode(dev(Q[:1], cuda), dev(Kw, cuda), dev(Vw, cuda), own1, heads=H, kv_heads=G, d=d, kv_len=L, scale=1.0,
                         window=window, kv_interleaved=True, kv_valid=word(kv_valid, cuda), workspace=ws)
            K.mha_decode(dev(Q[:1], cuda), dev(Kp, cuda), dev(Vp, cuda), at1, heads=H, kv_heads=G, d=d, kv_len=L, scale=1.0,
                         window=window, kv_interleaved=True, kv_valid=word(kv_valid, cuda), workspace=ws,
                         kv_first=word(first, cuda), kv_rows=rows)
            assert torch.equal(own1, at1), (first, kv_valid, window)
    # ... and the long-cache kernel (splits and their merge) over a window.
    if d == 64:
        rows, L = 6000, 4096
        Kb, Vb, q = bf(rng, rows, G, d), bf(rng, rows, G, d), bf(rng, 1, H, d)
        own1, at1 = out_like((1, H, d), cuda), out_like((1, H, d), cuda)
        K.mha_decode(q_t := dev(q, cuda), dev(Kb[1500:5596], cuda), dev(Vb[1500:5596], cuda), own1, heads=H, kv_heads=G, d=d,
                     kv_len=L, kv_interleaved=True, kv_valid=word(3000, cuda), workspace=ws)
        K.mha_decode(q_t, dev(Kb, cuda), dev(Vb, cuda), at1, heads=H, kv_heads=G, d=d, kv_len=L, kv_interleaved=True,
                     kv_valid=word(3000, cuda), workspace=ws, kv_first=word(1500, cuda), kv_rows=rows)
        assert torch.equal(own1, at1)
    with pytest.raises(ValueError, match="row by row"):
        K.mha_decode(dev(Q[:1], cuda), dev(Kb, cuda), dev(Vb, cuda), out_like((1, H, d), cuda), heads=H, kv_heads=G, d=d,
                     kv_len=96, kv_interleaved=False, workspace=ws, kv_first=word(0, cuda), kv_rows=300)


def test_mha_512_wide_heads_prefill_and_decode(cuda):
    """512-wide heads (a global layer's of Gemma 4): the prompt kernel under every mask and a bound,
    and the one-query kernel on either side of 2048 keys."""
    rng = np.random.default_rng(22)
    H, G, d, S, L = 4, 1, 512, 70, 200
    Q, Kc, Vc = bf(rng, S, H, d) * 0.25, bf(rng, L, G, d) * 0.25, bf(rng, L, G, d)
    for causal, window in ((True, None), (True, 37), (False, 20), (False, None)):
        got, want = run_prefill(cuda, Q, Kc, Vc, H=H, G=G, d=d, seq=S, seq_len=S, kv_len=L, causal=causal,
                                window=window, scale=1.0)
        close(got, want)
    Qp, Kp, Vp = Q.copy(), Kc.copy(), Vc.copy()
    Qp[40:], Kp[150:], Vp[150:] = np.nan, np.nan, np.nan
    got, want = run_prefill(cuda, Qp, Kp, Vp, H=H, G=G, d=d, seq=S, seq_len=S, kv_len=L, valid=40, kv_valid=150, scale=1.0)
    assert np.all(got[40:] == 0)
    close(got[:40], want[:40])
    for L, kv_valid, window in ((300, 257, None), (4096, 3000, None), (4096, 3000, 99)):
        H, G = 8, 2
        Q, Kc, Vc = bf(rng, 1, H, d) * 0.25, bf(rng, L, G, d) * 0.25, bf(rng, L, G, d)
        Kc[kv_valid:], Vc[kv_valid:] = np.nan, np.nan
        O = out_like((1, H, d), cuda, fill=float("nan"))
        K.mha_decode(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=d, kv_len=L, scale=1.0,
                     window=window, kv_interleaved=True, kv_valid=word(kv_valid, cuda),
                     workspace=K.mha_decode_workspace(H, d, cuda))
        want = ops.mha(Q, Kc, Vc, num_heads=H, num_KV_heads=G, seq_len=1, kv_len=L, d=d, scale=1.0, window=window,
                       heads_interleaved=True, kv_interleaved=True, kv_valid=kv_valid)
        close(O, want)


@pytest.mark.parametrize("E,H,G,d", [(2048, 32, 8, 64), (1000, 3, 1, 128), (4096, 8, 2, 128)])
def test_decode_qkv_reading_its_row_from_the_embedding_table(cuda, E, H, G, d):
    """A token's first layer: the fused q/k/v launch handed the embedding table and the word that names
    the row, against the same launch handed the row itself -- every output bit for bit, the row left
    in ``x`` for the residual sum, and a word past either end of the table held inside it."""
    rng = np.random.default_rng(E + d)
    vocab, L, pos = 77, 16, 9
    table, g = bf(rng, vocab, E), round_bf16(rng.uniform(0.9, 1.1, E).astype(np.float32))
    Wq, Wk, Wv = bf(rng, H * d, E, scale=0.02), bf(rng, G * d, E, scale=0.02), bf(rng, G * d, E, scale=0.02)
    angles = round_bf16(ops.rope_angles(d, L))
    dt, dg, dq, dk, dv, da = (dev(a, cuda) for a in (table, g, Wq, Wk, Wv, angles))
    position, angle_row = word(pos, cuda), word(pos, cuda)
    for token in (0, 41, vocab - 1, vocab + 5, -3):
        held = min(max(token, 0), vocab - 1)
        want_q, want_k, want_v = out_like((H * d,), cuda), out_like((L, G, d), cuda, fill=2.0), out_like((L, G, d), cuda, fill=2.0)
        K.decode_qkv(dev(table[held], cuda), dg, dq, dk, dv, da, want_q, want_k, want_v, eps=1e-5, hidden=E, heads=H,
                     kv_heads=G, d=d, cache_rows=L, position=position, angle_row=angle_row)
        x = out_like((E,), cuda, fill=float("nan"))
        got_q, got_k, got_v = out_like((H * d,), cuda), out_like((L, G, d), cuda, fill=2.0), out_like((L, G, d), cuda, fill=2.0)
        K.decode_qkv(x, dg, dq, dk, dv, da, got_q, got_k, got_v, eps=1e-5, hidden=E, heads=H, kv_heads=G, d=d,
                     cache_rows=L, position=position, angle_row=angle_row, table=dt, token=word(token, cuda))
        assert torch.equal(got_q, want_q) and torch.equal(got_k, want_k) and torch.equal(got_v, want_v), token
        assert np.array_equal(from_torch(x), table[held]), token


@pytest.mark.parametrize("H,G,d,rotary,ring,own_kv", [(4, 1, 128, 128, True, True), (4, 1, 256, 64, False, True),
                                                       (8, 2, 512, 512, True, True), (4, 1, 128, 128, False, False),
                                                       (16, 8, 64, 64, False, True)])
def test_decode_heads_is_the_separate_launches_bit_for_bit(cuda, H, G, d, rotary, ring, own_kv):
    """What lies between a token's projections and its attention where heads are normed one by one:
    per-head RMSNorm of q and k (gains) and v (none), RoPE on q and k (all of a head's columns, or the
    leading ones), k's and v's rows into their caches (twice for a ring) -- one launch against the
    launches of the separate operators bit for bit, and q's norm against the oracle."""
    rng = np.random.default_rng(H + d)
    rows = 24
    q, k, v = bf(rng, H, d), bf(rng, G, d), bf(rng, G, d)
    gq, gk = bf(rng, d, scale=0.3) + 1, bf(rng, d, scale=0.3) + 1
    angles = bf(rng, 1, rotary)
    dq, dk, dv, dgq, dgk, da = (dev(x, cuda) for x in (q, k, v, round_bf16(gq), round_bf16(gk), angles))
    # the separate launches
    def normed(x, gain, n):
        y = out_like((n, d), cuda)
        K.rmsnorm(x, gain, y, rows=n, cols=d, eps=1e-6)
        return y

    def roped(x, n):
        y = out_like((n, d), cuda)
        K.rope(x, da, y, rows=n, cols=rotary, angle_rows=1, row_cols=d)
        return y

    want_q = roped(normed(dq, dgq, H), H)
    close(normed(dq, dgq, H), ops.rms_norm(q, round_bf16(gq), epsilon=1e-6))
    row0, row1 = word(5, cuda), word(5 + rows // 2, cuda)
    got_q = out_like((H, d), cuda, fill=float("nan"))
    if not own_kv:
        K.decode_heads(dq, got_q, heads=H, kv_heads=G, d=d, eps=1e-6, norms=1, q_gain=dgq, q_angles=da, rotary=rotary)
        assert torch.equal(got_q, want_q)
        return
    want_k, want_v = roped(normed(dk, dgk, G), G), normed(dv, None, G)
    keys, values = out_like((rows, G, d), cuda, fill=3.0), out_like((rows, G, d), cuda, fill=3.0)
    K.decode_heads(dq, got_q, heads=H, kv_heads=G, d=d, eps=1e-6, norms=7, k=dk, v=dv, q_gain=dgq, k_gain=dgk,
                   q_angles=da, k_angles=da, rotary=rotary, keys=keys, values=values, row0=row0,
                   row1=row1 if ring else None, cache_rows=rows)
    assert torch.equal(got_q, want_q)
    held = [5, 5 + rows // 2] if ring else [5]
    for r in range(rows):
        if r in held:
            assert torch.equal(keys[r], want_k) and torch.equal(values[r], want_v), r
        else:
            assert bool((keys[r] == 3.0).all()) and bool((values[r] == 3.0).all()), r


@pytest.mark.parametrize("M,Kdim", [(128, 512), (256, 2048), (3000, 1536), (128, 8192)])
@pytest.mark.parametrize("activation", ["gelu_tanh", "silu"])
def test_gemv_with_an_activation_and_a_row_in_its_epilogue(cuda, M, Kdim, activation):
    """A projection of one row, its activation and the product with a given row (Gemma 4's per-layer
    input gate) in one launch: link by link against the oracle, and bit for bit against this library's
    own separate launches."""
    rng = np.random.default_rng(M + Kdim)
    W, x, row = bf(rng, M, Kdim, scale=0.05), bf(rng, Kdim), bf(rng, M)
    dW, dx, drow = dev(W, cuda), dev(x, cuda), dev(row, cuda)
    y = out_like((M,), cuda)
    K.gemv_fused(dW, dx, y, M=M, K=Kdim, residual=drow, epilogue=4 if activation == "gelu_tanh" else 5)
    u, a, want = out_like((M,), cuda), out_like((M,), cuda), out_like((M,), cuda)
    K.gemv(dW, dx, u, M=M, K=Kdim)
    close(u, ops.gemv(W, x))
    if activation == "gelu_tanh":
        K.unary(u, a, "gelu_tanh", n=M)
        close(a, ops.gelu(from_torch(u), approximate="tanh"))
    else:
        K.silu(u, a, n=M)
        close(a, ops.silu(from_torch(u)))
    K.mul(a, drow, want, n=M)
    assert torch.equal(y, want)


@pytest.mark.parametrize("L", [1024, 4096, 16384])
def test_mha_decode_llama_shape(cuda, L):
    rng = np.random.default_rng(15)
    H, G, d = 32, 8, 64
    Q, Kc, Vc = bf(rng, 1, H, d), bf(rng, L, G, d), bf(rng, L, G, d)
    O = out_like((1, H, d), cuda, fill=float("nan"))
    ws = K.mha_decode_workspace(H, d, cuda)
    K.mha_decode(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=d, kv_len=L,
                 scale=0.125, kv_interleaved=True, workspace=ws)
    want = ops.mha(Q, Kc, Vc, num_heads=H, num_KV_heads=G, seq_len=1, kv_len=L, d=d, scale=0.125,
                   heads_interleaved=True, kv_interleaved=True)
    close(O, want)


def test_mha_decode_is_as_accurate_deep_in_a_32k_cache_as_near_its_start(cuda):
    """The reference's long-context check (iron/tests/operators/test_mha_long_context.py:45-62): one
    query of Llama-3.2-1B's packed heads over a 32768-row cache of 55 distinct rows tiled over its
    length (every key block weighs alike and the outputs stay far from 0, so a running sum that loses
    a block's share shows), at positions 1023 and 32703, within 4 % of the output's peak -- and,
    float32 sums losing nothing of the kind here, within the stated bf16 tolerance as well."""
    rng = np.random.default_rng(0)
    H, G, d, L, distinct = 32, 8, 64, 32768, 55
    Kc = round_bf16(np.resize(rng.standard_normal((distinct, G, d)) * 2, (L, G, d)).astype(np.float32))
    Vc = round_bf16(np.resize(rng.standard_normal((distinct, G, d)), (L, G, d)).astype(np.float32))
    Q = round_bf16(rng.standard_normal((1, H, d)).astype(np.float32))
    ws = K.mha_decode_workspace(H, d, cuda)
    Kd, Vd, Qd = dev(Kc, cuda), dev(Vc, cuda), dev(Q, cuda)
    for position in (1023, L - 65):
        O = out_like((1, H, d), cuda, fill=float("nan"))
        K.mha_decode(Qd, Kd, Vd, O, heads=H, kv_heads=G, d=d, kv_len=L, kv_interleaved=True,
                     kv_valid=word(position + 1, cuda), workspace=ws)
        want = ops.mha(Q, Kc, Vc, num_heads=H, num_KV_heads=G, seq_len=1, kv_len=L, d=d, heads_interleaved=True,
                       kv_interleaved=True, kv_valid=position + 1)
        got = from_torch(O).reshape(want.shape)
        peak = float(np.abs(want).max())
        assert peak > 0.5 and np.abs(got - want).max() <= 0.04 * peak, (position, np.abs(got - want).max(), peak)
        close(got, want)


@pytest.mark.parametrize("H,G,d", [(32, 8, 64), (8, 8, 64), (24, 8, 128), (40, 8, 64), (4, 1, 256), (16, 8, 64), (12, 2, 64), (3, 1, 64)])
@pytest.mark.parametrize("kv_valid,window", [(1, None), (77, None), (700, None), (700, 99), (2048, 511)])
@pytest.mark.parametrize("L", [2048, 4096])  # the one-launch kernel, and the split one with its merge
def test_mha_decode_bounds_windows_groups(cuda, H, G, d, kv_valid, window, L):
    rng = np.random.default_rng(16)
    for interleaved in (True, False):
        ks = (L, G, d) if interleaved else (G, L, d)
        Q, Kc, Vc = bf(rng, 1, H, d), bf(rng, *ks), bf(rng, *ks)
        if interleaved:
            Kc[kv_valid:], Vc[kv_valid:] = np.nan, np.nan
        else:
            Kc[:, kv_valid:], Vc[:, kv_valid:] = np.nan, np.nan
        O = out_like((1, H, d), cuda, fill=float("nan"))
        ws = K.mha_decode_workspace(H, d, cuda)
        K.mha_decode(dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda), O, heads=H, kv_heads=G, d=d, kv_len=L,
                     window=window, kv_interleaved=interleaved, kv_valid=word(kv_valid, cuda), workspace=ws)
        want = ops.mha(Q, Kc, Vc, num_heads=H, num_KV_heads=G, seq_len=1, kv_len=L, d=d, window=window,
                       heads_interleaved=True, kv_interleaved=interleaved, kv_valid=kv_valid)
        close(O, want)


@pytest.mark.parametrize("H,G,d", [(32, 8, 64), (16, 1, 64), (7, 7, 64), (24, 8, 128), (26, 2, 128)])
@pytest.mark.parametrize("form,short_keys", [(1, 0), (2, 0), (2, 48)])
def test_mha_decode_every_form_at_every_context(cuda, H, G, d, form, short_keys):
    """The lane-per-column scans, and the one-shape launch both as a block a query head (few keys) and
    as runs of keys dealt over the chip with a merge behind (forced onto small contexts by
    ``short_keys``): contexts that end inside a wave's 16-key tile, at a run's edge and at the cache's
    last row; windows; rows past the bound and the whole workspace poisoned."""
    if form == 1 and H // G not in (1, 2, 3, 4, 5, 6, 8):
        pytest.skip("the lane-scan kernels take 1, 2, 3, 4, 5, 6 or 8 query heads a KV head")
    rng = np.random.default_rng(161)
    L = 3000
    Q, Kc, Vc = bf(rng, 1, H, d), bf(rng, L, G, d), bf(rng, L, G, d)
    dQ = dev(Q, cuda)
    ws = K.mha_decode_workspace(H, d, cuda)
    for kv_valid, window in ((1, None), (17, None), (48, None), (49, None), (777, None), (2049, None), (3000, None),
                             (2500, 100), (2500, 1500), (3000, 2999)):
        Kp, Vp = Kc.copy(), Vc.copy()
        Kp[kv_valid:], Vp[kv_valid:] = np.nan, np.nan
        ws.fill_(float("nan"))
        O = out_like((1, H, d), cuda, fill=float("nan"))
        K.mha_decode(dQ, dev(Kp, cuda), dev(Vp, cuda), O, heads=H, kv_heads=G, d=d, kv_len=L, window=window,
                     kv_interleaved=True, kv_valid=word(kv_valid, cuda), workspace=ws, form=form, short_keys=short_keys)
        want = ops.mha(Q, Kp, Vp, num_heads=H, num_KV_heads=G, seq_len=1, kv_len=L, d=d, window=window,
                       heads_interleaved=True, kv_interleaved=True, kv_valid=kv_valid)
        close(O, want)


def test_mha_decode_cost_follows_the_context_not_the_cache(cuda):
    """One compile, any context (AGENTS.md:246-255, iron/operators/mha.py:275-278): over a 131072-row
    cache -- Llama-3.2-1B's own max_seq_len -- a context of 600 keys, one just past what a single block
    takes, and the whole cache, each against the oracle; and the launches of the first are those of a
    2048-row cache's (one block a query head does the work), not the cache's."""
    rng = np.random.default_rng(162)
    H, G, d, L = 32, 8, 64, 131072
    Q = bf(rng, 1, H, d)
    Kc = round_bf16(np.resize(rng.standard_normal((4099, G, d)), (L, G, d)).astype(np.float32))
    Vc = round_bf16(np.resize(rng.standard_normal((4099, G, d)), (L, G, d)).astype(np.float32))
    dQ, dK, dV = dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda)
    ws = K.mha_decode_workspace(H, d, cuda)
    for kv_valid in (600, 2049, 40000, L):
        O = out_like((1, H, d), cuda, fill=float("nan"))
        K.mha_decode(dQ, dK, dV, O, heads=H, kv_heads=G, d=d, kv_len=L, kv_interleaved=True,
                     kv_valid=word(kv_valid, cuda), workspace=ws)
        want = ops.mha(Q, Kc[:kv_valid], Vc[:kv_valid], num_heads=H, num_KV_heads=G, seq_len=1, kv_len=kv_valid, d=d,
                       heads_interleaved=True, kv_interleaved=True)
        close(O, want)


def test_mha_decode_equals_last_row_of_prefill(cuda):
    """A size-independent property: the one-query kernel and the last row of the many-query one agree."""
    rng = np.random.default_rng(17)
    H, G, d, S = 32, 8, 64, 1536
    Q, Kc, Vc = bf(rng, S, H, d), bf(rng, S, G, d), bf(rng, S, G, d)
    dQ, dK, dV = dev(Q, cuda), dev(Kc, cuda), dev(Vc, cuda)
    O = out_like((S, H, d), cuda)
    K.mha_prefill(dQ, dK, dV, O, heads=H, kv_heads=G, d=d, seq=S, kv_len=S, q_interleaved=True, kv_interleaved=True)
    o1 = out_like((1, H, d), cuda)
    K.mha_decode(dQ[S - 1 :].contiguous(), dK, dV, o1, heads=H, kv_heads=G, d=d, kv_len=S, kv_interleaved=True,
                 workspace=K.mha_decode_workspace(H, d, cuda))
    close(from_torch(o1)[0], from_torch(O)[S - 1], rtol=1e-2, atol=1e-2)


# ------------------------------------------------------------------------ glue
def test_gather_rows_exact(cuda):
    rng = np.random.default_rng(18)
    table = bf(rng, 1000, 2048)
    ids = rng.integers(0, 1000, 300).astype(np.int32)
    out = out_like((300, 2048), cuda, fill=1.0)
    K.gather_rows(dev(table, cuda), torch.from_numpy(ids).to(cuda), out, valid=word(256, cuda))
    got = from_torch(out)
    assert np.array_equal(got[:256], ops.gather_rows(table, ids[:256])) and np.all(got[256:] == 1.0)
    # int32 rows, a row width that is not a multiple of 16 bytes.
    t32 = torch.arange(50 * 3, dtype=torch.int32, device=cuda).reshape(50, 3)
    o32 = torch.zeros((4, 3), dtype=torch.int32, device=cuda)
    K.gather_rows(t32, torch.tensor([7, 0, 49, 7], dtype=torch.int32, device=cuda), o32)
    assert torch.equal(o32.cpu(), t32.cpu()[[7, 0, 49, 7]])


def test_copy_rows_cache_write_table_row_and_last_row(cuda):
    rng = np.random.default_rng(19)
    L, G, d = 128, 8, 64
    cache = dev(np.zeros((L, G * d), np.float32), cuda)
    k = bf(rng, 1, G * d)
    K.copy_rows(dev(k, cuda), cache, rows=1, row_elems=G * d, src_rows=1, dst_rows=L, dst_row=word(37, cuda))
    got = from_torch(cache)
    assert np.array_equal(got[37], k[0]) and np.count_nonzero(got) == np.count_nonzero(k)
    # A chunk of rows at a per-call start, bounded.
    x = bf(rng, 32, G * d)
    K.copy_rows(dev(x, cuda), cache, rows=32, row_elems=G * d, src_rows=32, dst_rows=L,
                dst_row=word(64, cuda), valid=word(20, cuda))
    got = from_torch(cache)
    assert np.array_equal(got[64:84], x[:20]) and np.all(got[84:] == 0)
    # The last valid row picked out (src index), and a row past the end skipped.
    last = out_like((1, G * d), cuda, fill=4.0)
    K.copy_rows(dev(x, cuda), last, rows=1, row_elems=G * d, src_rows=32, dst_rows=1, src_row=word(19, cuda))
    assert np.array_equal(from_torch(last)[0], x[19])
    K.copy_rows(dev(x, cuda), last, rows=1, row_elems=G * d, src_rows=32, dst_rows=1, src_row=word(32, cuda))
    assert np.array_equal(from_torch(last)[0], x[19])


def test_argmax_first_of_ties_and_record(cuda):
    rng = np.random.default_rng(11)
    logits = round_bf16(rng.normal(0, 3, 128256))
    top = rng.choice(128256, 8, replace=False)
    logits[top] = logits.max()
    first = int(min(top.min(), np.argmax(logits)))  # nine equal maxima: the first wins
    tok = torch.full((1,), -1, dtype=torch.int32, device=cuda)
    rec = torch.full((16,), -1, dtype=torch.int32, device=cuda)
    K.argmax(dev(logits, cuda), tok, record=rec, at=word(5, cuda))
    assert int(tok.item()) == ops.argmax(logits) == first
    assert rec.cpu().tolist() == [-1] * 5 + [first] + [-1] * 10
    odd = round_bf16(rng.normal(0, 1, 1003))
    K.argmax(dev(odd, cuda), tok)
    assert int(tok.item()) == ops.argmax(odd)


# ---------------------------------------------- the sibling decoders' operators
@pytest.mark.parametrize("kind,ref,exact", [
    ("gelu_tanh", lambda x: ops.gelu(x), False), ("gelu_erf", lambda x: ops.gelu(x, "none"), False),
    ("relu", ops.relu, True), ("sigmoid", ops.sigmoid, False), ("tanh", ops.tanh, False),
    ("clamp", lambda x: ops.clamp(x, -0.75, 1.25), True)])
def test_unary_kinds_and_their_bound(cuda, kind, ref, exact):
    rng = np.random.default_rng(50)
    x = bf(rng, 10007, scale=3.0)   # odd: a tail short of a 16-byte piece
    y = out_like((10007,), cuda, fill=7.0)
    K.unary(dev(x, cuda), y, kind, low=-0.75, high=1.25)
    if exact:
        assert np.array_equal(from_torch(y), ref(x))
    else:
        close(y, ref(x), rtol=2.0**-7, atol=1e-5)
    # A bound read on the device leaves the rest as it was.
    y.fill_(7.0)
    K.unary(dev(x, cuda), y, kind, low=-0.75, high=1.25, valid=word(4001, cuda))
    got = from_torch(y)
    close(got[:4001], ref(x)[:4001], rtol=2.0**-7, atol=1e-5)
    assert np.all(got[4001:] == 7.0)


def test_axpy_and_its_bound(cuda):
    rng = np.random.default_rng(51)
    x, y = bf(rng, 70001, scale=4.0), bf(rng, 70001, scale=4.0)
    out = out_like((70001,), cuda, fill=7.0)
    for a in (3.0, 1.003, -0.5):
        K.axpy(dev(x, cuda), dev(y, cuda), out, a=a)
        assert np.array_equal(from_torch(out), ops.axpy(a, x, y))   # one fma, one rounding: exact
    out.fill_(7.0)
    K.axpy(dev(x, cuda), dev(y, cuda), out, a=3.0, valid=word(13, cuda))
    got = from_torch(out)
    assert np.array_equal(got[:13], ops.axpy(3.0, x, y)[:13]) and np.all(got[13:] == 7.0)


@pytest.mark.parametrize("rows,cols,weighted", [(1, 2048, True), (33, 1024, False), (16, 4096, True), (5, 8192, True),
                                                (3, 12288, True), (64, 768, True)])
def test_layernorm_rows(cuda, rows, cols, weighted):
    rng = np.random.default_rng(cols + rows)
    x = round_bf16(bf(rng, rows, cols, scale=2.0) + np.float32(1.5))
    w = round_bf16(rng.uniform(0.9, 1.1, cols).astype(np.float32)) if weighted else None
    y = out_like((rows, cols), cuda, fill=7.0)
    K.layernorm(dev(x, cuda), None if w is None else dev(w, cuda), y, rows=rows, cols=cols, eps=1e-5)
    close(y, ops.layer_norm(x, w))
    if rows > 2:
        y.fill_(7.0)
        K.layernorm(dev(x, cuda), None if w is None else dev(w, cuda), y, rows=rows, cols=cols, eps=1e-5,
                    valid=word(2, cuda))
        got = from_torch(y)
        close(got[:2], ops.layer_norm(x, w)[:2])
        assert np.all(got[2:] == 7.0)


@pytest.mark.parametrize("rows,cols,f32,addend,cap", [(32, 1024, False, False, None), (16, 4608, False, False, None),
                                                      (4, 32768, False, False, None), (32, 1024, True, False, None),
                                                      (64, 1536, True, True, 50.0), (16, 80, True, True, None)])
def test_softmax_rows_cap_addend_and_length(cuda, rows, cols, f32, addend, cap):
    rng = np.random.default_rng(cols)
    x = rng.normal(0, 4, (rows, cols)).astype(np.float32)
    x = x if f32 else round_bf16(x)
    add = rng.normal(0, 1, (rows, cols)).astype(np.float32) if addend else None
    xd = torch.from_numpy(x).to(cuda) if f32 else dev(x, cuda)
    ad = None if add is None else torch.from_numpy(add).to(cuda)
    y = out_like((rows, cols), cuda, fill=7.0)
    K.softmax(xd, y, rows=rows, cols=cols, addend=ad, soft_cap=cap)
    close(y, ops.softmax(x, add, soft_cap=cap), rtol=1e-2, atol=1e-4)
    assert abs(float(from_torch(y).sum(axis=-1).mean()) - 1.0) < 5e-3
    # A length read on the device: the first columns' softmax, zeros after them.
    n = cols // 3
    K.softmax(xd, y, rows=rows, cols=cols, addend=ad, soft_cap=cap, length=word(n, cuda))
    got = from_torch(y)
    close(got, ops.softmax(x, add, soft_cap=cap, length=n), rtol=1e-2, atol=1e-4)
    assert not got[:, n:].any()


def _draw_rows(rng, count, temperatures=(0.0, 0.05, 0.7, 1.0, 5.0), k_hi=65):
    from iron_amd.operators.sample import draw_row

    return np.stack([draw_row(rng.choice(temperatures), int(rng.integers(1, k_hi)), int(rng.integers(0, 1 << 53)))
                     for _ in range(count)])


def _host_draw(logits, row, k_max=64):
    return ops.sample_ref(logits, *ops.draw_words(row), k_max)


def _sample_rows(cuda, logits, rows, n=None, k_max=64):
    """The device's draw for each of ``rows`` (picked by a device word), recorded one per slot."""
    steps = len(rows)
    tok = torch.full((1,), -1, dtype=torch.int32, device=cuda)
    rec = torch.full((steps,), -1, dtype=torch.int32, device=cuda)
    lg, dr = dev(logits, cuda), torch.from_numpy(np.ascontiguousarray(rows)).to(cuda)
    for i in range(steps):
        K.sample(lg, dr, tok, n=n, row=word(4 * i, cuda), k_max=k_max, record=rec, at=word(i, cuda))
        assert int(tok.item()) == int(rec[i].item())
    return rec.cpu().tolist()


@pytest.mark.parametrize("vocab,drawable", [(4096, 4096), (128256, 128256), (51866, 51866), (151670, 151669),
                                            (1003, 1003), (100, 100)])
def test_sample_draws_the_host_token(cuda, vocab, drawable):
    rng = np.random.default_rng(vocab)
    logits = round_bf16(rng.normal(0, 3, vocab))
    logits[rng.choice(drawable, 8, replace=False)] = logits[:drawable].max()
    logits[drawable:] = logits.max() + 1   # padding no draw may take
    rows = _draw_rows(rng, 48)
    got = _sample_rows(cuda, logits, rows, n=drawable)
    want = [_host_draw(logits[:drawable], r) for r in rows]
    assert got == want
    assert len(set(got)) > 4   # the draws spread over candidates


def test_sample_ties_at_the_cut_go_to_the_lower_index(cuda):
    # Few distinct values: the top-k cut falls inside a run of equal logits, and the k kept are
    # those of the lowest index.
    rng = np.random.default_rng(21)
    logits = round_bf16(rng.integers(-3, 4, 128256).astype(np.float32) * 0.5)
    rows = _draw_rows(rng, 32, temperatures=(0.7, 1.0, 5.0))
    assert _sample_rows(cuda, logits, rows) == [_host_draw(logits, r) for r in rows]
    # All equal: more logits at the floor than the list holds (the slow path), uniform over the first k.
    flat = np.full(40000, 1.5, np.float32)
    got = _sample_rows(cuda, flat, rows)
    assert got == [_host_draw(flat, r) for r in rows] and max(got) < 64
    # The best first in memory, falling: every thread's maximum is its first logit.
    falling = round_bf16(np.linspace(8, -8, 20000, dtype=np.float32))
    assert _sample_rows(cuda, falling, rows) == [_host_draw(falling, r) for r in rows]


# One block's logits and a block more, rows whose lists are one group of sixteen a thread and four; lists with room for 16, 32 and 64 entries (k = 8, 9, 20, 21),
# blocks whose threads list more than 64 (k = 64); distinct values, few enough for equal ones at every cut, and whole blocks in falling order.
@pytest.mark.parametrize("vocab", [2048, 2049, 131072, 131073, 500001])
@pytest.mark.parametrize("values", ["spread", "close", "falling"])
def test_sample_draws_the_host_token_for_every_room_of_its_lists(cuda, vocab, values):
    from iron_amd.operators.sample import draw_row

    rng = np.random.default_rng(vocab)
    logits = {"spread": rng.normal(0, 3, vocab), "close": rng.normal(0, 0.3, vocab), "falling": -np.arange(vocab) % 2048 / 512.0}[values]
    logits = round_bf16(logits.astype(np.float32))
    rows = np.stack([draw_row(temperature, k, int(rng.integers(0, 1 << 53)))
                     for k in (2, 7, 8, 9, 20, 21, 41, 50, 63, 64) for temperature in (0.7, 50.0)])
    assert _sample_rows(cuda, logits, rows) == [_host_draw(logits, r) for r in rows]


def test_sample_special_values_and_row_bounds(cuda):
    from iron_amd.operators.sample import draw_row

    rng = np.random.default_rng(22)
    logits = round_bf16(rng.normal(0, 1, 5000))
    logits[[7, 1200]] = np.nan
    logits[[9, 4000]] = -np.inf
    logits[[100, 101]] = [-0.0, 0.0]
    rows = np.concatenate([_draw_rows(rng, 16), [draw_row(0.7, 50, 0), draw_row(0.7, 50, (1 << 53) - 1),
                                                 draw_row(1e-3, 64, 1 << 52), draw_row(np.nan, 5, 77),
                                                 draw_row(-1.0, 5, 77)]])
    assert _sample_rows(cuda, logits, rows) == [_host_draw(logits, r) for r in rows]
    infinite = logits.copy()
    infinite[3000] = np.inf
    assert _sample_rows(cuda, infinite, rows[:8]) == [3000] * 8
    hollow = np.full(3000, -np.inf, np.float32)
    hollow[[5, 2500]] = [np.nan, 2.0]
    assert _sample_rows(cuda, hollow, rows[16:18]) == [2500, 2500]
    # A k_max under the row's top-k caps it.
    assert _sample_rows(cuda, logits, rows[:16], k_max=3) == [_host_draw(logits, r, 3) for r in rows[:16]]
    # No draw rows, or a row outside them: greedy.
    tok = torch.full((1,), -1, dtype=torch.int32, device=cuda)
    dr = torch.from_numpy(np.ascontiguousarray(rows[:2])).to(cuda)
    for kw in (dict(draws=None), dict(draws=dr, row=word(8, cuda)), dict(draws=dr, row=word(-4, cuda))):
        K.sample(dev(logits, cuda), kw.pop("draws"), tok, **kw)
        assert int(tok.item()) == ops.sample_ref(logits, 0.0, 1, 0)
    with pytest.raises(Exception, match="k_max"):
        K.sample(dev(logits, cuda), dr, tok, k_max=65)


def test_sample_leaves_its_workspace_ready_for_the_next_draw(cuda):
    # The block count in the workspace's first words must be zero when a draw starts; every draw
    # puts it back, so one zeroed workspace serves any number of draws, of changing lengths.
    rng = np.random.default_rng(23)
    logits = round_bf16(rng.normal(0, 3, 128256))
    rows = _draw_rows(rng, 12)
    lg, dr = dev(logits, cuda), torch.from_numpy(np.ascontiguousarray(rows)).to(cuda)
    ws = K.sample_workspace(logits.size, cuda)
    tok = torch.full((1,), -1, dtype=torch.int32, device=cuda)
    for i, n in enumerate([128256, 100, 51866, 128256, 4096, 1003] * 2):
        K.sample(lg, dr, tok, n=n, row=word(4 * i, cuda), workspace=ws)
        assert int(tok.item()) == _host_draw(logits[:n], rows[i]), (i, n)
        assert not ws[:2].any(), (i, n)


def test_eval_words_advances_a_decode_step(cuda):
    words = torch.tensor([11, 40, 0, 0, 0, 0, 0, 0], dtype=torch.int32, device=cuda)
    # position += 1; kv_valid = position + 1; rope_row = min(position, 5); half = position >> 1;
    # ring_row = max(position - 3, 0) % 16; its mirror's = ring_row + 16
    exprs = torch.tensor([[1, 1, 1, 1, 0, -(2**31), 2**31 - 1, -1, 0], [2, 1, 1, 1, 0, -(2**31), 2**31 - 1, -1, 0],
                          [3, 1, 1, 0, 0, 0, 5, -1, 0], [4, 1, 1, 0, 1, -(2**31), 2**31 - 1, -1, 0],
                          [5, 1, 1, -3, 0, 0, 2**31 - 1, 15, 0], [6, 1, 1, -3, 0, 0, 2**31 - 1, 15, 16]],
                         dtype=torch.int32, device=cuda)
    K.eval_words(words, exprs)
    assert words.cpu().tolist() == [11, 41, 42, 5, 20, 6, 22, 0]


# A wave's steps in turn: a step's edges, the splits' (64 or 32 times 32 keys a round) and the lines between the few keys' form and this; one KV head a block and two,
# heads of one and of sixteen queries, a window that begins inside a step.
@pytest.mark.parametrize("H,G,d,window", [(32, 8, 64, None), (32, 8, 128, None), (6, 3, 64, None), (16, 1, 128, None), (4, 4, 64, 1000)])
def test_decode_attention_takes_keys_in_turn(cuda, H, G, d, window):
    rng = np.random.default_rng(H + d)
    L = 8200
    g = torch.Generator(device="cuda")
    g.manual_seed(d)
    q, k, v = (torch.randn(n, w, d, generator=g, device="cuda").to(torch.bfloat16) for n, w in ((1, H), (L, G), (L, G)))
    q *= 2
    o, workspace = torch.empty(H, d, dtype=torch.bfloat16, device="cuda"), K.mha_decode_workspace(H, d)
    for n in (384, 385, 448, 449, 512, 513, 544, 545, 576, 577, 704, 705, 736, 737, 1408, 2047, 2049, 2080, 4097, 8192, 8193, 8200, int(rng.integers(600, 8000))):
        past = k[n:].clone()
        k[n:] = float("nan")   # (what lies past the live keys is nobody's)
        K.mha_decode(q, k, v, o, heads=H, kv_heads=G, d=d, kv_len=L, kv_interleaved=True, kv_valid=torch.tensor([n], dtype=torch.int32, device="cuda"),
                     window=window, workspace=workspace)
        k[n:] = past
        lo = 0 if window is None else max(0, n - 1 - window)
        kd, vd = k[lo:n].double(), v[lo:n].double()
        p = torch.softmax(torch.einsum("ghd,kgd->ghk", q.double().reshape(G, H // G, d), kd) / d**0.5, -1)
        want = torch.einsum("ghk,kgd->ghd", p, vd).reshape(H, d)
        # the output's rounding; weights, scores' sums and exponentials in 32 bits
        assert ((o.double() - want).abs() <= 2**-8 * want.abs() + 2**-12 * vd.abs().max()).all(), n
        if n == 2049:   # an infinite value is the output where its key weighs anything
            v[1500, 0, 3] = float("inf")
            K.mha_decode(q, k, v, o, heads=H, kv_heads=G, d=d, kv_len=L, kv_interleaved=True, kv_valid=torch.tensor([n], dtype=torch.int32, device="cuda"),
                         window=window, workspace=workspace)
            assert torch.isinf(o[: H // G, 3]).all()
            v[1500, 0, 3] = 0.0


@pytest.mark.parametrize("d,n", [(64, 600), (64, 1400), (64, 5000), (128, 500), (128, 3000)])
def test_decode_attention_s_weights_have_32_bits(cuda, d, n):
    """Two values that cancel to their last bits, so that an output is what its weights were rounded by; and an infinite value behind a tiny weight."""
    H, L, q0 = 8, 8200, np.float32(2 * d**0.5)
    rng = np.random.default_rng(n)
    score = -round_bf16(np.linspace(0.3, 4.7, H, dtype=np.float32))   # a head's every second key; the others have 0
    weight = np.exp(score.astype(np.float64) * 2)
    top = round_bf16(rng.uniform(1, 2, (H, d)).astype(np.float32))
    q, k, v = np.zeros((1, H, d), np.float32), np.zeros((L, H, d), np.float32), np.zeros((L, H, d), np.float32)
    q[..., 0] = q0 if d == 64 else round_bf16(q0)
    k[1::2, :, 0], v[0::2], v[1::2] = score, top, -round_bf16((top / weight[:, None]).astype(np.float32))
    scale = 2 / float(q[0, 0, 0])
    n0, n1 = (n + 1) // 2, n // 2
    sums = n0 + n1 * weight[:, None]
    want = (n0 * top.astype(np.float64) + n1 * weight[:, None] * v[1]) / sums
    size = (n0 * top + n1 * weight[:, None] * np.abs(v[1])) / sums
    assert (np.abs(want) < 2**-13 * size).sum() > 2   # (elements that the output's own rounding hides nothing of)
    o, workspace = torch.empty(H, d, dtype=torch.bfloat16, device="cuda"), K.mha_decode_workspace(H, d)
    q, k, v = dev(q, cuda), dev(k, cuda), dev(v, cuda)

    def run():
        K.mha_decode(q, k, v, o, heads=H, kv_heads=H, d=d, kv_len=L, scale=scale, kv_interleaved=True, kv_valid=word(n, cuda), workspace=workspace)
        return from_torch(o).astype(np.float64)

    # the output's rounding; a weight's (its score's product with log2 e and its exponential, some 2^-22) and the sums'
    assert (np.abs(run() - want) <= 2**-8 * np.abs(want) + 2**-20 * size).all()
    k[33, :, 0], v[33, :, 1] = -43.25, float("inf")   # e^-86.5, which is still no denormal
    assert np.isposinf(run()[:, 1]).all()


# A head's rows one behind the other: a round of all waves filled to either side of five sixths, from where heads of 128 have their keys in runs; runs' and splits' edges, a round
# and one key more, two rounds, and a window of them; heads two a block and one, splits of which a wave's place wraps.
@pytest.mark.parametrize("H,G,d,window,round_", [(32, 8, 64, None, 8192), (8, 8, 128, None, 8192), (32, 16, 128, None, 4096), (6, 3, 128, None, 85 * 256),
                                                 (4, 1, 128, None, 32768), (8, 8, 128, 6900, 8192)])
def test_decode_attention_over_rows_of_a_head(cuda, H, G, d, window, round_):
    line = round_ - round_ // 6
    L = 2 * round_ + 700
    g = torch.Generator(device="cuda")
    g.manual_seed(d)
    q, k, v = (torch.randn(*n, d, generator=g, device="cuda").to(torch.bfloat16) for n in ((H,), (G, L), (G, L)))
    q *= 2
    o, workspace = torch.empty(H, d, dtype=torch.bfloat16, device="cuda"), K.mha_decode_workspace(H, d)
    for n in (2049, line - 1, line, line + 1, line + 33, line + 129, round_ - 31, round_, round_ + 1, 2 * line - 1, 2 * round_ - 33, 2 * round_ + 500):
        past = k[:, n:].clone()
        k[:, n:] = float("nan")   # (what lies past the live keys is nobody's)
        workspace.fill_(float("nan"))
        K.mha_decode(q, k, v, o, heads=H, kv_heads=G, d=d, kv_len=L, kv_valid=word(n, cuda), window=window, workspace=workspace)
        k[:, n:] = past
        lo = 0 if window is None else max(0, n - 1 - window)
        p = torch.softmax((q.double().reshape(G, H // G, d) @ k[:, lo:n].double().transpose(1, 2).contiguous()) / d**0.5, -1)
        want = (p @ v[:, lo:n].double()).reshape(H, d)
        assert ((o.double() - want).abs() <= 2**-8 * want.abs() + 2**-12 * v.double().abs().max()).all(), n

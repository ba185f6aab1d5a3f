"""GPU parity of the MFMA prefill GEMM with on-the-fly dequantisation
(config 3 shapes and ragged edges) against the oracle.  rel-L2 <= 5e-3."""
import ctypes as C

import numpy as np
import pytest
import torch

import int4_hip
import r4q_oracle as O
import r4q_synth as S
from conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 5e-3


def _run(dev, bits, M, N, K, seed):
    g = S.gen(seed)
    w, sz = S.weight(N, K, bits, g)
    x = (torch.randn(M, K, generator=g)).half()
    y = int4_hip.dbg_gemm(x.to(dev), w.to(dev), None if sz is None else sz.to(dev), M, N, K)
    want = O.gemm(x.numpy(), w.numpy(), None if sz is None else sz.numpy(), bits)
    return y.cpu().numpy(), want


@pytest.mark.parametrize("M,N,K", [(512, 17408, 5120), (512, 5120, 17408)])
def test_prefill_gemm_config3(dev, M, N, K):
    got, want = _run(dev, 4, M, N, K, seed=3)
    assert np.all(np.isfinite(got))
    assert rel_l2(got, want) <= TOL


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,K", [(17, 100, 32), (130, 129, 96), (256, 384, 1024), (64, 64, 64)])
def test_prefill_gemm_ragged(dev, bits, M, N, K):
    got, want = _run(dev, bits, M, N, K, seed=M + N + K + bits)
    assert rel_l2(got, want) <= TOL


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,K", [(2, 7168, 5120), (8, 17408, 5120), (8, 5120, 17408),
                                   (16, 1000, 5120), (9, 300, 1024), (3, 77, 256),
                                   (5, 33, 128), (12, 65, 512)])
def test_skinny_gemm_vs_oracle(dev, bits, M, N, K):
    """2 <= M <= 16 rows (batched decode): weights streamed once through the
    LDS ring, MFMA; the workspace the library asks for lets narrow shapes
    split along K.  Shapes whose K is not a whole number of ring steps take
    the per-row GEMV path (checked the same way)."""
    got, want = _run(dev, bits, M, N, K, seed=7 * M + N + K + bits)
    assert np.all(np.isfinite(got))
    assert rel_l2(got, want) <= TOL
    for r in range(M):
        assert rel_l2(got[r], want[r]) <= TOL


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,K", [(8, 5120, 17408), (16, 200, 2048), (4, 130, 1024)])
def test_skinny_gemm_without_workspace(dev, bits, M, N, K):
    """r4q_gemm (no workspace): one pass over K per 64-row tile, no split."""
    import r4q_lib as R
    g = S.gen(3 * M + N + K + bits)
    w, sz = S.weight(N, K, bits, g)
    x = (torch.randn(M, K, generator=g) * 0.5).half()
    want = O.gemm(x.numpy(), w.numpy(), None if sz is None else sz.numpy(), bits)
    xd, wd = x.to(dev), w.to(dev)
    sd = None if sz is None else sz.to(dev)
    y = torch.empty(M, N, dtype=torch.float16, device=dev)
    R.call("r4q_gemm", xd.data_ptr(), wd.data_ptr(), None if sd is None else sd.data_ptr(),
           y.data_ptr(), M, N, K, bits, R.stream_handle())
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.all(np.isfinite(got))
    assert rel_l2(got, want) <= TOL


@pytest.mark.parametrize("bits", [4, 8, 16])
def test_skinny_gemm_one_hot_columns_exact(dev, bits):
    """Row r of x = e_k(r): y[r] is column k(r) of the dequantised weight,
    bit for bit (the in-register dequantisation equals the dequant kernel)."""
    g = S.gen(41 + bits)
    N, K, M = 300, 1024, 8
    w, sz = S.weight(N, K, bits, g)
    W = O.dequant(w.numpy(), None if sz is None else sz.numpy(), bits)
    ks = [0, 1, 4, 31, 32, 517, 1000, 1023]
    x = torch.zeros(M, K, dtype=torch.float16)
    for r, k in enumerate(ks):
        x[r, k] = 1.0
    y = int4_hip.dbg_gemm(x.to(dev), w.to(dev), None if sz is None else sz.to(dev), M, N, K)
    y = y.cpu().numpy()
    for r, k in enumerate(ks):
        assert np.array_equal(y[r], W[:, k]), k


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,K", [(300, 1000, 2048), (257, 520, 32), (600, 256, 4096),
                                   (512, 7168, 5120), (256, 255, 96)])
def test_ring_gemm_ragged_and_split(dev, bits, M, N, K):
    """M >= 256: 256 x 256 tiles, ragged in M and N, K loops shorter than the
    copy ring (K = 32, 96), and split-K over a
    workspace (few tiles, long K)."""
    got, want = _run(dev, bits, M, N, K, seed=M + 3 * N + K + bits)
    assert np.all(np.isfinite(got))
    assert rel_l2(got, want) <= TOL
    for r in (0, M // 2, M - 1):
        assert rel_l2(got[r], want[r]) <= TOL, r


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("N,K", [(700, 1024), (300, 8192)])
def test_ring_gemm_one_hot_columns_exact(dev, bits, N, K):
    """Row r of x = e_k(r) over 300 rows: y[r] is column k(r) of the
    dequantised weight, bit for bit -- in one pass and with the K loop split
    (fp16 partials of zeros and one exact product)."""
    g = S.gen(43 + bits + K)
    M = 300
    w, sz = S.weight(N, K, bits, g)
    W = O.dequant(w.numpy(), None if sz is None else sz.numpy(), bits)
    ks = [(r * 997 + r // 7) % K for r in range(M)]
    x = torch.zeros(M, K, dtype=torch.float16)
    for r, k in enumerate(ks):
        x[r, k] = 1.0
    y = int4_hip.dbg_gemm(x.to(dev), w.to(dev), None if sz is None else sz.to(dev), M, N, K)
    y = y.cpu().numpy()
    for r, k in enumerate(ks):
        assert np.array_equal(y[r], W[:, k]), (r, k)


def test_ring_gemm_split_matches_unsplit(dev):
    """The split-K result equals the one-pass result within the rounding of
    its fp16 partials."""
    import ctypes as C
    import r4q_lib as R
    g = S.gen(77)
    M, N, K = 512, 768, 8192
    w, sz = S.int4_weight(N, K, g)
    x = torch.randn(M, K, generator=g).half()
    X, Wd, SZ = x.to(dev), w.to(dev), sz.to(dev)
    nws = C.c_size_t(0)
    R.call("r4q_gemm_workspace_bytes", M, N, K, 4, C.byref(nws))
    assert nws.value > 0  # this shape splits
    ws = torch.empty(nws.value, dtype=torch.uint8, device=dev)
    y1 = torch.empty(M, N, dtype=torch.float16, device=dev)
    y2 = torch.empty(M, N, dtype=torch.float16, device=dev)
    R.call("r4q_gemm", X.data_ptr(), Wd.data_ptr(), SZ.data_ptr(), y1.data_ptr(), M, N, K, 4,
           R.stream_handle())
    R.call("r4q_gemm_ws", X.data_ptr(), Wd.data_ptr(), SZ.data_ptr(), y2.data_ptr(), M, N, K, 4,
           ws.data_ptr(), nws.value, R.stream_handle())
    a, b = y1.float().cpu().numpy(), y2.float().cpu().numpy()
    assert rel_l2(b, a) <= 1e-3
    want = O.gemm(x.numpy(), w.numpy(), sz.numpy(), 4)
    assert rel_l2(b, want) <= TOL


def test_small_m_path_matches_gemv(dev):
    """M <= 16 rows agree with the batch-1 GEMV row by row (different
    accumulation order: tolerance, not bits)."""
    g = S.gen(5)
    N, K = 1000, 5120
    w, sz = S.int4_weight(N, K, g)
    x = torch.randn(8, K, generator=g).half()
    W, SZ, X = w.to(dev), sz.to(dev), x.to(dev)
    y = int4_hip.dbg_gemm(X, W, SZ, 8, N, K)
    for r in range(8):
        assert rel_l2(y[r], int4_hip.dbg_gemv(X[r].contiguous(), W, SZ, N, K)) <= 1e-3


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("bits,M,I,K", [(4, 8, 17408, 5120), (8, 8, 17408, 5120), (4, 2, 512, 5120),
                                        (8, 16, 2048, 1024), (16, 4, 1024, 2048)])
def test_gemm_silu_fwht_matches_gemm_then_silu(dev, bits, M, I, K, split):
    """r4q_gemm_silu_fwht_ws equals r4q_gemm_ws with the same workspace into
    [M, 2I] followed by r4q_silu_mul_fwht, bit for bit, over two calls: with
    a workspace that splits K (split sum + SiLU gate + FWHT-32 in the reduce)
    and, for M <= 8, without one (the unsplit GEMM over tiles of 32 gate rows
    and the 32 up rows of the same indices, the gate in its epilogue)."""
    import r4q_lib as R
    g = S.gen(7 * M + I + K + bits)
    w, sz = S.weight(2 * I, K, bits, g)
    wd = w.to(dev)
    sd = None if sz is None else sz.to(dev)
    b = C.c_size_t(0)
    R.call("r4q_gemm_workspace_bytes", M, 2 * I, K, bits, C.byref(b))
    assert b.value > 0
    ws = torch.empty(b.value if split else 0, dtype=torch.uint8, device=dev)
    wsp = ws.data_ptr() if split else None
    st = R.stream_handle()
    if not split and M > 8:  # above 8 rows the gate needs the split path: rejected
        x = torch.zeros(M, K, dtype=torch.float16, device=dev)
        y = torch.empty(M, I, dtype=torch.float16, device=dev)
        with pytest.raises(RuntimeError):
            R.call("r4q_gemm_silu_fwht_ws", x.data_ptr(), wd.data_ptr(),
                   None if sd is None else sd.data_ptr(), y.data_ptr(), M, I, K, bits, None, 0,
                   st)
        return
    for rep in range(2):
        x = (torch.randn(M, K, generator=g) * (0.5 + rep)).half().to(dev)
        gu = torch.empty(M, 2 * I, dtype=torch.float16, device=dev)
        want = torch.empty(M, I, dtype=torch.float16, device=dev)
        R.call("r4q_gemm_ws", x.data_ptr(), wd.data_ptr(), None if sd is None else sd.data_ptr(),
               gu.data_ptr(), M, 2 * I, K, bits, wsp, ws.numel(), st)
        R.call("r4q_silu_mul_fwht", gu.data_ptr(), gu.data_ptr() + 2 * I, want.data_ptr(),
               M, I, 2 * I, I, st)
        got = torch.full((M, I), float("nan"), dtype=torch.float16, device=dev)
        R.call("r4q_gemm_silu_fwht_ws", x.data_ptr(), wd.data_ptr(),
               None if sd is None else sd.data_ptr(), got.data_ptr(), M, I, K, bits,
               wsp, ws.numel(), st)
        torch.cuda.synchronize()
        assert torch.isfinite(want).all()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (bits, M, I, K, rep)


def test_gemm_silu_fwht_rejects_unsplit_shapes(dev):
    """One row, I off the 32-chunk grid, or more than 8 rows with a workspace
    too small to split K are errors (the caller uses r4q_gemm_ws +
    r4q_silu_mul_fwht there)."""
    import r4q_lib as R
    I, K = 512, 5120
    w, sz = S.weight(2 * I, K, 4, S.gen(5))
    wd, sd = w.to(dev), sz.to(dev)
    x = torch.zeros(16, K, dtype=torch.float16, device=dev)
    y = torch.empty(16, I, dtype=torch.float16, device=dev)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device=dev)
    st = R.stream_handle()
    for (M, II, nbytes) in ((1, I, ws.numel()), (8, I - 16, ws.numel()), (16, I, 256)):
        with pytest.raises(RuntimeError):
            R.call("r4q_gemm_silu_fwht_ws", x.data_ptr(), wd.data_ptr(), sd.data_ptr(),
                   y.data_ptr(), M, II, K, 4, ws.data_ptr(), nbytes, st)


def _ref32(x, w, sz, bits):
    """x @ deq(W)^T in float32 on the CPU: the oracle's dequantisation (bit-exact
    to the kernels') and a library matmul, for shapes too large for the
    float64 oracle GEMM to finish in seconds."""
    W = torch.from_numpy(O.dequant(w.numpy(), None if sz is None else sz.numpy(), bits)).float()
    return (x.float() @ W.T).numpy()


@pytest.mark.parametrize("bits", [4, 8, 16])
def test_ring_gemm_whole_tile_rounds_then_stream_k(dev, bits):
    """576 tiles of 256 x 256 (more than two rounds of 256 workgroups): the
    first two rounds' 512 tiles are computed whole, the remaining 64 tiles'
    K units are shared by 256 stream-K workgroups (pieces of tiles as fp16
    partials, summed in segment order)."""
    import ctypes as C
    import r4q_lib as R
    M, N, K = 2304, 16384, 768
    g = S.gen(91 + bits)
    w, sz = S.weight(N, K, bits, g)
    x = (torch.randn(M, K, generator=g) * 0.5).half()
    nws = C.c_size_t(0)
    R.call("r4q_gemm_workspace_bytes", M, N, K, bits, C.byref(nws))
    assert nws.value > 0
    SZ = None if sz is None else sz.to(dev)
    got = int4_hip.dbg_gemm(x.to(dev), w.to(dev), SZ, M, N, K).float().cpu().numpy()
    want = _ref32(x, w, sz, bits)
    assert np.all(np.isfinite(got))
    assert rel_l2(got, want) <= TOL
    for r in (0, 255, 256, 1023, 2047, 2048, 2200, M - 1):  # whole-tile and shared rows
        assert rel_l2(got[r], want[r]) <= TOL, r


@pytest.mark.parametrize("splits", [2, 5])
def test_ring_gemm_forced_split_counts(dev, splits):
    """The gemm_splits override shares every tile among about `splits`
    workgroups; results equal the default plan's within the rounding of fp16
    partials and the oracle's within the GEMM tolerance."""
    import ctypes as C
    import r4q_lib as R
    M, N, K = 512, 1280, 4096
    g = S.gen(17 + splits)
    w, sz = S.int4_weight(N, K, g)
    x = torch.randn(M, K, generator=g).half()
    X, Wd, SZ = x.to(dev), w.to(dev), sz.to(dev)
    base = int4_hip.dbg_gemm(X, Wd, SZ, M, N, K).float().cpu().numpy()
    try:
        R.tune("gemm_splits", splits)
        nws = C.c_size_t(0)
        R.call("r4q_gemm_workspace_bytes", M, N, K, 4, C.byref(nws))
        assert nws.value > 0
        got = int4_hip.dbg_gemm(X, Wd, SZ, M, N, K).float().cpu().numpy()
    finally:
        R.tune("gemm_splits", 0)
    assert rel_l2(got, base) <= 1e-3
    assert rel_l2(got, O.gemm(x.numpy(), w.numpy(), sz.numpy(), 4)) <= TOL


def _plan(M, N, K, bits, ws=0):
    """(tile rows, tile columns, whole tiles, stream-K workgroups)."""
    import r4q_lib as R
    v = (C.c_int32 * 4)()
    R.call("r4q_gemm_plan", M, N, K, bits, ws, v, 4)
    return tuple(v)


def _gemm_whole(x, w, sz, M, N, K, bits):
    """The product without a workspace: whole tiles."""
    import r4q_lib as R
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device=x.device)
    R.call("r4q_gemm", x.data_ptr(), w.data_ptr(), None if sz is None else sz.data_ptr(),
           y.data_ptr(), M, N, K, bits, R.stream_handle())
    return y


@pytest.mark.parametrize("M,N,K", [(512, 17408, 5120), (512, 5120, 17408), (600, 256, 4096),
                                   (512, 7168, 5120), (300, 1280, 2048)])
def test_tile_gemm_vs_oracle_and_smaller_tiles(dev, M, N, K):
    """INT4 prompt shapes, a ragged M and split-K shapes against the oracle; in
    whole 256 x 256 tiles an output is one chain over k, so the first 255 rows
    alone, which take smaller tiles, give the same bits."""
    g = S.gen(M + 5 * N + K)
    w, sz = S.int4_weight(N, K, g)
    x = torch.randn(M, K, generator=g).half()
    X, Wd, SZ = x.to(dev), w.to(dev), sz.to(dev)
    got = int4_hip.dbg_gemm(X, Wd, SZ, M, N, K).float().cpu().numpy()
    assert np.all(np.isfinite(got))
    want = _ref32(x, w, sz, 4) if N * K > 4e7 else O.gemm(x.numpy(), w.numpy(), sz.numpy(), 4)
    assert rel_l2(got, want) <= TOL
    for r in (0, M // 2, M - 1):
        assert rel_l2(got[r], want[r]) <= TOL, r
    assert _plan(M, N, K, 4)[:2] == (256, 256) and _plan(255, N, K, 4)[0] <= 128
    whole = _gemm_whole(X, Wd, SZ, M, N, K, 4)
    few = _gemm_whole(X[:255].contiguous(), Wd, SZ, 255, N, K, 4)
    assert torch.equal(few.view(torch.int16), whole[:255].view(torch.int16))


@pytest.mark.parametrize("splits", [0, 3])
def test_tile_gemm_one_hot_columns_exact(dev, splits):
    """Row r of x = e_k(r): y[r] is column k(r) of the dequantised weight, bit
    for bit -- in the default plan and with every tile shared by about 3
    workgroups (fp16 partials of zeros and one exact product, summed by the
    reduce)."""
    import r4q_lib as R
    g = S.gen(211 + splits)
    M, N, K = 300, 384, 2048
    w, sz = S.int4_weight(N, K, g)
    W = O.dequant(w.numpy(), sz.numpy(), 4)
    ks = [(r * 631 + r // 5) % K for r in range(M)]
    x = torch.zeros(M, K, dtype=torch.float16)
    for r, k in enumerate(ks):
        x[r, k] = 1.0
    R.tune("gemm_splits", splits)
    try:
        y = int4_hip.dbg_gemm(x.to(dev), w.to(dev), sz.to(dev), M, N, K).cpu().numpy()
    finally:
        R.tune("gemm_splits", 0)
    for r, k in enumerate(ks):
        assert np.array_equal(y[r], W[:, k]), (r, k)


# (M, N, tile) that the rule takes to each tile of 17 .. 255 rows; N ragged
TILES = [(31, 4003, (32, 64)), (47, 8259, (48, 64)), (63, 8259, (64, 64)), (64, 16500, (64, 128)),
         (95, 16500, (96, 128)), (127, 16502, (128, 128)), (200, 34810, (128, 128))]


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,tile", TILES)
def test_every_tile_of_17_to_255_rows(dev, bits, M, N, tile):
    """Each tile shape in each format, on shapes that the rule takes there, K
    several times round the ring (17 x 128 + 32, 34 x 64 + 32 k) with a partial
    last step: against fp32 sums (fp16 output rounding 2.9e-4 rel-L2), and the
    same bits as its first 17 rows alone, which take 32 x 64 tiles."""
    K = 2208
    if bits == 16 and tile[0] == 48:
        tile = (64, 64)  # 48 x 64 does not exist for FP16 weights
    assert _plan(M, N, K, bits) == (*tile, -(-M // tile[0]) * -(-N // tile[1]), 0)
    assert _plan(17, N, K, bits)[:2] == (32, 64)
    g = S.gen(M + N + bits)
    w, sz = S.weight(N, K, bits, g)
    x = torch.randn(M, K, generator=g).half().to(dev)
    wd, sd = w.to(dev), None if sz is None else sz.to(dev)
    W = wd if bits == 16 else (int4_hip.dequant_int4 if bits == 4 else int4_hip.dequant_int8)(
        wd, sd, N, K)
    want = x.float() @ W.float().T
    y = int4_hip.dbg_gemm(x, wd, sd, M, N, K)
    assert torch.isfinite(y).all()
    err = (y.float() - want).norm(dim=1) / want.norm(dim=1)
    assert err.max().item() <= 6e-4, err.argmax().item()
    few = int4_hip.dbg_gemm(x[:17].contiguous(), wd, sd, 17, N, K)
    assert torch.equal(few.view(torch.int16), y[:17].view(torch.int16))


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,K", [(17, 131, 32), (32, 128, 160), (33, 260, 1056), (64, 129, 4128),
                                   (65, 640, 2080), (96, 127, 224), (97, 513, 4096),
                                   (128, 20000, 96), (129, 1000, 1312), (255, 383, 4192),
                                   (256, 257, 1056), (257, 70, 96), (513, 1030, 2080)])
def test_tile_gemm_edges(dev, bits, M, N, K):
    """32 x 64 tiles (narrow N takes every M below 256 there; 128 x 20000: 128 x
    128) and 256 x 256 ones: rows and widths one past and one short of a tile,
    widths off the 16-byte store, K shorter than a step and ending inside one,
    split and unsplit (no workspace).  The fp16 output rounds within 2^-12
    relative (rel-L2 below 2.9e-4), a fp16 partial (M >= 256) as much again per
    segment: 1e-3 is twice their sum over the at most 16 segments' random
    signs.  In whole tiles an output is one chain over k, so rows alone in a
    smaller tile (their first 17) give the same bits."""
    g = S.gen(M + 7 * N + K + bits)
    w, sz = S.weight(N, K, bits, g)
    x = torch.randn(M, K, generator=g).half()
    X, Wd, SZ = x.to(dev), w.to(dev), None if sz is None else sz.to(dev)
    want = _ref32(x, w, sz, bits)
    split = int4_hip.dbg_gemm(X, Wd, SZ, M, N, K)
    whole = _gemm_whole(X, Wd, SZ, M, N, K, bits)
    for y in (split, whole):
        got = y.float().cpu().numpy()
        assert np.all(np.isfinite(got))
        assert rel_l2(got, want) <= 1e-3
        for r in (0, M // 2, M - 1):
            assert rel_l2(got[r], want[r]) <= 1e-3, r
    few = int4_hip.dbg_gemm(X[:17].contiguous(), Wd, SZ, 17, N, K)
    assert torch.equal(few.view(torch.int16), whole[:17].view(torch.int16))


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,K", [(40, 200, 288), (120, 150, 2080), (260, 300, 352)])
def test_tile_gemm_one_hot_and_infinite_rows(dev, bits, M, N, K):
    """Row r of x = e_k(r) gives column k(r) of the dequantised weight bit for
    bit, K ending inside a step; an infinity in the row's last element reaches
    only its own row and, times a non-zero weight, stays an infinity (a step
    past K multiplies zeros, not the repeated last elements)."""
    g = S.gen(5 * M + N + K + bits)
    w, sz = S.weight(N, K, bits, g)
    W = O.dequant(w.numpy(), None if sz is None else sz.numpy(), bits)
    ks = [(r * 97 + r // 3) % K for r in range(M)]
    ks[1] = K - 1
    x = torch.zeros(M, K, dtype=torch.float16)
    for r, k in enumerate(ks):
        x[r, k] = 1.0
    x[2, :] = 0.0
    x[2, K - 1] = float("inf")
    y = int4_hip.dbg_gemm(x.to(dev), w.to(dev), None if sz is None else sz.to(dev), M, N, K)
    y = y.cpu().numpy()
    for r, k in enumerate(ks):
        if r != 2:
            assert np.array_equal(y[r], W[:, k]), (r, k)
    nz = W[:, K - 1] != 0
    assert np.array_equal(y[2][nz], np.where(W[nz, K - 1] > 0, np.inf, -np.inf).astype(np.float16))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,tile", [
    (17, 70, 1056, (32, 64)), (48, 8259, 352, (48, 64)), (64, 8259, 1184, (64, 64)),
    (64, 16500, 608, (64, 128)), (96, 16500, 736, (96, 128)), (128, 16500, 352, (128, 128)),
    (255, 300, 2080, (32, 64))])
def test_tile_gemm_zero_points_of_any_value(dev, bits, M, N, K, tile):
    """fp16((q - zp) * scale) holds for every zero-point below 256 rows, whole
    number or not, in every tile shape: row r of x = e_k(r) gives column k(r) of
    the oracle's dequantised weight bit for bit where blocks with other
    zero-points sit among the usual ones, in some weight rows only, and in a
    last partial step."""
    assert _plan(M, N, K, bits)[:2] == tile
    g = S.gen(3 * M + N + K + bits)
    w, sz = S.weight(N, K, bits, g)
    z = sz.view(N, K // 32, 2)[:, :, 1]
    odd = torch.tensor([0.5, 7.25, -0.5, -100.0625, 1e-6, 0.1, 1024.0, 1025.0, 2047.0, 3001.0,
                        -1000.5, 60000.0]).half()
    pick = torch.randint(0, len(odd), z.shape, generator=g)
    where = torch.rand(z.shape, generator=g) < 0.02
    where[: N // 3, : K // 64] = False  # steps without any
    where[:, -1] |= torch.rand(N, generator=g) < 0.3
    z[where] = odd[pick[where]]
    W = O.dequant(w.numpy(), sz.numpy(), bits)
    assert np.all(np.isfinite(W))
    ks = [(r * 97 + r // 3) % K for r in range(M)]
    ks[1] = K - 1
    x = torch.zeros(M, K, dtype=torch.float16)
    x[torch.arange(M), torch.tensor(ks)] = 1.0
    y = int4_hip.dbg_gemm(x.to(dev), w.to(dev), sz.to(dev), M, N, K).cpu().numpy()
    for r, k in enumerate(ks):
        assert np.array_equal(y[r], W[:, k]), (r, k)

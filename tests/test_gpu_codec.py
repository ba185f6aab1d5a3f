"""GPU parity of the byte/integer kernels: bit-exact against the oracle."""
import numpy as np
import pytest
import torch

import int4_hip
import r4q_oracle as O
import r4q_synth as S
from conftest import fp8_golden_table

pytestmark = pytest.mark.gpu


def test_fp16_to_fp8_all_bit_patterns(dev):
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    x = torch.from_numpy(bits.view(np.int16)).view(torch.float16).to(dev)
    got = int4_hip.fp16_to_fp8(x).cpu().numpy()
    want = O.fp8_encode(bits.view(np.float16).astype(np.float32))
    assert np.array_equal(got, want)
    assert np.array_equal(got, fp8_golden_table())


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1000003])
def test_fp16_to_fp8_ragged_sizes(dev, n):
    g = S.gen(n)
    x = (torch.randn(n, generator=g) * 50).half()
    got = int4_hip.fp16_to_fp8(x.to(dev)).cpu().numpy()
    assert np.array_equal(got, O.fp8_encode(x.float().numpy()))


def test_fp8_to_fp16_all_codes(dev):
    c = torch.arange(256, dtype=torch.int32).to(torch.uint8)
    got = int4_hip.fp8_to_fp16(c.to(dev)).cpu().float().numpy()
    want = O.fp8_value(c.numpy())
    ok = ~np.isnan(want)
    assert np.array_equal(got[ok].astype(np.float64), want[ok])


@pytest.mark.parametrize("N,K", [(17408, 5120), (5120, 17408), (3, 32), (7, 96)])
def test_dequant_int4_bit_exact(dev, N, K):
    g = S.gen(N + K)
    w, sz = S.int4_weight(N, K, g)
    got = int4_hip.dequant_int4(w.to(dev), sz.to(dev), N, K).cpu().numpy()
    want = O.dequant_int4(w.numpy(), sz.numpy())
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))


def test_dequant_int4_exhaustive_scales(dev):
    """All (q, zp) pairs times every finite fp16 scale."""
    x = np.arange(65536, dtype=np.uint32).astype(np.uint16).view(np.float16)
    scales = x[np.isfinite(x)]
    N, K = scales.size, 512
    q = np.tile(np.concatenate([np.arange(16), np.arange(16)]).astype(np.uint8), 16)
    packed = O.pack_int4(np.broadcast_to(q, (N, K)))
    zeros = np.broadcast_to(np.arange(16, dtype=np.uint8), (N, 16))
    sz = O.interleave_scale_zero(np.broadcast_to(scales[:, None], (N, 16)), zeros)
    got = int4_hip.dequant_int4(torch.from_numpy(packed).to(dev),
                                torch.from_numpy(np.ascontiguousarray(sz)).to(dev), N, K)
    want = O.dequant_int4(packed, sz)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("N,K", [(5120, 17408), (9, 64)])
def test_dequant_int8_bit_exact(dev, N, K):
    g = S.gen(N * 3 + K)
    w, sz = S.int8_weight(N, K, g)
    got = int4_hip.dequant_int8(w.to(dev), sz.to(dev), N, K).cpu().numpy()
    want = O.dequant_int8(w.numpy(), sz.numpy())
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("n", [1, 7, 8, 9, 1023, 1024, 1025, 8191, 8192, 8193, 16397])
def test_fp8_codecs_at_every_alignment(dev, n):
    """Whole and partial turns of a workgroup, with the source at each
    alignment the entry points take: 8 bytes for fp16, 1 for codes."""
    bits = (np.arange(n + 8, dtype=np.uint32) * 40503 + n).astype(np.uint16)
    x = torch.from_numpy(bits.view(np.int16)).view(torch.float16).to(dev)
    codes = torch.from_numpy((bits >> 3).astype(np.uint8)).to(dev)
    for off in (0, 4, 8):
        got = int4_hip.fp16_to_fp8(x[off:off + n]).cpu().numpy()
        assert np.array_equal(got, fp8_golden_table()[bits[off:off + n]])
    for off in (0, 1, 4, 8):
        got = int4_hip.fp8_to_fp16(codes[off:off + n]).cpu().double().numpy()
        want = O.fp8_value((bits[off:off + n] >> 3).astype(np.uint8))
        ok = ~np.isnan(want)
        assert np.array_equal(got[ok], want[ok])


@pytest.mark.parametrize("n", [(1 << 23) - 1, 1 << 23, (1 << 23) + 1, (1 << 23) + 8200])
def test_fp8_codecs_either_side_of_one_turn(dev, n):
    """The last size with one turn per thread and the first with four, with
    partial turns and remainders: every code against the tables."""
    bits = torch.arange(n, dtype=torch.int32, device=dev) * 40503 + n
    x = bits.to(torch.int16).view(torch.float16)
    enc = torch.from_numpy(fp8_golden_table()).to(dev)
    assert torch.equal(int4_hip.fp16_to_fp8(x), enc[(bits & 0xFFFF).long()])
    codes = (bits >> 3).to(torch.uint8)
    val = torch.from_numpy(O.fp8_value(np.arange(256, dtype=np.uint8))).to(dev)
    want = val[codes.long()]
    got = int4_hip.fp8_to_fp16(codes).double()
    assert torch.equal(got[~want.isnan()], want[~want.isnan()])


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K", [(1, 32), (1, 8160), (1, 8192), (255, 32), (257, 64), (3, 8224)])
def test_dequant_turn_edges(dev, bits, N, K):
    g = S.gen(N + K + bits)
    w, sz = (S.int4_weight if bits == 4 else S.int8_weight)(N, K, g)
    f, o = ((int4_hip.dequant_int4, O.dequant_int4) if bits == 4
            else (int4_hip.dequant_int8, O.dequant_int8))
    got = f(w.to(dev), sz.to(dev), N, K).cpu().numpy()
    assert np.array_equal(got.view(np.uint16), o(w.numpy(), sz.numpy()).view(np.uint16))


def test_dequant_rejects_bad_shape(dev):
    w = torch.zeros(4, 24, dtype=torch.uint8, device=dev)
    s = torch.zeros(4, 3, dtype=torch.float16, device=dev)
    with pytest.raises((RuntimeError, ValueError)):
        int4_hip.dequant_int4(w, s, 4, 48)

"""GPU tail-biting trellis encoder (trellis_encode_tiles) against the CPU oracle's C
restatement of qtip.viterbi_tb / _viterbi_pass (src/trellis/qtip.py:124-196).

The GPU DP runs the oracle's fp32 operations in the same order without contraction and
with the same tie rules, so the bar is bit-identity of the packed symbols and of the
dequantized values (stricter than the reference's own test, which pins only equal MSE
because its PyTorch and Triton DPs differ: tests/test_triton_kernel.py:24-44)."""
import sys

import numpy as np
import pytest
import torch

from oracle import trellis_np as tn
from oracle import viterbi as ov

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("K", [2, 3, 4])
@pytest.mark.parametrize("cb", ["mcg", "3inst", "1mad"])
def test_encode_bit_exact_vs_oracle(te, gpu_device, K, cb):
    _say(f"[encode] K={K} cb={cb}")
    rng = np.random.default_rng(100 + K)
    n = 24
    w = (rng.standard_normal((n, 256)) * tn.codebook_rms(cb)).astype(np.float32)
    bits_o, dq_o, _ = ov.viterbi_tb(w, K, tn.codebook_lut(cb))
    packed_o = tn.pack_bits(bits_o, K)
    bits_g, dq_g = te.encode_tiles(torch.from_numpy(w).to(gpu_device), K, cb)
    assert np.array_equal(bits_g.cpu().numpy().view(np.uint32), packed_o)
    assert np.array_equal(dq_g.cpu().numpy().view(np.uint32), dq_o.view(np.uint32))


@pytest.mark.parametrize("K", [2, 3, 4])
def test_encode_decode_round_trip_and_quality(te, gpu_device, K):
    """decode(encode(w)) == dq through the packed stream (the tail-biting wrap closes), and
    the distortion of N(0,1) targets under MCG is the quality the reference pins for its
    encoders (K=2 ~0.073; it falls by ~4x per extra bit)."""
    _say(f"[encode] round trip K={K}")
    g = torch.Generator(device=gpu_device)
    g.manual_seed(K)
    w = torch.randn((512, 256), generator=g, device=gpu_device)
    bits, dq = te.encode_tiles(w, K, "mcg")
    rec = te.PackedRecord(16, 16 * 512, K, bits[:].cpu().numpy().view(np.uint32),
                          np.ones(16 * 512, np.float16), np.ones(16, np.float16),
                          np.ones(16 * 512, np.float16), np.ones(16, np.float16), 1.0)
    lin = te.PackedLinear(rec, device=gpu_device)
    dec = lin.decode_tiles()
    assert torch.equal(dec, dq)
    mse = ((w - dq) ** 2).mean().item()
    # the oracle's C encoder on 96 N(0,1) tiles: 0.0746, 0.0182, 0.00469
    want = {2: 0.0746, 3: 0.0182, 4: 0.00469}[K]
    assert abs(mse - want) / want < 0.05, mse


def test_encode_many_tiles_persistent(te, gpu_device):
    """More tiles than workgroups (each workgroup loops over tiles and reuses its
    backpointer region): every tile still equals the oracle's encode."""
    _say("[encode] 1000 tiles")
    rng = np.random.default_rng(5)
    w = rng.standard_normal((1000, 256)).astype(np.float32)
    bits_g, _ = te.encode_tiles(torch.from_numpy(w).to(gpu_device), 3, "mcg", want_dq=False)
    bits_o, _, _ = ov.viterbi_tb(w, 3, tn.codebook_lut("mcg"))
    assert np.array_equal(bits_g.cpu().numpy().view(np.uint32), tn.pack_bits(bits_o, 3))


def _encode_np(w, K, lut):
    """The two-pass encode of one tile in numpy fp32, with q = 0 where no candidate lies below
    FLT_MAX (the C oracle leaves such a step's backpointer as it was)."""
    E, Q, top = 1 << (16 - K), 1 << K, np.float32(np.finfo(np.float32).max)
    v = lut.reshape(Q, E)

    def one(seq, overlap):
        cost = np.zeros(E, np.float32)
        if overlap is not None:
            cost[:] = top / np.float32(4)
            cost[overlap] = 0
        back = []
        for t in range(256):
            d = np.float32(seq[t]) - v
            c = d * d + np.repeat(cost.reshape(Q, E >> K), Q, axis=1)
            c = np.where(c < top, c, top)            # also NaN -> FLT_MAX
            q = c.argmin(0)                          # the smallest q on ties
            cost = c[q, np.arange(E)]
            back.append(q)
        e = int(cost.argmin()) if overlap is None else overlap
        states = np.empty(256, np.int64)
        for t in range(255, -1, -1):
            states[t] = (int(back[t][e]) << (16 - K)) | e
            e = int(states[t]) >> K
        return states

    first = one(np.roll(w, 128), None)
    return one(w, int(first[128]) >> K)


@pytest.mark.parametrize("K", [2, 3, 4])
@pytest.mark.parametrize("cb", ["mcg", "1mad"])
def test_encode_ties_and_non_finite_targets(te, gpu_device, K, cb):
    """Targets whose minimum is shared by many candidates (zeros, constants, magnitudes that
    swamp the codebook), and ones whose costs overflow or are NaN, where no candidate lies
    below FLT_MAX and q = 0 stands: the path equals the plain fp32 passes, bit for bit."""
    _say(f"[encode] ties and non-finite K={K} cb={cb}")
    rng = np.random.default_rng(K)
    rows = [np.zeros(256), np.tile([1.0, -1.0], 128), np.full(256, 1e6), np.full(256, -3e18),
            np.full(256, 1.5e19), np.full(256, np.inf), np.full(256, np.nan)]
    for at, v in ((0, np.nan), (127, np.inf), (128, -np.inf), (255, np.nan), (200, 1.2e19)):
        row = rng.standard_normal(256)
        row[at] = v
        rows.append(row)
    w = np.stack(rows).astype(np.float32)
    lut = tn.codebook_lut(cb)
    with np.errstate(all="ignore"):
        states = np.stack([_encode_np(r, K, lut) for r in w])
    bits_g, dq_g = te.encode_tiles(torch.from_numpy(w).to(gpu_device), K, cb)
    want = tn.pack_bits((states & ((1 << K) - 1)).astype(np.int32), K)
    assert np.array_equal(bits_g.cpu().numpy().view(np.uint32), want)
    assert np.array_equal(dq_g.cpu().numpy().view(np.uint32), lut[states].view(np.uint32))

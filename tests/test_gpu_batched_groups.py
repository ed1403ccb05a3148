"""The batched kernels' several-matrix instantiations at every column-block width, forced with
TRELLIS_BGEMM_NC: groups of members of different n and k, whole outputs against the float64
oracle and, bit for bit, against each member's own call (its one-matrix instantiation, the same
sums in the same order when the k-ranges are the same), with f32 and f16 outputs, f32 and f16
inputs, row strides above k and n, one k-range and the shortest ones, both MFMA modes."""
import sys

import numpy as np
import pytest
import torch

from oracle import trellis_np as tn

pytestmark = pytest.mark.gpu
TOL = 1e-3    # the reference's metric, max |dy| / max |y|; f16 outputs add at most 2^-11


@pytest.mark.parametrize("x_dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("nc", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("shapes,K,cb,V", [(((512, 1024), (512, 1024)), 3, "mcg", 1),
                                           (((272, 336), (1040, 528), (128, 2064)), 2, "3inst", 2),
                                           (((400, 1040), (256, 2048)), 4, "1mad", 1)])
def test_group_equals_members_and_oracle(te, gpu_device, monkeypatch, shapes, K, cb, V, nc, x_dtype):
    batch = 16 * nc + 3      # a whole column block and a ragged one
    print(f"[groups] nc={nc} shapes={shapes} K={K} cb={cb} V={V} batch={batch} x={x_dtype}", flush=True)
    sys.stdout.flush()
    lins, xs, wants = [], [], []
    rng = np.random.default_rng(batch)
    for i, (n, k) in enumerate(shapes):
        bits, rec = tn.synthetic_record(n, k, K, seed=n + k + i, codebook=cb, V=V)
        lins.append(te.PackedLinear(te.PackedRecord(rec.n, rec.k, rec.K, bits, rec.su, rec.sv, rec.isc,
                                                    rec.osc, float(rec.scale), codebook=rec.codebook,
                                                    V=rec.V), device=gpu_device))
        x = rng.standard_normal((batch, k)).astype(np.float16)
        wants.append(tn.packed_linear_ref(bits, rec, x))
        buf = torch.full((batch, k + 10), float("nan"), dtype=x_dtype, device=gpu_device)
        buf[:, 4:4 + k] = torch.from_numpy(x).to(gpu_device)
        xs.append(buf[:, 4:4 + k])
    grp = te.PackedGroup(lins)
    monkeypatch.setenv("TRELLIS_BGEMM_NC", str(nc))
    for kr in ("65536", "16"):           # one k-range of every member, and the shortest
        monkeypatch.setenv("TRELLIS_BGEMM_KR", kr)
        for f16 in (False, True):
            for dt, pad in ((torch.float32, 0), (torch.float16, 0), (torch.float32, 3), (torch.float16, 3)):
                bufs = [torch.full((batch, n + pad), 7.0, dtype=dt, device=gpu_device) for n, _ in shapes]
                outs = grp(xs, [b[:, :n] for b, (n, _) in zip(bufs, shapes)], mma_f16=f16)
                for lin, x, y, b, want in zip(lins, xs, outs, bufs, wants):
                    what = (kr, f16, dt, pad, lin.n_out, lin.k_in)
                    assert torch.equal(y, lin(x, out_dtype=dt, mma_f16=f16)), what
                    tol = TOL + (2.0 ** -11 if dt == torch.float16 else 0)
                    assert tn.rel_err(y.float().cpu().numpy(), want) < tol, what
                    rest = b[:, lin.n_out:]
                    assert torch.equal(rest, torch.full_like(rest, 7.0)), what

"""TRELLIS_BGEMM_NC outside the widths that exist (1, 2, 4, 8, 16) counts as unset: the same plan
(its workspace, on the host) and the same results (on the GPU) as without it."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import trellis_np as tn

UNLISTED = ["3", "-1", "32", "7", "x"]


def _bytes(te, n, k, batch):
    d = te._capi.TrellisDesc(bits=16, su=16, sv=16, isc_scaled=16, osc=16, n_out=n, k_in=k, K=3, V=1,
                             codebook=0, block_in=16, block_out=16, nwords=24)
    need = ctypes.c_size_t(0)
    te._capi.check(te.library().trellis_workspace_bytes(ctypes.byref(d), batch, ctypes.byref(need)))
    return need.value


@pytest.mark.parametrize("nc", UNLISTED)
def test_unlisted_width_plans_as_unset(te, monkeypatch, nc):
    monkeypatch.setenv("TRELLIS_SMALL_BATCH_GEMV", "0")
    cases = [(n, k, b) for n, k in ((256, 2048), (4096, 4096), (272, 336)) for b in (5, 12, 16, 33, 100, 513)]
    want = [_bytes(te, *c) for c in cases]
    monkeypatch.setenv("TRELLIS_BGEMM_NC", nc)
    assert [_bytes(te, *c) for c in cases] == want


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [5, 12, 16, 40])
def test_unlisted_width_results(te, gpu_device, monkeypatch, batch):
    monkeypatch.setenv("TRELLIS_SMALL_BATCH_GEMV", "0")
    bits, rec = tn.synthetic_record(256, 2048, 3, seed=5)
    lin = te.PackedLinear(te.PackedRecord(rec.n, rec.k, rec.K, bits, rec.su, rec.sv, rec.isc, rec.osc,
                                          float(rec.scale), codebook=rec.codebook, V=rec.V),
                          device=gpu_device)
    x = np.random.default_rng(batch).standard_normal((batch, 2048)).astype(np.float16)
    xt = torch.from_numpy(x).to(gpu_device)
    for f16 in (False, True):
        monkeypatch.delenv("TRELLIS_BGEMM_NC", raising=False)
        want = lin(xt, mma_f16=f16)
        monkeypatch.setenv("TRELLIS_BGEMM_NC", "3")
        assert torch.equal(lin(xt, mma_f16=f16), want)
        assert tn.rel_err(want.cpu().numpy(), tn.packed_linear_ref(bits, rec, x)) < 1e-3

"""Every column-block width of the batched kernels (32, 64, 128 and 256 columns), forced with
TRELLIS_BGEMM_NC, at the edges of their tiles against the float64 oracle: k-ranges that do not
divide among the waves (1, 3, 21, 129 tile columns: an odd last tile of a pair, waves with no
share), the last output block partly or wholly inside one band, ragged last column blocks
and 32-row chunks, outputs at addresses that forbid 16-byte stores, both MFMA modes."""
import sys

import numpy as np
import pytest
import torch

from oracle import trellis_np as tn

pytestmark = pytest.mark.gpu
TOL = 1e-3    # the reference's metric, max |dy| / max |y|; f16 outputs add at most 2^-11


@pytest.mark.parametrize("nc", [2, 4, 8, 16])
@pytest.mark.parametrize("n,k,K,cb,V,batch", [
    (16, 16, 3, "mcg", 1, 17), (144, 48, 2, "3inst", 1, 33), (272, 336, 3, "1mad", 1, 65),
    (128, 2064, 4, "mcg", 1, 97), (400, 2048, 3, "mcg", 2, 129), (96, 640, 4, "1mad", 2, 257),
    (1040, 528, 2, "mcg", 1, 31), (256, 1024, 3, "3inst", 1, 64)])
def test_widths_at_tile_edges(te, gpu_device, monkeypatch, nc, n, k, K, cb, V, batch):
    print(f"[widths] nc={nc} n={n} k={k} K={K} cb={cb} V={V} batch={batch}", flush=True)
    sys.stdout.flush()
    bits, rec = tn.synthetic_record(n, k, K, seed=n + k, codebook=cb, V=V)
    lin = te.PackedLinear(te.PackedRecord(rec.n, rec.k, rec.K, bits, rec.su, rec.sv, rec.isc, rec.osc,
                                          float(rec.scale), codebook=rec.codebook, V=rec.V),
                          device=gpu_device)
    x = np.random.default_rng(batch).standard_normal((batch, k)).astype(np.float16)
    xt = torch.from_numpy(x).to(gpu_device)
    want = tn.packed_linear_ref(bits, rec, x)
    monkeypatch.setenv("TRELLIS_BGEMM_NC", str(nc))
    for f16 in (False, True):
        for kr in ("0", "8"):      # the planner's k-range, and (one tile or pair a wave) the shortest
            monkeypatch.setenv("TRELLIS_BGEMM_KR", kr)
            y = lin(xt, mma_f16=f16)
            assert tn.rel_err(y.cpu().numpy(), want) < TOL, (f16, kr)
            assert torch.equal(y, lin(xt, mma_f16=f16)), (f16, kr)
            # rows of f16 at odd element offsets: no 4-byte alignment; the padding stays
            buf = torch.full((batch, n + 3), 7.0, dtype=torch.float16, device=gpu_device)
            lin(xt, out=buf[:, 1:1 + n], mma_f16=f16)
            assert tn.rel_err(buf[:, 1:1 + n].float().cpu().numpy(), want) < TOL + 2.0 ** -11, (f16, kr)
            pad = torch.cat([buf[:, :1], buf[:, 1 + n:]], 1)
            assert torch.equal(pad, torch.full_like(pad, 7.0)), (f16, kr)


@pytest.mark.parametrize("n,k,K,cb,V,batch,f16", [
    (144, 48, 3, "mcg", 1, 17, True), (272, 336, 2, "3inst", 2, 33, True), (128, 2064, 4, "1mad", 1, 65, True),
    (400, 1040, 3, "mcg", 1, 129, True), (96, 8192, 3, "mcg", 1, 64, True), (144, 528, 4, "mcg", 2, 257, True),
    (272, 8192, 3, "mcg", 1, 17, False), (128, 8208, 2, "3inst", 2, 64, False),
    (272, 528, 3, "mcg", 1, 65, False), (144, 1024, 2, "3inst", 1, 128, False), (96, 512, 4, "mcg", 1, 700, True)])
def test_shared_activation_kernel(te, gpu_device, monkeypatch, capfd, n, k, K, cb, V, batch, f16):
    """bgemm_shared_kernel above 16 rows, where the planner picks it (as its log says), split k
    and odd tiles included."""
    print(f"[shared] n={n} k={k} K={K} cb={cb} V={V} batch={batch} f16={f16}", flush=True)
    monkeypatch.setenv("TRELLIS_PLAN_LOG", "1")
    bits, rec = tn.synthetic_record(n, k, K, seed=n + k, codebook=cb, V=V)
    lin = te.PackedLinear(te.PackedRecord(rec.n, rec.k, rec.K, bits, rec.su, rec.sv, rec.isc, rec.osc,
                                          float(rec.scale), codebook=rec.codebook, V=rec.V),
                          device=gpu_device)
    x = np.random.default_rng(batch).standard_normal((batch, k)).astype(np.float16)
    xt = torch.from_numpy(x).to(gpu_device)
    y = lin(xt, mma_f16=f16)
    assert "shared=1" in capfd.readouterr().err
    assert tn.rel_err(y.cpu().numpy(), tn.packed_linear_ref(bits, rec, x)) < TOL
    assert torch.equal(y, lin(xt, mma_f16=f16))


@pytest.mark.parametrize("kr", ["0", "24"])      # the planner's, and one that splits the longer k
@pytest.mark.parametrize("n,k,K,cb,V,batch", [(12304, 336, 3, "mcg", 1, 129), (4112, 528, 2, "3inst", 2, 760),
                                              (12304, 336, 4, "1mad", 1, 129)])
def test_shared_exact_128_columns(te, gpu_device, monkeypatch, capfd, kr, n, k, K, cb, V, batch):
    """Its 12-wave instantiation (exact mode, 128 columns, steps of 6 tile columns), single and in
    a group, with k-ranges that end inside a step and ragged last column blocks."""
    print(f"[shared 128] n={n} k={k} K={K} cb={cb} V={V} batch={batch} kr={kr}", flush=True)
    monkeypatch.setenv("TRELLIS_PLAN_LOG", "1")
    monkeypatch.setenv("TRELLIS_BGEMM_KR", kr)
    bits, rec = tn.synthetic_record(n, k, K, seed=n + k, codebook=cb, V=V)
    lin = te.PackedLinear(te.PackedRecord(rec.n, rec.k, rec.K, bits, rec.su, rec.sv, rec.isc, rec.osc,
                                          float(rec.scale), codebook=rec.codebook, V=rec.V),
                          device=gpu_device)
    grp = te.PackedGroup([lin, lin])
    x = np.random.default_rng(batch).standard_normal((batch, k)).astype(np.float16)
    xt = torch.from_numpy(x).to(gpu_device)
    y = lin(xt)
    log = capfd.readouterr().err
    assert "shared=1" in log and " nc=8 " in log, log
    assert tn.rel_err(y.cpu().numpy(), tn.packed_linear_ref(bits, rec, x)) < TOL
    ys = grp([xt, xt])
    assert torch.equal(ys[0], ys[1]) and tn.rel_err(ys[0].cpu().numpy(), y.cpu().numpy()) < 1e-5

"""Host-side workspace sizing of the packed linear (no GPU): a run of growing batch sizes
replaces the workspace O(log n) times, and the buffers kept alive for captured graphs stay
smaller together than the current one. The size of a batch covers every smaller one."""
import ctypes
import importlib

import pytest
import torch

from conftest import PKG


class _Owner:
    def __init__(self):
        self._ws = None
        self._ws_retired = []
        self.device = torch.device("cpu")


def test_workspace_growth_is_geometric():
    pl = importlib.import_module(PKG + ".packed_linear")
    owner = _Owner()
    # prefill lengths 1..4096 on a 4096-wide linear: ~16 KB of workspace per row
    needs = [16384 * b + 1024 for b in range(1, 4097)]
    for need in needs:
        ws = pl._grow_workspace(owner, need)
        assert ws.numel() >= need
        assert ws.numel() & (ws.numel() - 1) == 0      # a power of two
        assert ws.numel() < 2 * need or ws.numel() == 256
    assert len(owner._ws_retired) <= (needs[-1]).bit_length()
    assert sum(w.numel() for w in owner._ws_retired) < owner._ws.numel()
    # a smaller request keeps the current buffer
    cur = owner._ws
    assert pl._grow_workspace(owner, 100) is cur
    assert pl._ws_size(1) == 256 and pl._ws_size(256) == 256 and pl._ws_size(257) == 512


@pytest.mark.parametrize("knob", [None, ("TRELLIS_BGEMM_NC", "1"), ("TRELLIS_BGEMM_NC", "2"),
                                  ("TRELLIS_BGEMM_NC", "16"), ("TRELLIS_SMALL_BATCH_GEMV", "0")])
@pytest.mark.parametrize("shapes", [((4096, 4096),), ((7584, 848),), ((4096, 12288),), ((512, 512),), ((16, 16),),
                                    ((4096, 4096), (1024, 4096), (1024, 4096)), ((272, 336), (1040, 2064))])
def test_size_covers_every_smaller_batch(te, monkeypatch, shapes, knob):
    """Calls check their own plan's need, which a query at that batch never reports less than:
    sizes that never fall with the batch cover every smaller call."""
    lib = te.library()
    if knob:
        monkeypatch.setenv(*knob)
    for codebook in (0, 2):
        descs = [te._capi.TrellisDesc(bits=16, su=16, sv=16, isc_scaled=16, osc=16, n_out=n, k_in=k, K=3, V=1,
                                      codebook=codebook, block_in=16, block_out=16, nwords=24)
                 for n, k in shapes]
        ptrs = (ctypes.POINTER(te._capi.TrellisDesc) * len(descs))(*[ctypes.pointer(d) for d in descs])
        need, last = ctypes.c_size_t(0), 0
        for batch in (*range(1, 300), 383, 384, 385, 511, 512, 513, 576, 577, 1023, 1024, 1025, 2048, 2049, 5000):
            te._capi.check(lib.trellis_workspace_bytes_group(ptrs, len(descs), batch, ctypes.byref(need)))
            assert need.value >= last, (batch, need.value, last)
            last = need.value


@pytest.mark.parametrize("shapes", [((4096, 4096),), ((12304, 336),), ((4864, 896), (4864, 896)), ((2048, 8192),),
                                    ((272, 336), (1040, 2064))])
def test_calls_fit_the_size(te, monkeypatch, shapes):
    """Every smaller call, in either mode and output type (which choose the kernel), passes the
    library's size check with the size of 700 rows; the address it is given is refused next
    (TRELLIS_ERR_ALIGN, 8), before anything is launched."""
    lib, n = te.library(), len(shapes)
    for codebook in (0, 2):
        descs = [te._capi.TrellisDesc(bits=16, su=16, sv=16, isc_scaled=16, osc=16, n_out=no, k_in=k, K=3, V=1,
                                      codebook=codebook, block_in=16, block_out=16, nwords=24)
                 for no, k in shapes]
        ptrs = (ctypes.POINTER(te._capi.TrellisDesc) * n)(*[ctypes.pointer(d) for d in descs])
        at = (ctypes.c_void_p * n)(*[16] * n)
        ldx = (ctypes.c_int64 * n)(*[k for _, k in shapes])
        ldy = (ctypes.c_int64 * n)(*[no for no, _ in shapes])
        need = ctypes.c_size_t(0)
        te._capi.check(lib.trellis_workspace_bytes_group(ptrs, n, 700, ctypes.byref(need)))
        for batch in range(1, 701):
            for ydt in (te._capi.DT_F32, te._capi.DT_F16):
                for flags in (0, te._capi.MMA_F16):
                    st = lib.trellis_packed_linear_group_ex(ptrs, n, at, ldx, batch, te._capi.DT_F16, at, ldy, ydt,
                                                            16, need.value, flags, None)
                    assert st == 8, (batch, ydt, flags, st)

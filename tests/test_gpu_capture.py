"""The fused scan launch inside a HIP graph: every replay works on its own
records.  A graph's replays share the epoch their flags are published under, so
without the clearing kernel of the capture a replay could take the records the
one before left, on inputs that have changed since, for its own."""
import ctypes as C

import pytest
import torch

import test_zz_no_alloc as no_alloc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("static_scratch", [False, True])
@pytest.mark.parametrize("B,T,H,N", [(1, 2048, 12, 128), (2, 600, 4, 64), (1, 64, 2, 64)])
def test_replays_on_changed_inputs_equal_eager_calls(B, T, H, N, static_scratch):
    """Five replays, the inputs changed and eager work and a synchronisation
    between them: y and the states equal an eager call's bit for bit."""
    from mamba3 import _lib
    L = _lib.lib()
    inp = no_alloc._inputs(7, B, T, H, N, 1, torch.bfloat16)
    h0, u0, a0 = inp["state"]
    st_c = _lib.SsmStateC(h0.data_ptr(), u0.data_ptr(), a0.data_ptr())
    cin = _lib.ScanInputsC(B, T, H, 64, N, 1, _lib.M3_BF16, inp["x"].data_ptr(), inp["b"].data_ptr(),
                           inp["c"].data_ptr(), inp["dt"].data_ptr(), inp["a_log"].data_ptr(),
                           inp["lam"].data_ptr(), inp["theta"].data_ptr(), inp["d_skip"].data_ptr(),
                           C.pointer(st_c), 64, 1, None, 0)
    need = int(L.m3_scan_workspace_bytes(C.byref(cin)))
    assert 0 < need <= 32 << 20
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    cin.workspace, cin.workspace_bytes = ws.data_ptr(), need
    y = torch.empty_like(inp["x"])
    h, u, ang = torch.empty_like(h0), torch.empty_like(u0), torch.empty_like(a0)
    cout = _lib.ScanOutputC(y.data_ptr(), _lib.SsmStateC(h.data_ptr(), u.data_ptr(), ang.data_ptr()))
    fn = L.m3_scan_no_alloc if static_scratch else L.m3_scan
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    before = L.m3_launch_count()
    with torch.cuda.graph(graph, stream=side):
        _lib.check(fn(C.byref(cin), C.byref(cout), C.c_void_p(side.cuda_stream)))
    assert L.m3_launch_count() - before == 2   # the flags, and the one fused launch
    for rep in range(5):
        for t in (y, h, u, ang):
            t.fill_(float("nan"))
        if rep:
            inp["x"].copy_(torch.randn_like(inp["x"]))
            h0.normal_()
            inp["dt"].mul_(0.9)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        ref = no_alloc._call(inp, no_alloc=False)
        for name, r, got in zip(("y", "h", "last_u", "angle"), ref[:4], (y, h, u, ang)):
            assert torch.equal(r, got), (rep, name)

"""The two GEMM launches of the dual-expert FFN as one launch (wx_dual_swiglu_ffn_fused: gate/up tiles and down tiles in
one grid, a down tile waiting on counters for the gate/up tiles of its rows) against the two launches it replaces
(act.py:79-82, 142-154 per expert): bit-equal results, a workspace that every call leaves zero, the shapes it hands
back to the two launches, and HIP graph replays."""

import pytest
import torch

import oracle
from wallx_mi355 import _lib, native

pytestmark = pytest.mark.gpu


def _case(dev, T, m0, H, I0, I1, seed):
    g = torch.Generator().manual_seed(seed)
    ws = [(torch.randn(s, generator=g) * 0.03).to(torch.bfloat16).to(dev)
          for s in ((I0, H), (I0, H), (H, I0), (I1, H), (I1, H), (H, I1))]
    packed = [native.pack_weight(w, cache=False) for w in ws]
    types = torch.cat([torch.zeros(m0, dtype=torch.bool), torch.ones(T - m0, dtype=torch.bool)])
    types = types[torch.randperm(T, generator=g)].to(dev)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    res = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    rmap, off, inv, _ = native.partition(types, 2, 0, None, want_sorted=True)
    xt = native.permute_rows_tiled(x, rmap, off, None, inv)
    return ws, packed, types, x, res, off, inv, xt


def _workspace(dev):
    return torch.zeros(_lib.load().wx_ffn_fused_workspace_bytes() // 4, dtype=torch.int32, device=dev)


def _two_launches(p, xt, hm, out, res, off, inv, T, H, I0, I1, rows, stream):
    _lib.call("wx_dual_swiglu_gate_up", xt.data_ptr(), hm.data_ptr(), off.data_ptr(), p[0], p[1], p[3], p[4], T, H, I0, I1,
              rows, stream)
    if res is not None:
        _lib.call("wx_dual_down_proj_residual", hm.data_ptr(), out.data_ptr(), res.data_ptr(), off.data_ptr(), p[2], p[5],
                  T, H, I0, I1, rows, inv.data_ptr(), stream)
    else:
        _lib.call("wx_dual_down_proj", hm.data_ptr(), out.data_ptr(), off.data_ptr(), p[2], p[5], T, H, I0, I1, rows,
                  inv.data_ptr(), stream)


def _one_launch(p, xt, hm, out, res, off, inv, T, H, I0, I1, rows, ws, stream, x_rows=None):
    """x_rows: the activations in token order; xt is then the buffer that the call permutes them into."""
    _lib.call("wx_dual_swiglu_ffn_fused", None if x_rows is None else x_rows.data_ptr(), xt.data_ptr(), out.data_ptr(),
              None if res is None else res.data_ptr(), off.data_ptr(), p[0], p[1], p[2], p[3], p[4], p[5], hm.data_ptr(),
              T, H, I0, I1, rows, inv.data_ptr(), None if ws is None else ws.data_ptr(), stream)


# one round of 128 x 128 tiles per GEMM (the shapes that run as one launch): a denoise step's 2048 action tokens, all
# rows on expert 0, both experts with ragged tiles, a single row on one expert; then shapes that go to two launches
@pytest.mark.parametrize("T,m0,H,I0,I1,with_res,known_rows", [
    (2048, 0, 2048, 1536, 1024, False, True), (2048, 0, 2048, 1536, 1024, True, True), (1024, 1024, 256, 512, 1024, False, True),
    (1500, 700, 512, 448, 320, True, True), (129, 1, 1024, 64, 1024, False, True), (300, 300, 96, 32, 32, True, True),
    (2048, 0, 2048, 1536, 1024, False, False),   # rows only known on the device: too many for the one launch ...
    (512, 0, 2048, 1536, 1024, False, False), (300, 200, 512, 448, 320, True, False),   # ... and few enough for it
    (4096, 100, 2048, 1024, 1024, True, True),   # more tiles than CUs
])
def test_one_launch_ffn_equals_two_launches(dev, T, m0, H, I0, I1, with_res, known_rows):
    ws_, packed, types, x, res, off, inv, xt = _case(dev, T, m0, H, I0, I1, T + H + I0)
    p = [t.data_ptr() for t in packed]
    stream = torch.cuda.current_stream().cuda_stream
    pad = native.padded_sorted_rows(T)
    hm = [torch.zeros(pad * max(I0, I1), dtype=torch.bfloat16, device=dev) for _ in range(2)]
    out = [torch.full((T, H), v, dtype=torch.bfloat16, device=dev) for v in (7.0, 9.0)]
    rows = _lib.i64x2((m0, T - m0)) if known_rows else None
    r = res if with_res else None
    work = _workspace(dev)
    _two_launches(p, xt, hm[0], out[0], r, off, inv, T, H, I0, I1, rows, stream)
    xt2 = torch.full_like(xt, 3.0)
    for call in range(4):  # every call after the first runs on the workspace the one before it left
        out[1].fill_(9.0)
        if call < 2:
            _one_launch(p, xt, hm[1], out[1], r, off, inv, T, H, I0, I1, rows, work, stream)
        else:  # ... and with the permute inside the launch (the gate/up tiles read the token rows)
            _one_launch(p, xt2, hm[1], out[1], r, off, inv, T, H, I0, I1, rows, work, stream, x_rows=x)
        torch.cuda.synchronize()
        assert torch.equal(out[0], out[1]), f"call {call}"
        assert torch.equal(hm[0], hm[1]), f"call {call}"
        assert int(work.abs().sum()) == 0, f"call {call}: counters or the error flag left set"
    # against the oracle
    wc = [tuple(w.cpu() for w in ws_[:3]), tuple(w.cpu() for w in ws_[3:])]
    ref = oracle.sparse_moe_block_ref(x.cpu()[None], types.cpu()[None], wc)[0].float()
    if with_res:
        ref = (res.cpu().float() + ref).to(torch.bfloat16).float()
    err = (out[1].cpu().float() - ref).abs()
    assert not (err > 2e-2 + 1e-2 * ref.abs()).any(), float(err.max())


@pytest.mark.parametrize("hint", [(4096, 0), (3968, 128), (128, 3968), (0, 4096)])
def test_one_launch_ffn_with_row_counts_that_are_not_the_devices(dev, hint):
    """The host's row counts choose the launch; the kernels read the split from expert_offsets.  Counts that are not
    the device's (here 2049 + 2047 rows) may pick the one launch for a problem with more tiles than it has workgroups
    for -- gate/up workgroups then take several tiles each, and so do down workgroups, each tile behind its own wait
    -- and the result does not change."""
    T, m0, H, I0, I1 = 4096, 2049, 1024, 64, 1024
    _, packed, _, x, res, off, inv, xt = _case(dev, T, m0, H, I0, I1, 17)
    p = [t.data_ptr() for t in packed]
    stream = torch.cuda.current_stream().cuda_stream
    pad = native.padded_sorted_rows(T)
    hm = [torch.zeros(pad * max(I0, I1), dtype=torch.bfloat16, device=dev) for _ in range(2)]
    out = [torch.full((T, H), v, dtype=torch.bfloat16, device=dev) for v in (7.0, 9.0)]
    work = _workspace(dev)
    _two_launches(p, xt, hm[0], out[0], res, off, inv, T, H, I0, I1, None, stream)
    xt2 = torch.full_like(xt, 3.0)
    for call in range(2):
        if call == 0:
            _one_launch(p, xt, hm[1], out[1], res, off, inv, T, H, I0, I1, _lib.i64x2(hint), work, stream)
        else:
            _one_launch(p, xt2, hm[1], out[1], res, off, inv, T, H, I0, I1, _lib.i64x2(hint), work, stream, x_rows=x)
        torch.cuda.synchronize()
        assert torch.equal(out[0], out[1]) and torch.equal(hm[0], hm[1]), f"call {call}"
        assert int(work.abs().sum()) == 0


def test_one_launch_ffn_without_a_workspace_is_the_two_launches(dev):
    T, m0, H, I0, I1 = 700, 200, 256, 384, 128
    _, packed, _, _, _, off, inv, xt = _case(dev, T, m0, H, I0, I1, 5)
    p = [t.data_ptr() for t in packed]
    stream = torch.cuda.current_stream().cuda_stream
    pad = native.padded_sorted_rows(T)
    hm = [torch.zeros(pad * max(I0, I1), dtype=torch.bfloat16, device=dev) for _ in range(2)]
    out = [torch.empty(T, H, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    rows = _lib.i64x2((m0, T - m0))
    _two_launches(p, xt, hm[0], out[0], None, off, inv, T, H, I0, I1, rows, stream)
    _one_launch(p, xt, hm[1], out[1], None, off, inv, T, H, I0, I1, rows, None, stream)
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1]) and torch.equal(hm[0], hm[1])
    lib = _lib.load()
    work = _workspace(dev)
    assert lib.wx_dual_swiglu_ffn_fused(None, xt.data_ptr(), out[1].data_ptr(), None, off.data_ptr(), *p, hm[1].data_ptr(),
                                        T, H, I0, I1, rows, inv.data_ptr(), work.data_ptr() + 2, stream) == -1
    assert b"aligned" in lib.wx_last_error_string()
    assert lib.wx_dual_swiglu_ffn_fused(None, xt.data_ptr(), out[1].data_ptr(), out[0].data_ptr(), off.data_ptr(), *p,
                                        hm[1].data_ptr(), T, H, I0, I1, rows, None, work.data_ptr(), stream) == -1
    assert b"out_row_id" in lib.wx_last_error_string()  # a residual is added in token order
    assert lib.wx_dual_swiglu_ffn_fused(out[0].data_ptr(), xt.data_ptr(), out[1].data_ptr(), None, off.data_ptr(), *p,
                                        hm[1].data_ptr(), T, H, I0, I1, rows, None, work.data_ptr(), stream) == -1
    assert b"out_row_id" in lib.wx_last_error_string()  # ... and rows are gathered through it


def test_one_launch_ffn_replays_from_a_hip_graph(dev):
    """Captured once, replayed with the program's own eager launches and synchronisations in between: every replay
    equals the eager result, and the counters are zero after each."""
    T, m0, H, I0, I1 = 2048, 0, 1024, 512, 1024
    _, packed, _, x, res, off, inv, xt = _case(dev, T, m0, H, I0, I1, 11)
    p = [t.data_ptr() for t in packed]
    pad = native.padded_sorted_rows(T)
    rows = _lib.i64x2((m0, T - m0))
    hm = [torch.zeros(pad * max(I0, I1), dtype=torch.bfloat16, device=dev) for _ in range(2)]
    out = [torch.empty(T, H, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    work = _workspace(dev)
    _two_launches(p, xt, hm[0], out[0], res, off, inv, T, H, I0, I1, rows, torch.cuda.current_stream().cuda_stream)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _one_launch(p, xt, hm[1], out[1], res, off, inv, T, H, I0, I1, rows, work, side.cuda_stream)
    torch.cuda.current_stream().wait_stream(side)
    xt2 = torch.zeros_like(xt)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _one_launch(p, xt2, hm[1], out[1], res, off, inv, T, H, I0, I1, rows, work,
                    torch.cuda.current_stream().cuda_stream, x_rows=x)
    for replay in range(4):
        out[1].zero_()
        hm[1].zero_()
        xt2.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], out[1]) and torch.equal(hm[0], hm[1]), f"replay {replay}"
        assert int(work.abs().sum()) == 0
        # eager work of the program between replays, on the same workspace
        _one_launch(p, xt, hm[1], out[1], res, off, inv, T, H, I0, I1, rows, work, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("residual", [False, True])
def test_block_forward_with_and_without_the_one_launch_ffn(dev, residual, monkeypatch):
    """native.packed_block_forward (wx_moe_block_forward) hands the library its per-stream counter workspace; switched
    off, it makes the two launches.  Same bits."""
    T, H, I0, I1 = 1024, 512, 768, 256
    g = torch.Generator().manual_seed(3)
    ws = [(torch.randn(s, generator=g) * 0.05).to(torch.bfloat16).to(dev)
          for s in ((I0, H), (I0, H), (H, I0), (I1, H), (I1, H), (H, I1))]
    experts = native.PackedExperts([native.pack_weight(w, cache=False) for w in ws], (H, I0, I1))
    types = (torch.rand(T, generator=g) < 0.3).to(dev)
    x = (torch.randn(T, H, generator=g) * 2.0).to(torch.bfloat16).to(dev)
    rmap, off, inv, _ = native.partition(types, 2, 0, None, want_sorted=True)
    n1 = int(types.sum())
    rows = _lib.i64x2((T - n1, n1))
    got = {}
    for flag in (True, False):
        monkeypatch.setattr(native, "_one_launch_ffn", flag)  # (what native.set_one_launch_ffn sets)
        got[flag] = native.packed_block_forward(experts, x, rmap, inv, off, rows, residual=residual)
    torch.cuda.synchronize()
    assert torch.equal(got[True], got[False])


def test_one_launch_ffn_on_two_streams_at_once(dev):
    """Two streams issue the one launch at the same time, each with a workspace of its own (what
    native.packed_block_forward keeps per stream): workgroups of both launches share the CUs, each launch's down tiles
    wait on its own counters, and both results are those of the separate launches.  (With two such launches resident
    an XCD's 64 workgroup places cannot all be held by waiting down workgroups of the other launch -- one launch has
    at most 32 of them per XCD -- so the gate/up workgroups of either always find a place.)"""
    T, m0, H, I0, I1 = 2048, 0, 2048, 1536, 1024
    pad = native.padded_sorted_rows(T)
    rows = _lib.i64x2((m0, T - m0))
    lanes = []
    for seed in (21, 22):
        _, packed, _, x, res, off, inv, xt = _case(dev, T, m0, H, I0, I1, seed)
        p = [t.data_ptr() for t in packed]
        hm = [torch.zeros(pad * max(I0, I1), dtype=torch.bfloat16, device=dev) for _ in range(2)]
        out = [torch.empty(T, H, dtype=torch.bfloat16, device=dev) for _ in range(2)]
        _two_launches(p, xt, hm[0], out[0], res, off, inv, T, H, I0, I1, rows, torch.cuda.current_stream().cuda_stream)
        lanes.append(dict(packed=packed, p=p, x=x, res=res, off=off, inv=inv, xt=torch.zeros_like(xt), hm=hm, out=out,
                          work=_workspace(dev), stream=torch.cuda.Stream()))
    torch.cuda.synchronize()
    for rep in range(3):
        for ln in lanes:
            ln["out"][1].zero_()
            ln["hm"][1].zero_()
        torch.cuda.synchronize()
        for _ in range(12):  # the host issues faster than a launch runs: the two streams' launches overlap
            for ln in lanes:
                _one_launch(ln["p"], ln["xt"], ln["hm"][1], ln["out"][1], ln["res"], ln["off"], ln["inv"], T, H, I0, I1,
                            rows, ln["work"], ln["stream"].cuda_stream, x_rows=ln["x"])
        torch.cuda.synchronize()
        for i, ln in enumerate(lanes):
            assert torch.equal(ln["out"][0], ln["out"][1]) and torch.equal(ln["hm"][0], ln["hm"][1]), f"rep {rep} stream {i}"
            assert int(ln["work"].abs().sum()) == 0, f"rep {rep} stream {i}: counters or the error flag left set"


# Few rows (a denoise step of one robot, or a few): tiles of 16 or 32 rows whose contraction is cut over a workgroup's
# wavefronts.  The edges of its row blocks, both tile heights, the last row count it takes at these widths (256) and the
# first it does not, both experts, and a hidden size whose last column tile is half empty.
@pytest.mark.parametrize("T,m0,H,I0,I1", [
    (1, 0, 2048, 1536, 1024), (15, 0, 2048, 1536, 1024), (16, 0, 2048, 1536, 1024), (17, 0, 2048, 1536, 1024),
    (32, 0, 2048, 1536, 1024), (128, 0, 2048, 1536, 1024), (129, 0, 2048, 1536, 1024), (217, 0, 2048, 1536, 1024),
    (256, 0, 2048, 1536, 1024), (257, 0, 2048, 1536, 1024), (40, 23, 512, 448, 96), (33, 33, 288, 64, 32),
    (50, 1, 1280, 320, 1024), (1024, 700, 256, 64, 32),
    # a wide expert: without row counts the large tiles are launched as well, and the device settles which form runs
    (32, 0, 2048, 11008, 1024), (217, 3, 2048, 11008, 1024), (256, 0, 2048, 11008, 1024),
])
def test_few_rows(dev, T, m0, H, I0, I1):
    ws_, packed, types, x, res, off, inv, xt = _case(dev, T, m0, H, I0, I1, T + H)
    p = [t.data_ptr() for t in packed]
    stream = torch.cuda.current_stream().cuda_stream
    pad = native.padded_sorted_rows(T)
    rows = _lib.i64x2((m0, T - m0))
    work = _workspace(dev)
    got = []
    for form in range(5):  # one launch and two, with and without the row counts on the host, and with the permute inside
        hm = torch.zeros(pad * max(I0, I1), dtype=torch.bfloat16, device=dev)
        out = torch.full((T, H), 7.0, dtype=torch.bfloat16, device=dev)
        known = rows if form % 2 == 0 else None
        if form < 2:
            _two_launches(p, xt, hm, out, res, off, inv, T, H, I0, I1, known, stream)
        else:
            _one_launch(p, xt, hm, out, res, off, inv, T, H, I0, I1, known, work, stream, x_rows=x if form == 4 else None)
        torch.cuda.synchronize()
        assert int(work.abs().sum()) == 0, f"form {form}"
        got.append((out, hm))
    for form, (out, hm) in enumerate(got):
        assert torch.equal(out, got[0][0]) and torch.equal(hm, got[0][1]), f"form {form}"
    wc = [tuple(w.cpu() for w in ws_[:3]), tuple(w.cpu() for w in ws_[3:])]
    ref = oracle.sparse_moe_block_ref(x.cpu()[None], types.cpu()[None], wc)[0].float()
    ref = (res.cpu().float() + ref).to(torch.bfloat16).float()
    err = (got[0][0].cpu().float() - ref).abs()
    # (the bound of the other tests of this FFN: bf16 steps of the intermediate and of the result)
    assert not (err > 2e-2 + 1e-2 * ref.abs()).any(), float(err.max())


@pytest.mark.parametrize("T,m0,H,I0,I1", [(32, 0, 2048, 1536, 1024), (217, 0, 2048, 1536, 1024), (19, 0, 768, 512, 1024),
                                          (40, 23, 512, 448, 96), (1, 0, 256, 64, 32),
                                          (9, 4, 1024, 64, 32), (9, 4, 1280, 64, 32), (9, 4, 1536, 64, 32), (9, 4, 1792, 64, 32)])
def test_few_rows_with_the_norm_inside(dev, T, m0, H, I0, I1):
    """The RMSNorm inside the few-rows launch gives what the norm's own launch gives, bit for bit; row counts on the host
    that are not the device's change neither the launch's result nor its workspace.  (217 rows have tiles of 32 rows and a norm
    of their own again.)"""
    _, packed, types, x, _, off, inv, _ = _case(dev, T, m0, H, I0, I1, T + H + 1)
    rmap = native.partition(types, 2, 0, None, want_sorted=True)[0]
    experts = native.PackedExperts(packed, (H, I0, I1))
    norm = (torch.randn(H, generator=torch.Generator().manual_seed(3)) * 0.1 + 1).to(torch.bfloat16).to(dev)

    def run(rows, one):
        old = native.set_one_launch_ffn(one)
        try:
            return native.packed_block_forward(experts, x, rmap, inv, off, rows, (norm, 1e-6), True)
        finally:
            native.set_one_launch_ffn(old)

    want = run(_lib.i64x2((m0, T - m0)), False)
    assert torch.equal(run(_lib.i64x2((m0, T - m0)), True), want)
    assert torch.equal(run(_lib.i64x2((m0, T - m0)), True), want)  # on the workspace the call before it left
    assert torch.equal(run(None, True), want)
    if m0 == 0:
        assert torch.allclose(run(_lib.i64x2((T, 0)), True).float(), want.float(), rtol=1e-2, atol=2e-2)
    torch.cuda.synchronize()


# The tile shapes of the one launch at their edges (its rows are taken for the narrow expert's where the host does not know
# better), several tiles per workgroup on a wide expert and on a mix, a contraction longer than one round of loads, and hidden
# sizes whose last column tile is short.
@pytest.mark.parametrize("T,m0,H,I0,I1", [
    (33, 0, 2048, 11008, 1024), (64, 0, 2048, 11008, 1024), (65, 1, 2048, 11008, 1024), (128, 64, 2048, 11008, 1024),
    (129, 128, 2048, 11008, 1024), (224, 0, 2048, 1536, 1024), (225, 0, 2048, 1536, 1024), (256, 200, 2048, 4096, 1024),
    (31, 31, 2048, 11008, 1024), (70, 70, 4096, 96, 64), (40, 9, 288, 320, 32), (200, 100, 1056, 640, 96),
    # one expert's tiles behind the other's, in the gate/up part and in the down part, the first expert's and the second's
    (256, 248, 2048, 11008, 1024), (128, 120, 2048, 11008, 1024), (256, 8, 2048, 1024, 4096), (250, 3, 512, 96, 4064),
    # more rows than CUs: a row block more than the grid has eights of workgroups for, and one tile to every CU
    (512, 504, 256, 64, 32), (992, 496, 512, 256, 256), (1024, 1017, 256, 32, 64),
])
def test_few_rows_tiles_whatever_rows_the_host_expects(dev, T, m0, H, I0, I1):
    """One launch equals two, bit for bit, with the row counts known, unknown, and not the device's; with the norm inside it
    equals the norm's own launch and those."""
    ws_, packed, types, x, res, off, inv, xt = _case(dev, T, m0, H, I0, I1, T + I0)
    p = [t.data_ptr() for t in packed]
    stream = torch.cuda.current_stream().cuda_stream
    pad = native.padded_sorted_rows(T)
    work = _workspace(dev)
    hm = [torch.zeros(pad * max(I0, I1), dtype=torch.bfloat16, device=dev) for _ in range(2)]
    out = [torch.full((T, H), 7.0, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    _two_launches(p, xt, hm[0], out[0], res, off, inv, T, H, I0, I1, None, stream)
    for counts in ((m0, T - m0), None, (0, T), (T, 0), (T // 2, T - T // 2)):
        for rows_in in (x, None):
            out[1].fill_(9.0)
            hm[1].zero_()
            _one_launch(p, xt, hm[1], out[1], res, off, inv, T, H, I0, I1, None if counts is None else _lib.i64x2(counts), work,
                        stream, x_rows=rows_in)
            torch.cuda.synchronize()
            assert torch.equal(out[0], out[1]) and torch.equal(hm[0], hm[1]), f"counts {counts}"
            assert int(work.abs().sum()) == 0, f"counts {counts}"
    wc = [tuple(w.cpu() for w in ws_[:3]), tuple(w.cpu() for w in ws_[3:])]
    ref = oracle.sparse_moe_block_ref(x.cpu()[None], types.cpu()[None], wc)[0].float()
    ref = (res.cpu().float() + ref).to(torch.bfloat16).float()
    err = (out[0].cpu().float() - ref).abs()
    # (the bound of the other tests of this FFN, widened with the root of the contraction where it is longer than theirs)
    assert not (err > 2e-2 * max(1.0, I0 / 2048) ** 0.5 + 1e-2 * ref.abs()).any(), float(err.max())
    if H % 256 == 0 and H <= 2048:
        rmap = native.partition(types, 2, 0, None, want_sorted=True)[0]
        experts = native.PackedExperts(packed, (H, I0, I1))
        norm = (torch.randn(H, generator=torch.Generator().manual_seed(3)) * 0.1 + 1).to(torch.bfloat16).to(dev)
        got = []
        for one, counts in ((False, (m0, T - m0)), (True, (m0, T - m0)), (True, None), (True, (0, T)), (True, (T, 0))):
            old = native.set_one_launch_ffn(one)
            try:
                got.append(native.packed_block_forward(experts, x, rmap, inv, off, None if counts is None else _lib.i64x2(counts),
                                                       (norm, 1e-6), True))
            finally:
                native.set_one_launch_ffn(old)
        assert all(torch.equal(got[0], g) for g in got[1:])


@pytest.mark.parametrize("T,m0,H,I0,I1", [(33, 0, 512, 448, 256), (40, 23, 512, 448, 96), (200, 90, 256, 384, 128)])
def test_few_rows_keep_the_projections(dev, T, m0, H, I0, I1):
    """With the gate and up projections kept for a backward pass the intermediate is the same, and it is their SwiGLU."""
    _, packed, _, _, _, off, inv, xt = _case(dev, T, m0, H, I0, I1, T)
    p = [t.data_ptr() for t in packed]
    stream = torch.cuda.current_stream().cuda_stream
    pad0, pad1 = (m0 + 255) // 256 * 256, (T - m0 + 255) // 256 * 256
    n = native.padded_sorted_rows(T) * max(I0, I1)
    hm, hk, gate, up = (torch.zeros(n, dtype=torch.bfloat16, device=dev) for _ in range(4))
    for rows in (_lib.i64x2((m0, T - m0)), None):
        _lib.call("wx_dual_swiglu_gate_up", xt.data_ptr(), hm.data_ptr(), off.data_ptr(), p[0], p[1], p[3], p[4], T, H, I0, I1,
                  rows, stream)
        _lib.call("wx_dual_swiglu_gate_up_keep", xt.data_ptr(), hk.data_ptr(), gate.data_ptr(), up.data_ptr(), off.data_ptr(),
                  p[0], p[1], p[3], p[4], T, H, I0, I1, rows, stream)
        torch.cuda.synchronize()
        used = pad0 * I0 + pad1 * I1
        assert torch.equal(hm, hk)
        want = torch.nn.functional.silu(gate[:used].float()).to(torch.bfloat16).float() * up[:used].float()
        # one bf16 step of silu(gate) and one of the product
        assert torch.allclose(hk[:used].float(), want, rtol=2.0 ** -6, atol=1e-6)
        assert float(gate.abs().max()) > 0 and float(up.abs().max()) > 0


def _norm_block(dev, T, seed):
    """A few-rows block with the norm inside: (forward of x into out through the C ABI on a stream, x, row counts)."""
    H, I0, I1 = 2048, 1536, 1024
    _, packed, types, x, _, off, inv, _ = _case(dev, T, 0, H, I0, I1, seed)
    rmap = native.partition(types, 2, 0, None, want_sorted=True)[0]
    experts = native.PackedExperts(packed, (H, I0, I1))
    norm = (torch.randn(H, generator=torch.Generator().manual_seed(seed)) * 0.1 + 1).to(torch.bfloat16).to(dev)
    x_elems, h_elems = experts.sizes(T)
    xt, hm = (torch.zeros(n, dtype=torch.bfloat16, device=dev) for n in (x_elems, h_elems))
    work, rows = _workspace(dev), _lib.i64x2((0, T))

    def run(x, out, stream, one=True):
        _lib.call("wx_moe_block_forward", x.data_ptr(), out.data_ptr(), rmap.data_ptr(), inv.data_ptr(), off.data_ptr(),
                  *experts.ptrs, xt.data_ptr(), hm.data_ptr(), T, H, I0, I1, rows, norm.data_ptr(), 1e-6, 1,
                  work.data_ptr() if one else None, stream)

    return run, x, work, (packed, norm, experts)


@pytest.mark.parametrize("rows", [(32, 117), (217, 256), (217, 32), (129, 224)])
def test_few_rows_with_the_norm_in_place_on_two_streams_and_replayed(dev, rows):
    """The one launch with the norm where its output is its input, on two streams at once, and from a HIP graph whose
    input changes between replays: the separate launches' bits, and a workspace that is zero again.  Up to 128 rows two
    workgroups share a CU and a launch's waiting ones take 32 of an XCD's 64 places at most; from 129 rows on a workgroup has
    its CU to itself, and at most 31 of an XCD's 32 are taken by a launch that waits.  Both kinds, and one of each."""
    blocks = [_norm_block(dev, T, seed) for T, seed in zip(rows, (31, 32))]
    here = torch.cuda.current_stream().cuda_stream
    want = []
    for run, x, work, _ in blocks:
        want.append(torch.empty_like(x))
        run(x, want[-1], here, one=False)
        y = x.clone()
        run(y, y, here)  # in place
        assert torch.equal(y, want[-1])
    streams = [torch.cuda.Stream() for _ in blocks]
    outs = [torch.zeros_like(x) for _, x, _, _ in blocks]
    torch.cuda.synchronize()
    for _ in range(20):
        for (run, x, _, _), out, st in zip(blocks, outs, streams):
            run(x, out, st.cuda_stream)
    torch.cuda.synchronize()
    for (_, _, work, _), out, ref in zip(blocks, outs, want):
        assert torch.equal(out, ref) and int(work.abs().sum()) == 0

    run, x, work, _ = blocks[0]
    still, out = x.clone(), torch.empty_like(x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(still, out, torch.cuda.current_stream().cuda_stream)
    for scale in (1.0, 0.5, 3.0):
        still.copy_(x * scale)
        ref = torch.empty_like(x)
        run(still, ref, here, one=False)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and int(work.abs().sum()) == 0

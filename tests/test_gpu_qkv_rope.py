"""GPU parity of the q / k / v projection with M-RoPE in the GEMM epilogue (vl.py:955-964 as one launch) against the
oracle: an fp32 linear layer rounded to bf16, then mrope_apply_ref in eager bf16, in both channel layouts (the
PyTorch path's, vl.py:763-769, and the CUDA kernel's, csrc/rope.cu:104-117, which the flash-attention class of
vl.py:962-964 runs).  Tolerance |x - ref| <= 2e-2 + 1e-2 |ref|."""

import pytest
import torch
import torch.nn.functional as F

import oracle
from wallx_mi355 import _lib, native, workloads as wl
from wallx_mi355.fusions import ops

pytestmark = pytest.mark.gpu


def _close(got, ref, what):
    got, ref = got.float().cpu(), ref.float()
    assert got.shape == ref.shape, what
    err = (got - ref).abs()
    bad = err > 2e-2 + 1e-2 * ref.abs()
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()} outside tolerance, max abs err {float(err.max())}"


def _reference(x, w, b, pos, nq, nkv, rows=None, layout="hf"):
    """(q, k, v) [B, H, S, D] from the oracle; rows: optional token subset (flattened indices) to evaluate."""
    B, S, H = x.shape
    D = 128
    xf = x.reshape(B * S, H)
    cos, sin = oracle.rotary_cos_sin_ref(pos, wl.text_inv_freq(), torch.bfloat16)
    if rows is not None:
        xf = xf[rows]
        cos = cos.reshape(3, 1, B * S, D)[:, :, rows]
        sin = sin.reshape(3, 1, B * S, D)[:, :, rows]
        B, S = 1, rows.numel()
    qkv = F.linear(xf.float(), w.float(), None if b is None else b.float()).to(torch.bfloat16)
    q, k, v = qkv.split([nq * D, nkv * D, nkv * D], dim=-1)
    q = q.reshape(B, S, nq, D).transpose(1, 2)
    k = k.reshape(B, S, nkv, D).transpose(1, 2)
    v = v.reshape(B, S, nkv, D).transpose(1, 2)
    rq, rk = oracle.mrope_apply_ref(q, k, cos, sin, list(wl.MROPE_SECTION), layout, eager_rounding=True)
    return rq, rk, v


@pytest.mark.parametrize("layout", ["hf", "csrc"])
@pytest.mark.parametrize("B,S,H,nq,nkv,with_bias", [(2, 300, 512, 4, 2, True), (1, 37, 256, 2, 1, False),
                                                   (3, 256, 1024, 3, 1, True), (1, 1, 64, 1, 1, True),
                                                   # more than a round of large tiles; the last 104 rows are a strip of small ones
                                                   (2, 436, 64, 160, 1, True)])
def test_qkv_rope_projection(dev, B, S, H, nq, nkv, with_bias, layout):
    g = torch.Generator().manual_seed(B * 1000 + S)
    x = torch.randn(B, S, H, generator=g).to(torch.bfloat16)
    n = (nq + 2 * nkv) * 128
    w = (torch.randn(n, H, generator=g) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, generator=g) * 0.5).to(torch.bfloat16) if with_bias else None
    pos = torch.stack([torch.randint(0, 60, (B, S), generator=g), torch.randint(100, 160, (B, S), generator=g),
                       torch.randint(300, 360, (B, S), generator=g)])  # distinct planes
    width = 64 if layout == "hf" else 128  # the CUDA kernel's layout rotates d and d + 64 by different planes
    table = ops.multimodal_rope_table(pos.to(dev), wl.text_inv_freq().to(dev), wl.MROPE_SECTION, layout)
    assert table.shape == (B * S, width) and table.dtype == torch.int32
    # the table itself: bf16 cos / sin of the oracle's builder, packed
    cos, sin = oracle.rotary_cos_sin_ref(pos, wl.text_inv_freq(), torch.bfloat16)
    amap = oracle.mrope_axis_map(wl.MROPE_SECTION, 128, layout)[:width]
    cos_sel = cos[amap, :, :, torch.arange(width)].permute(1, 2, 0).reshape(B * S, width)
    sin_sel = sin[amap, :, :, torch.arange(width)].permute(1, 2, 0).reshape(B * S, width)
    tb = table.cpu()
    got_cos = (tb << 16).view(torch.float32)
    got_sin = (tb & -65536).view(torch.float32)
    assert float((got_cos != cos_sel.float()).float().mean()) < 5e-3  # sincosf of the device vs the host: a bf16 step now and then
    assert float((got_sin != sin_sel.float()).float().mean()) < 5e-3
    assert bool(((got_cos - cos_sel.float()).abs() <= 2.0 ** -7).all()) and bool(((got_sin - sin_sel.float()).abs() <= 2.0 ** -7).all())
    q, k, v = ops.qkv_projection_with_rope(x.to(dev), w.to(dev), None if b is None else b.to(dev), table, nq, nkv)
    assert q.shape == (B, nq, S, 128) and k.shape == (B, nkv, S, 128) and v.shape == (B, nkv, S, 128)
    rq, rk, rv = _reference(x, w, b, pos, nq, nkv, layout=layout)
    if layout == "csrc":  # the two layouts must not coincide on these positions (distinct planes)
        hq, _, _ = _reference(x, w, b, pos, nq, nkv, layout="hf")
        assert not torch.equal(hq, rq)
    _close(q, rq, "q")
    _close(k, rk, "k")
    _close(v, rv, "v")
    # the same numbers as the two-step path on the device (projection by torch, then the rope kernel from positions)
    qkv = F.linear(x.to(dev), w.to(dev), None if b is None else b.to(dev))
    q2, k2, _ = qkv.split([nq * 128, nkv * 128, nkv * 128], dim=-1)
    gq, gk = ops.multimodal_rope_from_positions(q2.reshape(B, S, nq, 128).transpose(1, 2), k2.reshape(B, S, nkv, 128).transpose(1, 2),
                                                pos.to(dev), wl.text_inv_freq().to(dev), list(wl.MROPE_SECTION), layout)
    _close(q, gq.cpu(), "q vs two-step path")
    _close(k, gk.cpu(), "k vs two-step path")


def test_qkv_rope_projection_config5_shape(dev):
    """The prefill shape: 16 x 912 tokens, hidden 2048, 16 query and 2 KV heads (N = 2560); the oracle on a sample of
    tokens, every column."""
    ids, grid = wl.config2_tokens(batch=16, tail_text=96)
    pos, _ = oracle.rope_index_ref(ids, 2, wl.IMAGE_TOKEN_ID, wl.VIDEO_TOKEN_ID, wl.VISION_START_TOKEN_ID, 2,
                                   image_grid_thw=grid)
    B, S = ids.shape
    g = torch.Generator().manual_seed(7)
    x = torch.randn(B, S, 2048, generator=g).to(torch.bfloat16)
    w = (torch.randn(2560, 2048, generator=g) * 0.02).to(torch.bfloat16)
    b = (torch.randn(2560, generator=g) * 0.02).to(torch.bfloat16)
    table = ops.multimodal_rope_table(pos.to(dev), wl.text_inv_freq().to(dev), wl.MROPE_SECTION)
    q, k, v = ops.qkv_projection_with_rope(x.to(dev), w.to(dev), b.to(dev), table, 16, 2)
    rows = torch.cat([torch.arange(0, B * S, 97), torch.tensor([B * S - 1])])  # spread over every row tile
    rq, rk, rv = _reference(x, w, b, pos, 16, 2, rows)
    pick = lambda t: t.transpose(1, 2).reshape(B * S, -1, 128)[rows.to(dev)].cpu()  # noqa: E731  [rows, heads, D]
    _close(pick(q), rq[0].transpose(0, 1), "q sample")
    _close(pick(k), rk[0].transpose(0, 1), "k sample")
    _close(pick(v), rv[0].transpose(0, 1), "v sample")


def test_qkv_rope_rejects_what_it_cannot_do(dev):
    lib = _lib.load()
    pos = torch.zeros(3, 1, 4, dtype=torch.int64, device=dev)
    p = pos.data_ptr()
    assert lib.wx_qkv_rope_proj(p, p, None, p, 32, p, 4, 64, 1, 1, 64, None) == -2
    assert b"head_dim" in lib.wx_last_error_string()


@pytest.mark.parametrize("layout", ["hf", "csrc"])
@pytest.mark.parametrize("B,S,H,nq,nkv,with_bias", [(2, 200, 512, 4, 2, True), (1, 37, 256, 2, 1, False)])
def test_qkv_rope_projection_backward(dev, B, S, H, nq, nkv, with_bias, layout):
    """Gradients of the fused projection against torch autograd of the fp32 expression it fuses (linear, then the
    oracle's M-RoPE in fp32 on the same cos / sin): d hidden, d weight, d bias for a random cotangent on q, k and v.
    The fused op rounds the forward and the rotated gradient to bf16 like the eager bf16 path, so the comparison
    carries the GEMM tolerance, scaled to each gradient's magnitude."""
    g = torch.Generator().manual_seed(B * 77 + S)
    D = 128
    n = (nq + 2 * nkv) * D
    x = torch.randn(B, S, H, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, H, generator=g) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, generator=g) * 0.5).to(torch.bfloat16) if with_bias else None
    pos = torch.stack([torch.randint(0, 60, (B, S), generator=g), torch.randint(100, 160, (B, S), generator=g),
                       torch.randint(300, 360, (B, S), generator=g)])
    cq = torch.randn(B, nq, S, D, generator=g).to(torch.bfloat16)
    ck = torch.randn(B, nkv, S, D, generator=g).to(torch.bfloat16)
    cv = torch.randn(B, nkv, S, D, generator=g).to(torch.bfloat16)
    # reference: fp32 autograd through linear and the oracle's rotation
    xr, wr = x.float().requires_grad_(True), w.float().requires_grad_(True)
    br = None if b is None else b.float().requires_grad_(True)
    cos, sin = oracle.rotary_cos_sin_ref(pos, wl.text_inv_freq(), torch.bfloat16)
    qkv = F.linear(xr, wr, br)
    q, k, v = qkv.split([nq * D, nkv * D, nkv * D], dim=-1)
    q = q.reshape(B, S, nq, D).transpose(1, 2)
    k = k.reshape(B, S, nkv, D).transpose(1, 2)
    v = v.reshape(B, S, nkv, D).transpose(1, 2)
    rq, rk = oracle.mrope_apply_ref(q, k, cos.float(), sin.float(), list(wl.MROPE_SECTION), layout)
    ((rq * cq.float()).sum() + (rk * ck.float()).sum() + (v * cv.float()).sum()).backward()
    # fused op
    xd, wd = x.to(dev).requires_grad_(True), w.to(dev).requires_grad_(True)
    bd = None if b is None else b.to(dev).requires_grad_(True)
    table = ops.multimodal_rope_table(pos.to(dev), wl.text_inv_freq().to(dev), wl.MROPE_SECTION, layout)
    gq, gk, gv = ops.qkv_projection_with_rope(xd, wd, bd, table, nq, nkv, mrope_section=wl.MROPE_SECTION)
    torch.autograd.backward([gq, gk, gv], [cq.to(dev), ck.to(dev), cv.to(dev)])

    def close(got, ref, what):
        got, ref = got.float().cpu(), ref.float()
        s = float(ref.pow(2).mean().sqrt())
        bad = (got - ref).abs() > 2e-2 * s + 1e-2 * ref.abs()
        assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()} outside tolerance (rms {s})"

    close(xd.grad, xr.grad, "d hidden_states")
    close(wd.grad, wr.grad, "d qkv_weight")
    if b is not None:
        close(bd.grad, br.grad, "d qkv_bias")
    # the forward under autograd is the same launch as without it
    with torch.no_grad():
        q0, k0, v0 = ops.qkv_projection_with_rope(x.to(dev), w.to(dev), None if b is None else b.to(dev), table, nq, nkv)
    assert torch.equal(q0, gq) and torch.equal(k0, gk) and torch.equal(v0, gv)


@pytest.mark.parametrize("layout", ["hf", "csrc"])
@pytest.mark.parametrize("rows", [1, 127, 129, 3072, 3073])  # 3072 rows are the last of the 128 x 128 tiles at this width
def test_qkv_rope_projection_of_few_rows_is_a_slice_of_many(dev, rows, layout):
    """The tile shape follows the row count and a row's result does not: every accumulator sums its K steps in order."""
    T, H, nq, nkv = 3400, 256, 16, 2
    g = torch.Generator().manual_seed(5)
    n = (nq + 2 * nkv) * 128
    x = torch.randn(1, T, H, generator=g).to(torch.bfloat16).to(dev)
    w = (torch.randn(n, H, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    b = (torch.randn(n, generator=g) * 0.5).to(torch.bfloat16).to(dev)
    pos = torch.randint(0, 300, (3, 1, T), generator=g)

    def run(m):
        table = ops.multimodal_rope_table(pos[:, :, :m].contiguous().to(dev), wl.text_inv_freq().to(dev), wl.MROPE_SECTION, layout)
        return ops.qkv_projection_with_rope(x[:, :m].contiguous(), w, b, table, nq, nkv)

    for got, want in zip(run(rows), run(T)):
        assert torch.equal(got, want[:, :, :rows])
    pick = torch.tensor(sorted({0, rows // 2, rows - 1}))
    for got, ref in zip(run(rows), _reference(x.cpu(), w.cpu(), b.cpu(), pos, nq, nkv, rows=pick, layout=layout)):
        _close(got[:, :, pick.to(dev)], ref, f"{rows} rows")


@pytest.mark.parametrize("layout", ["hf", "csrc"])
@pytest.mark.parametrize("rows", [200, 3400])  # the 128 x 128 tiles alone, and the 256 x 256 tiles
def test_qkv_rope_projection_with_table_and_bias_at_any_element(dev, rows, layout):
    """The packed table at any word and the bias at any bf16 value: what the aligned buffers give, bit for bit."""
    H, nq, nkv = 64, 16, 2
    g = torch.Generator().manual_seed(11)
    n = (nq + 2 * nkv) * 128
    x = torch.randn(1, rows, H, generator=g).to(torch.bfloat16).to(dev)
    w = (torch.randn(n, H, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    b = (torch.randn(n, generator=g) * 0.5).to(torch.bfloat16).to(dev)
    pos = torch.randint(0, 300, (3, 1, rows), generator=g)
    table = ops.multimodal_rope_table(pos.to(dev), wl.text_inv_freq().to(dev), wl.MROPE_SECTION, layout)
    want = ops.qkv_projection_with_rope(x, w, b, table, nq, nkv)
    for off in (1, 2, 3):
        t2 = table.new_empty(table.numel() + 4)[off:off + table.numel()].view_as(table).copy_(table)
        b2 = b.new_empty(n + 8)[off:off + n].copy_(b)
        assert t2.data_ptr() % 16 == 4 * off and b2.data_ptr() % 8 == 2 * off
        for got, ref in zip(ops.qkv_projection_with_rope(x, w, b2, t2, nq, nkv), want):
            assert torch.equal(got, ref)


@pytest.mark.parametrize("layout", ["hf", "csrc"])
@pytest.mark.parametrize("B,S,nq,nkv,order", [(1, 1, 1, 1, "bshd"), (1, 15, 4, 2, "bhsd"), (3, 17, 5, 1, "split"), (2, 2050, 16, 2, "bshd"),
                                              (1, 4113, 3, 3, "mixed"), (2, 33, 2, 1, "none"), (2, 40, 4, 1, "expanded")])
def test_gradient_of_the_projection_before_the_rotation(dev, B, S, nq, nkv, order, layout):
    """wx_qkv_rope_bwd: the q and k heads as rope_from_table's adjoint gives them, the v heads as they are, bit for bit, and the
    column sums against 64 bits: fp32 sums of T values (T 2^-24 of the sum of sizes bounds any order) and one rounding."""
    g = torch.Generator(device=dev).manual_seed(S)
    D, section = 128, list(wl.MROPE_SECTION)
    pos = torch.randint(0, 500, (3, B, S), device=dev, generator=g)
    table = native.mrope_table(pos, wl.text_inv_freq().to(dev), section, layout)

    def grad(n, how):
        if how == "bshd":
            return torch.randn((B, S, n, D), device=dev, generator=g).to(torch.bfloat16).transpose(1, 2)
        if how == "split":  # heads of a wider matrix, at an offset that is not a multiple of 16 bytes
            return torch.randn((B, S, n * D + 12), device=dev, generator=g).to(torch.bfloat16)[..., 4:4 + n * D].view(B, S, n, D).transpose(1, 2)
        if how == "expanded":
            return torch.randn((1, n, 1, 1), device=dev, generator=g).to(torch.bfloat16).expand(B, n, S, D)
        return torch.randn((B, n, S, D), device=dev, generator=g).to(torch.bfloat16)

    hows = {"mixed": ("bhsd", "bshd", "float"), "none": ("bshd", None, "bhsd")}.get(order, (order,) * 3)
    grads = [None if h is None else (grad(n, "bhsd").float() if h == "float" else grad(n, h)) for h, n in zip(hows, (nq, nkv, nkv))]
    out, bias = native.qkv_rope_bwd(*grads, table, B, S, nq, nkv, True)
    full = [torch.zeros((B, n, S, D), dtype=torch.bfloat16, device=dev) if t is None else t.to(torch.bfloat16).contiguous() for t, n in zip(grads, (nq, nkv, nkv))]
    rq, rk = torch.empty_like(full[0]), torch.empty_like(full[1])
    native.rope_from_table(full[0], full[1], table, rq, rk, [2 * v for v in section], backward=True, layout=layout)
    want = torch.cat((rq, rk, full[2]), 1).transpose(1, 2).reshape(B * S, -1)
    assert torch.equal(out, want)
    exact, size = want.double().sum(0), want.double().abs().sum(0)
    assert bool(((bias.double() - exact).abs() <= 2 ** -8 * exact.abs() + B * S * 2 ** -24 * size + 1e-30).all())
    again, none = native.qkv_rope_bwd(*grads, table, B, S, nq, nkv, False)
    assert none is None and torch.equal(again, out)


def test_projection_backward_with_one_output_used_or_changed_in_place(dev):
    g = torch.Generator(device=dev).manual_seed(5)
    h = torch.randn((2, 24, 64), device=dev, generator=g).to(torch.bfloat16).requires_grad_()
    w = (torch.randn((4 * 128, 64), device=dev, generator=g) * 0.1).to(torch.bfloat16).requires_grad_()
    pos = torch.randint(0, 90, (3, 2, 24), device=dev, generator=g)
    table = ops.multimodal_rope_table(pos, wl.text_inv_freq().to(dev), wl.MROPE_SECTION)
    seed = torch.randn((2, 1, 24, 128), device=dev, generator=g).to(torch.bfloat16)
    q, k, v = ops.qkv_projection_with_rope(h, w, None, table, 2, 1)
    assert q.transpose(1, 2).stride() == (24 * 512, 512, 128, 1) and v.data_ptr() == q.data_ptr() + 3 * 256
    dw = torch.autograd.grad(v, w, seed, retain_graph=True)[0]
    assert not dw[:384].any() and dw[384:].any()
    k.mul_(2)
    (dk,) = torch.autograd.grad(k, w, seed)
    q1, k1, v1 = ops.qkv_projection_with_rope(h, w, None, table, 2, 1)
    (once,) = torch.autograd.grad(k1, w, seed)
    assert torch.equal(dk, 2 * once)
    with pytest.raises(RuntimeError, match="table must be"):
        bad = ops.qkv_projection_with_rope(h, w, None, table, 2, 1, layout="csrc")
        torch.autograd.grad(bad[0].sum(), w)

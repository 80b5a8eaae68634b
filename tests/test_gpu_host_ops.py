"""The native host side of the row and rotary ops (csrc/host_ops.cpp) against the general path in native.py: what it takes
gives the same bits, and whatever has to be warned of, copied or refused it leaves alone."""
import threading
import warnings

import pytest
import torch

from wallx_mi355 import _lib, native, workloads as wl
from wallx_mi355.fusions import ops

SECTION = list(wl.MROPE_SECTION)


def _rope_inputs(dev, form, dtype, layout, order, rows=2, row_len=5):
    g = torch.Generator(device=dev).manual_seed(3)
    D = 128
    make = {"bshd": lambda n: torch.randn((rows, row_len, n, D), generator=g, device=dev).to(dtype).transpose(1, 2),
            "bhsd": lambda n: torch.randn((rows, n, row_len, D), generator=g, device=dev).to(dtype),
            "packed": lambda n: torch.randn((rows, row_len, n + 3, D), generator=g, device=dev).to(dtype)[:, :, 2:2 + n].transpose(1, 2),
            "expanded": lambda n: torch.randn((1, n, 1, D), generator=g, device=dev).to(dtype).expand(rows, n, row_len, D)}[order]
    q, k = make(4), make(2)
    pos = torch.randint(0, 300, (3, rows, row_len), generator=g, device=dev)
    freq = wl.text_inv_freq(D).to(dev)
    if form == 1:
        return q, k, pos, freq
    if form == 2:
        return q, k, native.mrope_table(pos, freq, SECTION, layout), None
    angle = pos.float()[..., None] * torch.cat((freq, freq))
    return q, k, angle.cos().to(dtype), angle.sin().to(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("order", ["bshd", "bhsd", "packed", "expanded"])
@pytest.mark.parametrize("form,dtype", [(0, torch.bfloat16), (0, torch.float16), (0, torch.float32), (1, torch.bfloat16), (1, torch.float32),
                                        (2, torch.bfloat16)])
@pytest.mark.parametrize("layout", ["hf", "csrc"])
def test_rope_as_the_general_path(dev, form, dtype, layout, order):
    q, k, a, b = _rope_inputs(dev, form, dtype, layout, order)
    doubled = [2 * v for v in SECTION]
    for backward in (0, 1):
        made = _lib.host().rope(form, q, k, a, b, SECTION, layout, backward)
        want = torch.empty(q.shape, dtype=dtype, device=dev), torch.empty(k.shape, dtype=dtype, device=dev)
        if form == 0:
            (native.rope_bwd(q, k, None, None, a, b, *want, doubled, layout) if backward else native.rope(q, k, a, b, *want, doubled, layout))
        elif form == 1:
            native.rope_from_positions(q, k, a, b, *want, doubled, backward=bool(backward), layout=layout)
        else:
            native.rope_from_table(q, k, a, *want, doubled, backward=bool(backward), layout=layout)
        for x, w in zip(made, want):
            assert x.is_contiguous() and x.shape == w.shape and torch.equal(x, w)


@pytest.mark.gpu
def test_rope_leaves_alone_what_the_general_path_is_for(dev):
    q, k, c, s = _rope_inputs(dev, 0, torch.bfloat16, "hf", "bshd")
    rope = _lib.host().rope

    class Sub(torch.Tensor):
        pass

    assert rope(0, q, k, c, s, SECTION, "hf", 0) is not None
    for args in ((q.cpu(), k, c, s), (q, k.float(), c, s), (q, k, c.transpose(1, 2), s), (q, k[:1], c, s), (q[..., ::2], k, c, s),
                 (q, k, c[:2], s), (q.as_subclass(Sub), k, c, s), (q, k, c, None), (q.double(), k.double(), c.double(), s.double())):
        assert rope(0, *args, SECTION, "hf", 0) is None
    for section, layout in (([16, 24], "hf"), ([16.0, 24, 24], "hf"), ("abc", "hf"), (SECTION, "other"), (SECTION, 0)):
        assert rope(0, q, k, c, s, section, layout, 0) is None
    with pytest.raises(RuntimeError, match="covers 120 channels"):
        ops.multimodal_rope(q, k, c, s, [16, 24, 20])
    with pytest.raises(RuntimeError, match="list of 3 integers"):
        ops.multimodal_rope(q, k, c, s, [16, 24])
    with pytest.warns(UserWarning, match="`cos` of multimodal_rope op is discontiguous"):
        got = ops.multimodal_rope(q, k, c.transpose(1, 2).contiguous().transpose(1, 2), s, SECTION)
    assert all(torch.equal(x, y) for x, y in zip(got, ops.multimodal_rope(q, k, c, s, SECTION)))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,topk,num_out", [(1, 1, 0), (257, 1, 0), (257, 1, 100), (300, 3, 0), (4099, 2, 5000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_permute_and_unpermute_as_the_general_path(dev, tokens, topk, num_out, dtype, monkeypatch):
    g = torch.Generator(device=dev).manual_seed(tokens)
    x = torch.randn((tokens, 72), generator=g, device=dev).to(dtype)
    ids = torch.randint(0, 5, (tokens, topk), generator=g, device=dev, dtype=torch.int32)
    host = _lib.host()
    rmap, _, _, ws = native.partition(ids, native.MAX_EXPERTS, num_out)
    want = native.permute_rows(x, rmap, topk, num_out or tokens * topk)
    out, got = host.permute(x, ids, num_out, *ws, native.MAX_EXPERTS)
    used = int((rmap >= 0).sum())
    assert torch.equal(got, rmap) and torch.equal(out[:used], want[:used])
    assert host.permute(x, ids, num_out, ws[0][:1], ws[1], native.MAX_EXPERTS) is None  # too little scratch
    assert host.permute(x, ids.long(), num_out, *ws, native.MAX_EXPERTS) is None
    assert host.permute(x.t(), ids, num_out, *ws, native.MAX_EXPERTS) is None
    if not num_out:
        probs = torch.rand((tokens, topk), generator=g, device=dev)
        for p in (None, probs):
            assert torch.equal(host.unpermute(out, rmap, p, tokens, topk), native.unpermute(out, rmap, torch.tensor([]) if p is None else p, tokens, topk))
        assert host.unpermute(out, rmap[:-1], None, tokens, topk) is None  # a short map
        assert host.unpermute(out, rmap.long(), None, tokens, topk) is None
    if topk == 1:
        grad = torch.randn((tokens, 72), generator=g, device=dev).to(dtype)
        assert torch.equal(host.unpermute_bwd(grad, out, rmap, None), native.unpermute_rows_bwd(grad, out, rmap))
        assert host.unpermute_bwd(grad, out[:, :40], rmap, None) is None
        assert host.unpermute_bwd(grad, out, rmap, torch.ones((tokens, 1), device=dev)) is None  # a weight whose gradient is zeros
    else:
        grad = torch.randn((tokens, 72), generator=g, device=dev).to(dtype)
        probs = torch.rand((tokens, topk), generator=g, device=dev)
        got = host.unpermute_bwd(grad, out, rmap, probs)
        for a, b in zip(got, native.unpermute_bwd(grad, out, rmap, probs)):
            assert a.dtype == b.dtype and torch.equal(a, b)
        assert host.unpermute_bwd(grad, out, rmap, probs.double()) is None and host.unpermute_bwd(grad, out, rmap[:-1], probs) is None
        assert host.unpermute_bwd(grad, out, rmap, probs[:-1]) is None


@pytest.mark.gpu
def test_permute_in_checked_mode_still_refuses_wild_ids(dev):
    x = torch.randn((8, 64), device=dev)
    ids = torch.full((8, 1), native.MAX_EXPERTS, dtype=torch.int32, device=dev)
    _, _, ws = native.permute(x, ids, 0, [], 0)
    native.set_checked(True)
    try:
        with pytest.raises(RuntimeError, match="outside"):
            native.permute(x, ids, 0, ws, 0)
    finally:
        native.set_checked(False)


def test_tensors_on_the_cpu_are_left_alone():
    q, k, c = torch.zeros(1, 4, 2, 128), torch.zeros(1, 2, 2, 128), torch.zeros(3, 1, 2, 128)
    x, ids = torch.zeros(4, 8), torch.zeros(4, 1, dtype=torch.int32)
    host = _lib.host()
    assert host.rope(0, q, k, c, c, SECTION, "hf", 0) is None
    assert host.permute(x, ids, 0, x, ids, 256) is None
    assert host.unpermute(x, ids.view(-1), None, 4, 1) is None and host.unpermute_bwd(x, x, ids.view(-1), None) is None
    with pytest.raises(TypeError):
        host.bind(1)


@pytest.mark.gpu
def test_recorded_into_a_graph_on_another_stream(dev):
    """The native host side under capture: every replay on new contents equals the eager calls."""
    q, k, c, s = _rope_inputs(dev, 0, torch.bfloat16, "hf", "bshd", rows=3, row_len=70)
    g = torch.Generator(device=dev).manual_seed(9)
    x = torch.randn((5000, 64), generator=g, device=dev).to(torch.bfloat16)
    ids = torch.randint(0, 3, (5000, 1), generator=g, device=dev, dtype=torch.int32)

    def work():
        rq, rk = ops.multimodal_rope(q, k, c, s, SECTION)
        permuted, rmap = ops.permute(x, ids)
        return rq, rk, permuted, ops.unpermute(permuted, rmap)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        work()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = work()
    for _ in range(3):
        for t in (q, k, x):
            t.copy_(torch.randn(t.shape, generator=g, device=dev).to(t.dtype))
        ids.copy_(torch.randint(0, 3, ids.shape, generator=g, device=dev, dtype=torch.int32))
        graph.replay()
        got = [t.clone() for t in out]
        torch.cuda.synchronize()
        for a, b in zip(got, work()):
            assert torch.equal(a, b)


@pytest.mark.gpu
def test_from_several_threads_with_streams_of_their_own(dev):
    """Forward and backward from four threads at once, each on a stream of its own, equal the calls one after the other."""
    import threading

    inputs = [_rope_inputs(dev, 0, torch.bfloat16, "hf", "bshd", rows=1 + i, row_len=33 + i) for i in range(4)]

    def one(i):
        q, k, c, s = inputs[i]
        q, k = q.detach().requires_grad_(), k.detach().requires_grad_()
        out = ops.multimodal_rope(q, k, c, s, SECTION)
        return [t.detach() for t in out] + list(torch.autograd.grad(out, (q, k), [t.detach() for t in out]))

    want = [one(i) for i in range(4)]
    got, errors = [None] * 4, []
    torch.cuda.synchronize()

    def thread(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(5):
                    got[i] = one(i)
            stream.synchronize()
        except Exception as exc:  # noqa: BLE001 - reported below
            errors.append(exc)

    threads = [threading.Thread(target=thread, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for a, b in zip(got, want):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.gpu
@pytest.mark.parametrize("ids_dtype", [torch.int32, torch.int64])
def test_recorded_permute_is_its_own_beside_calls_of_other_sizes_and_types(dev, ids_dtype):
    """More than 4096 keys: one launch writes histograms that the next reads.  A graph replayed after calls that need
    larger scratch gives its own result, and writes nothing into memory allocated since."""
    g = torch.Generator(device=dev).manual_seed(2)
    x = torch.randn((5000, 64), generator=g, device=dev).to(torch.bfloat16)
    ids = torch.randint(0, 3, (5000, 1), generator=g, device=dev, dtype=ids_dtype)
    big, big_ids = torch.randn((40000, 64), generator=g, device=dev), torch.randint(0, 3, (40000, 1), generator=g, device=dev, dtype=ids_dtype)

    def call(x, ids):
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            return ops.permute(x, ids)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(x, ids)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, rmap = call(x, ids)
    for _ in range(3):
        call(big, big_ids)
        since = [torch.full((n,), 7, dtype=torch.uint8, device=dev) for n in (1, 512, 1024, 10240, 20480, 40960, 1 << 20) for _ in range(8)]
        ids.copy_(torch.randint(0, 3, ids.shape, generator=g, device=dev, dtype=ids_dtype))
        graph.replay()
        torch.cuda.synchronize()
        want, want_map = call(x, ids)
        assert torch.equal(rmap, want_map) and torch.equal(out, want)
        assert all(bool((t == 7).all()) for t in since)


@pytest.mark.gpu
def test_permute_from_several_threads_with_streams_of_their_own(dev):
    """Forward and backward of more than 4096 keys from four threads at once equal the calls one after the other."""
    g = torch.Generator(device=dev).manual_seed(11)
    cases = []
    for i in range(4):
        dtype = (torch.bfloat16, torch.float32)[i & 1]
        cases.append((torch.randn((4500 + 1000 * i, 64), generator=g, device=dev).to(dtype),
                      torch.randint(0, 2 + i, (4500 + 1000 * i, 1 + i % 2), generator=g, device=dev, dtype=torch.int32)))

    def one(i):
        x, ids = cases[i][0].detach().requires_grad_(), cases[i][1]
        out, rmap = ops.permute(x, ids)
        return [out.detach(), rmap, *torch.autograd.grad(out, x, out.detach())]

    want = [one(i) for i in range(4)]
    got, errors = [[] for _ in range(4)], []
    torch.cuda.synchronize()

    def thread(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(10):
                    got[i].append(one(i))
            stream.synchronize()
        except Exception as exc:  # noqa: BLE001 - reported below
            errors.append(exc)

    threads = [threading.Thread(target=thread, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for made, expect in zip(got, want):
        assert len(made) == 10
        for result in made:
            assert all(torch.equal(a, b) for a, b in zip(result, expect))


@pytest.mark.gpu
def test_permute_keeps_the_status_word_of_a_workspace_and_nothing_else_of_it(dev):
    x = torch.randn((5000, 64), device=dev)
    ids = torch.zeros((5000, 1), dtype=torch.int32, device=dev)
    _, _, ws = native.permute(x, ids, 0, [], 0)
    before = ws[0].fill_(3).clone()
    out, rmap, again = native.permute(x, ids, 0, ws, 0)
    assert again is ws and torch.equal(ws[0], before) and not int(ws[1]) and torch.equal(out, x)
    native.permute(x, ids.fill_(native.MAX_EXPERTS), 0, ws, 0)
    assert int(ws[1]) == 1 and torch.equal(ws[0], before)
    native.permute(x, ids.long(), 0, ws, 0)  # the general path
    assert torch.equal(ws[0], before)
    assert native.permute(x, ids.zero_(), 0, None, 0)[2] is None


@pytest.mark.gpu
def test_wrappers_of_the_transforms_are_left_alone(dev):
    """vmap's, grad's and functionalization's tensors are exact torch.Tensors that are none inside; a fake one is a subclass."""
    q, k, c, s = _rope_inputs(dev, 0, torch.bfloat16, "hf", "bshd")
    x, ids = torch.randn((6, 64), device=dev), torch.zeros((6, 1), dtype=torch.int32, device=dev)
    rmap = torch.arange(6, dtype=torch.int32, device=dev)
    host, seen = _lib.host(), []

    def calls(q, x):
        seen.append([host.rope(0, q, k, c, s, SECTION, "hf", 0), host.permute(x, ids, 0, None, None, 256), host.unpermute(x, rmap, None, 6, 1),
                     host.unpermute_bwd(x, x, rmap, None)])
        return q

    calls(q, x)
    assert all(r is not None for r in seen.pop())
    torch.func.vmap(calls)(q[None], x[None])
    torch.func.grad(lambda q, x: calls(q, x).float().sum())(q.contiguous(), x)
    torch.func.functionalize(calls)(q, x)
    torch.func.jvp(lambda t: calls(q, t), (x,), (x,))
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        calls(mode.from_tensor(q), mode.from_tensor(x))
    half = torch.randn((6, 64, 2), device=dev)
    calls(torch.view_as_complex(torch.randn((*q.shape, 2), device=dev)).conj().imag, torch.view_as_complex(half).conj().imag)  # negation pending
    assert len(seen) == 6 and all(r is None for results in seen for r in results), seen


@pytest.mark.gpu
def test_backwards_and_the_other_forms_recorded_into_a_graph(dev):
    """Forward and backward of all three forms of the rotary op, and of permute and unpermute with and without weights."""
    q, k, c, s = _rope_inputs(dev, 0, torch.bfloat16, "hf", "bshd", rows=2, row_len=70)
    pos, freq = _rope_inputs(dev, 1, torch.bfloat16, "hf", "bshd", rows=2, row_len=70)[2:]
    table = native.mrope_table(pos, freq, SECTION)
    g = torch.Generator(device=dev).manual_seed(9)
    q, k = q.requires_grad_(), k.requires_grad_()
    x = torch.randn((5000, 64), generator=g, device=dev).to(torch.bfloat16).requires_grad_()
    probs = torch.rand((5000, 2), generator=g, device=dev).requires_grad_()
    ids = torch.rand((5000, 4), generator=g, device=dev).argsort(1)[:, :2].to(torch.int32).contiguous()
    dq, dk, dx = (torch.randn(t.shape, generator=g, device=dev).to(t.dtype) for t in (q, k, x))

    def work():
        out = []
        for rotated in (ops.multimodal_rope(q, k, c, s, SECTION), ops.multimodal_rope_from_positions(q, k, pos, freq, SECTION),
                        ops.multimodal_rope_from_table(q, k, table, SECTION)):
            out += [t.detach() for t in rotated] + list(torch.autograd.grad(rotated, (q, k), (dq, dk)))
        permuted, rmap = ops.permute(x, ids)
        out += [permuted.detach(), rmap, *torch.autograd.grad(ops.unpermute(permuted, rmap, probs), (x, probs), dx)]
        one, one_map = ops.permute(x, ids[:, :1].contiguous())
        return out + [one.detach(), *torch.autograd.grad(ops.unpermute(one, one_map), x, dx)]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        work()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = work()
    for _ in range(3):
        with torch.no_grad():
            for t in (q, k, x, probs, dq, dk, dx):
                t.copy_(torch.randn(t.shape, generator=g, device=dev).to(t.dtype))
            ids.copy_(torch.rand((5000, 4), generator=g, device=dev).argsort(1)[:, :2])
        graph.replay()
        got = [t.clone() for t in out]
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, work()))

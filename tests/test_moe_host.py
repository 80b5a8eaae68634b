"""Host-side logic of the drop-in MoE block that needs no GPU: tensors made under torch.inference_mode() have no
version counter (reading `_version` raises), so nothing derived from them may be cached against one; an expert list
other than wall-x's own (two silu experts) selects the generic path instead of raising."""

from types import SimpleNamespace

import pytest
import torch

from wallx_mi355 import moe


def _cfg(inters=(96, 32), acts=("silu", "silu"), hidden=64):
    return SimpleNamespace(experts=[dict(hidden_size=hidden, intermediate_size=i, hidden_act=a)
                                    for i, a in zip(inters, acts)])


def test_version_of_inference_tensors_is_none():
    normal = torch.zeros(3)
    assert moe._version_of(normal) == normal._version
    with torch.inference_mode():
        made_inside = torch.zeros(3)
        assert moe._version_of(made_inside) is None
        with pytest.raises(RuntimeError):
            made_inside._version  # what the guard exists for
        assert moe._version_of(normal) == normal._version  # a normal tensor keeps its counter in inference mode


def test_host_row_counts_from_inference_mode_tensors_are_read_on_every_call():
    block = moe.SparseMoeBlock(_cfg(), 2)
    with torch.inference_mode():
        start, end = torch.tensor([0, 5]), torch.tensor([5, 12])
        rows = block._host_rows(start, end, 12)
        assert list(rows) == [5, 7] and block._rows_seen is None  # nothing to check a later call against
        end[1] = 11  # an in-place write no counter records
        assert block._host_rows(start, end, 11) is not None and list(block._host_rows(start, end, 11)) == [5, 6]
    start, end = torch.tensor([0, 5]), torch.tensor([5, 12])
    first = block._host_rows(start, end, 12)
    assert block._host_rows(start, end, 12) is first  # tracked tensors: answered from the cache
    end[1] = 11
    assert list(block._host_rows(start, end, 11)) == [5, 6]  # the version counter moved
    assert block._host_rows(start, end, 12) is None  # counts that do not add up to the token count are not used


def test_expert_lists_other_than_two_silu_experts_select_the_generic_path():
    assert moe.SparseMoeBlock(_cfg(), 2)._fused
    three = moe.SparseMoeBlock(_cfg((96, 32, 48), ("silu",) * 3), 3)
    assert not three._fused and len(three.experts) == 3
    gelu = moe.SparseMoeBlock(_cfg(acts=("gelu", "silu")), 2)
    assert not gelu._fused
    x = torch.linspace(-3, 3, 13)
    assert torch.allclose(gelu.experts[0].act_fn(x), torch.nn.functional.gelu(x))
    assert torch.allclose(gelu.experts[1].act_fn(x), torch.nn.functional.silu(x))
    with pytest.raises(KeyError):
        moe.SparseMoeBlock(_cfg(acts=("no_such_activation", "silu")), 2)
    with pytest.raises(RuntimeError, match="generic ops"):
        gelu.pack_for_inference()
    # the reference's parameter names (act.py:74-76, 101-103), whatever the path
    assert sorted(three.state_dict()) == sorted(f"experts.{e}.{p}_proj.weight" for e in range(3)
                                                for p in ("gate", "up", "down"))


@pytest.mark.parametrize("rows,inter,launches", [
    # (rows of the launch's two problems, whether it accumulates), in order; 256 columns: 2 * ceil(rows / 256) <= 8 CUs is few
    ((100, 20), (64, 16), [(100, 100, False), (20, 20, False)]),
    ((1024, 1024), (64, 16), [(1024, 1024, False), (1024, 1024, False)]),
    ((1025, 20), (64, 16), [(1025, 20, False), (1025, 20, True)]),  # many rows on the wide expert
    ((100, 1025), (64, 16), [(100, 100, False), (0, 1025, False), (0, 1025, True)]),  # ... and on the narrow one
    ((1025, 100), (16, 64), [(1025, 0, False), (1025, 0, True), (100, 100, False)]),
    ((0, 1024), (64, 16), [(1024, 1024, False)]),
    ((0, 1025), (64, 16), [(0, 1025, False), (0, 1025, True)]),  # no row on the wide expert
    ((1025, 0), (16, 64), [(1025, 0, False), (1025, 0, True)]),
    ((0, 0), (64, 16), [(0, 0, False), (0, 0, True)]),
    ((100, 20), (32, 32), [(100, 20, False), (100, 20, True)]),  # neither is the wide one
    ((100, 20), (31, 16), [(100, 20, False), (100, 20, True)]),
    ((20, 0), (32, 32), [(20, 20, False)]),
])
def test_input_grads_share_launches_by_each_experts_own_tiles(monkeypatch, rows, inter, launches):
    """Which launches dX = dG Wg + dU Wu takes, and that no split of the rows leaves a product, a row or the sum out."""
    made = []

    def dual(in0, in1, w0, w1, out0, out1, trans_a, trans_b, add_expert0=None, add_expert1=None):
        made.append((in0.size(0), in1.size(0), add_expert0 is not None or add_expert1 is not None))
        for a, w, out, add in ((in0, w0, out0, add_expert0), (in1, w1, out1, add_expert1)):
            y = (a.float() @ w.float()).to(torch.bfloat16)
            out.copy_(y if add is None else y + add)

    monkeypatch.setattr(moe.native, "asym_dual_gmm", dual)
    monkeypatch.setattr(moe, "_cus", lambda device: 8)
    g = torch.Generator().manual_seed(sum(rows))
    n = lambda *s: torch.randn(s, generator=g).to(torch.bfloat16)
    dg, du = ([n(m, i) for m, i in zip(rows, inter)] for _ in range(2))
    wg, wu = ([n(i, 256) for i in inter] for _ in range(2))
    got = moe._input_grads(dg, du, wg, wu, 256)
    assert made == launches
    want = torch.cat([(a.float() @ b.float()).to(torch.bfloat16) + (c.float() @ d.float()).to(torch.bfloat16)
                      for a, b, c, d in zip(dg, wg, du, wu)])
    assert torch.equal(got, want)

"""The native host module (csrc/host_ops.cpp) belongs to one torch and one Python: of others it is built anew and never
loaded, and without it the ops go their general path."""
import importlib.util
import os
import sysconfig

import pytest
import torch

from wallx_mi355 import _lib, native, workloads as wl
from wallx_mi355.fusions import ops

_spec = importlib.util.spec_from_file_location("csrc_build", os.path.join(os.path.dirname(__file__), "..", "wall-x_amd", "csrc", "build.py"))
csrc_build = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(csrc_build)


def test_its_file_names_the_torch_and_the_python_it_is_for():
    assert os.path.realpath(csrc_build.host_lib()) == os.path.realpath(_lib.host_path())
    name = os.path.basename(_lib.host_path())
    assert torch.__version__ in name and name.endswith(sysconfig.get_config_var("EXT_SUFFIX"))


def test_another_torch_builds_it_again(monkeypatch, tmp_path):
    built = []

    def run(cmd):
        built.append(cmd[-1])
        open(cmd[-1], "w").close()

    monkeypatch.setattr(csrc_build, "OUT_DIR", str(tmp_path))
    monkeypatch.setattr(csrc_build, "_run", run)
    first = csrc_build.build_host(verbose=False)
    assert csrc_build.build_host(verbose=False) == first and built == [first]
    monkeypatch.setattr(torch, "__version__", "0.0.1+other")
    second = csrc_build.build_host(verbose=False)
    assert second != first and built == [first, second]
    os.utime(second, (1, 1))  # older than its source, its header or the script with its flags
    csrc_build.build_host(verbose=False)
    assert built == [first, second, second]


def _without(monkeypatch):
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(torch, "__version__", "0.0.1+other")
    with pytest.warns(UserWarning, match="is missing"):
        return _lib.host()


def test_one_of_another_torch_is_not_loaded(monkeypatch):
    host = _without(monkeypatch)
    assert _lib.host() is host
    assert host.rope(0, None, None, None, None, [], "hf", 0) is None and host.permute() is None
    assert host.unpermute() is None and host.unpermute_bwd() is None


@pytest.mark.gpu
def test_the_ops_without_it(dev, monkeypatch):
    g = torch.Generator(device=dev).manual_seed(4)
    q, k = (torch.randn((2, 33, n, 128), generator=g, device=dev).to(torch.bfloat16).transpose(1, 2).requires_grad_() for n in (4, 2))
    pos = torch.randint(0, 300, (3, 2, 33), generator=g, device=dev)
    freq = wl.text_inv_freq(128).to(dev)
    table = native.mrope_table(pos, freq, wl.MROPE_SECTION)
    angle = pos.float()[..., None] * torch.cat((freq, freq))
    c, s = angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16)
    x = torch.randn((5000, 64), generator=g, device=dev).requires_grad_()
    ids = torch.rand((5000, 6), generator=g, device=dev).argsort(1)[:, :2].to(torch.int32).contiguous()
    probs = torch.rand((5000, 2), generator=g, device=dev).requires_grad_()

    def work():
        out = [*ops.multimodal_rope(q, k, c, s, wl.MROPE_SECTION), *ops.multimodal_rope_from_positions(q, k, pos, freq, wl.MROPE_SECTION),
               *ops.multimodal_rope_from_table(q, k, table, wl.MROPE_SECTION)]
        grads = torch.autograd.grad(out, (q, k), [t.detach() for t in out])
        permuted, rmap = ops.permute(x, ids)
        y = ops.unpermute(permuted, rmap, probs)
        one, one_map = ops.permute(x, ids[:, :1].contiguous())
        z = ops.unpermute(one, one_map)
        return [*out, *grads, permuted, rmap, y, z, *torch.autograd.grad((y, z), (x, probs), (y.detach(), z.detach()))]

    with_it = work()
    assert _lib.host() is not _lib._NoHost
    _without(monkeypatch)
    assert all(torch.equal(a, b) for a, b in zip(work(), with_it))

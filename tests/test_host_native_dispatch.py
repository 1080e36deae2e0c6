"""The native dispatcher kernels (csrc/torch_binding.cpp) without a GPU: fake device tensors go through the autograd kernel and end
in the Meta implementation, so what is accepted and what is refused can be checked here."""

import os
import shutil
import subprocess
import sys

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

import ops_rec
from ops_rec import _build

built = pytest.mark.skipif(not os.path.exists(_build.BINDING_PATH), reason="the libraries have not been built")


def attend(delta, **grads):
    """``hstu_jagged`` on fake device tensors, those named in ``grads`` requiring a gradient."""
    with FakeTensorMode():
        make = lambda name, *shape: torch.empty(*shape, dtype=torch.bfloat16, device="cuda", requires_grad=grads.get(name, False))  # noqa: E731
        q, k, v, mask = make("q", 7, 2, 64), make("k", 7, 2, 64), make("v", 7, 2, 64), make("mask", 2, 2, 8, 8)
        offs = torch.empty(3, dtype=torch.int32, device="cuda")
        args = (8, 8, 1.0, offs, offs) if delta else (8, 1.0, offs)
        return ops_rec.ascendc.attention.hstu_jagged(q, k, v, mask, None, 3, *args)


@pytest.mark.parametrize("delta", [False, True], ids=["equal", "delta"])
def test_a_mask_that_requires_grad_is_refused_only_where_a_gradient_is_recorded(delta):
    with torch.no_grad():
        assert attend(delta, mask=True).shape == (7, 2, 64)
        assert attend(delta, mask=True, q=True).shape == (7, 2, 64)
    for grads in (dict(mask=True), dict(mask=True, q=True)):
        with pytest.raises(NotImplementedError, match="mask is a non-differentiable input"):
            attend(delta, **grads)
    assert attend(delta, q=True).requires_grad and not attend(delta).requires_grad


@built
@pytest.mark.parametrize("what", ["absent", "not a library", "not this module"])
def test_a_binding_that_does_not_load_leaves_the_python_kernels(what, tmp_path):
    package = os.path.dirname(ops_rec.__file__)
    shutil.copytree(package, tmp_path / "ops_rec", ignore=shutil.ignore_patterns("_lib", "__pycache__"))
    (tmp_path / "ops_rec" / "_lib").mkdir()
    path = tmp_path / "ops_rec" / "_lib" / "_torch_binding.so"
    if what == "not a library":
        path.write_bytes(b"built for something else")
    elif what == "not this module":
        shutil.copy(os.path.join(package, "_lib", "libhstu_mi355.so"), path)
    code = (
        "import ops_rec, torch\n"
        "from torch._subclasses.fake_tensor import FakeTensorMode\n"
        "assert ops_rec._dispatch.binding is None and ops_rec.__file__.startswith(%r)\n"
        "for op in ('hstu_jagged.equal', 'hstu_jagged_backward.delta', 'hstu_paged', 'ln_mul', 'in_linear_silu_backward'):\n"
        "    assert torch._C._dispatch_has_kernel_for_dispatch_key('ops_rec::' + op, 'CUDA'), op\n"
        "with FakeTensorMode():\n"
        "    q, offs = torch.empty(7, 2, 64, device='cuda', requires_grad=True), torch.empty(3, dtype=torch.int32, device='cuda')\n"
        "    out = ops_rec.ascendc.attention.hstu_jagged(q, q, q, None, None, 0, 8, 1.0, offs)\n"
        "    assert out.shape == q.shape and out.requires_grad\n" % str(tmp_path)
    )
    done = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, PYTHONPATH=str(tmp_path)), cwd=tmp_path, capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    assert ("does not load" in done.stderr) == (what != "absent")


@built
def test_the_native_kernels_are_the_ones_registered():
    assert ops_rec._dispatch.binding is not None and ops_rec._dispatch._lib is None
    for op in ("hstu_jagged.equal", "hstu_jagged_backward.delta", "hstu_paged", "ln_mul", "in_linear_silu_backward"):
        assert torch._C._dispatch_has_kernel_for_dispatch_key("ops_rec::" + op, "CUDA"), op


def test_building_loads_no_library_that_it_replaces():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = (
        "import sys, __graft_entry__ as g\n"
        "b = g._builder()\n"
        "assert b.BINDING_PATH.startswith(g._ROOT) and callable(b.build)\n"
        "assert 'ops_rec' not in sys.modules\n"
        "assert not [line for line in open('/proc/self/maps') if 'libhstu_mi355' in line]\n"
    )
    subprocess.run([sys.executable, "-c", code], cwd=root, check=True, timeout=120)


def test_a_packet_of_unknown_layout_is_left_as_it_is():
    from ops_rec import _ops

    packet = type("Packet", (), {})()
    _ops._pick_overload_by_argument(packet, 8)
    assert not vars(packet)
    assert torch.ops.ops_rec.hstu_jagged._op.__name__ == "call"  # (and this torch's layout is known)

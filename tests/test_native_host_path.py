"""The native host path around the library (hpfp8/_native.so): what the package does without it."""
import os
import subprocess
import sys

import pytest

import _util as U

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hyper-parallel_amd")


def test_package_is_imported_without_the_native_host_path():
    code = ("import sys, warnings; sys.modules['hpfp8._native'] = None\n"
            "with warnings.catch_warnings(record=True) as seen:\n"
            "    warnings.simplefilter('always'); import hpfp8\n"
            "assert hpfp8.ops._native is None and any('_native.so' in str(w.message) for w in seen), seen\n"
            "import torch; print(hpfp8.ops._gpu(torch.zeros(1)), hpfp8.Fp8Linear(128, 128).weight.shape[0])")
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, PYTHONPATH=PKG), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split() == ["False", "128"]


def test_a_module_built_for_another_torch_is_stale_and_not_used(monkeypatch):
    """Its classes might be laid out otherwise: the build makes it again (and not the library), the package goes without it."""
    import importlib.util
    from hpfp8 import _lib
    spec = importlib.util.spec_from_file_location("hpfp8_build", os.path.join(PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    monkeypatch.setattr(build, "_older", lambda out, deps: False)
    assert not build.native_stale() and not build.needs_build()
    monkeypatch.setattr(build, "_native_tag", lambda: "torch 2.1")
    assert build.native_stale() and build.needs_build() and not build.library_stale()
    ran = []
    monkeypatch.setattr(build, "_run", lambda cmd, verbose: ran.append(cmd[0]))
    build.build()
    assert ran == ["g++"]
    assert _lib.load_native() is not None
    monkeypatch.setattr(_lib, "native_tag", lambda: "torch 2.1")
    with pytest.warns(RuntimeWarning, match="built for torch"):
        assert _lib.load_native() is None


@pytest.mark.gpu
@pytest.mark.parametrize("recipe", ["blockwise", "blockwise_pow2", "per_tensor"])
def test_step_without_the_native_host_path_has_the_same_bits(gpu, recipe, monkeypatch):
    import torch
    import hpfp8
    from hpfp8 import ops
    x, w, b = (U.randn_bf16(s, i, d).to(gpu).requires_grad_(True) for i, (s, d) in enumerate((((130, 384), 1.0), ((256, 384), 0.05), ((256,), 1.0))))
    go = U.randn_bf16((130, 256), 3, 0.01).to(gpu)

    def step():
        y = hpfp8.fp8_linear(x, w, b, recipe=recipe)
        return [y.detach(), *torch.autograd.grad(y, (x, w, b), go)]

    want = step()
    monkeypatch.setattr(ops, "_native", None)
    for one, other in zip(step(), want):
        assert torch.equal(one, other)

"""The host extension (csrc/host.cpp) against the Python path it stands in for: every call gives the
same tensors, bit for bit, or the same refusal, whichever of the two serves it. The CPU part checks that
it takes no CPU tensors and that its table of entry points is the C ABI's."""
import re
import warnings
from pathlib import Path

import pytest
import torch

import synth
from conftest import pkg

ROOT = Path(__file__).resolve().parents[1]


def test_entry_point_table_matches_the_extension():
    src = (ROOT / "minisglang-rdna4_amd" / "csrc" / "host.cpp").read_text()
    members = re.findall(r"decltype\(&(\w+)\)", src[src.index("struct Abi"):src.index("Abi abi;")])
    assert tuple(members) == pkg("_host")._ENTRY_POINTS


def test_cpu_tensors_and_wrong_counts_are_left_alone():
    m = pkg("_host").load()
    x = torch.zeros(2, 128, dtype=torch.bfloat16)
    w = torch.zeros(2, 1, 1024, dtype=torch.uint8)
    s = torch.ones(1, 32, dtype=torch.float16)
    assert m.linear(x, w, s, None, 128, False, None, None, False, 0) is None
    assert m.rms_norm(x, None, 1e-6, False, None, True) is None
    assert m.moe(x, w, s, None, w, s, None, None, 2, True, False, 16, True, True, True, True) is None
    for f in (m.linear, m.rms_norm, m.moe, m.bind):
        with pytest.raises(TypeError):
            f(x)


@pytest.mark.parametrize("why", ["missing", "another torch", "not a library"])
def test_python_path_serves_without_the_extension(monkeypatch, tmp_path, why):
    """One warning, then a stand-in that takes no call (the GPU tests below run every form on it)."""
    host = pkg("_host")
    monkeypatch.setattr(host, "_mod", None)
    if why == "missing":
        monkeypatch.setattr(host, "_PATH", tmp_path / "w4a8_host.so")
    elif why == "another torch":
        monkeypatch.setattr(host, "_running", lambda: "torch 1.0, Python 3.10")
    else:
        (tmp_path / "w4a8_host.so").write_bytes(b"not a library")
        monkeypatch.setattr(host, "_PATH", tmp_path / "w4a8_host.so")
    with pytest.warns(RuntimeWarning, match="Python host path"):
        m = host.load()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert host.load() is m
    assert m.linear(*range(10)) is None and m.rms_norm(*range(6)) is None and m.moe(*range(16)) is None


def test_the_built_extension_is_for_this_torch():
    assert pkg("_host")._extension().built_for == pkg("_host")._running()


class _Off:
    """The extension as if it took no call."""

    linear = rms_norm = moe = staticmethod(lambda *a: None)


def _both(monkeypatch, fn):
    """fn() with the extension and without it: (result or exception) of each."""
    out = []
    for off in (False, True):
        with monkeypatch.context() as mp:
            if off:
                mp.setattr(pkg("_host"), "_mod", _Off)
            try:
                out.append(fn())
            except Exception as e:  # noqa: BLE001  (the refusals are compared)
                out.append((type(e), str(e)))
    torch.cuda.synchronize()
    return out


def _same(a, b):
    if isinstance(a, torch.Tensor):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    elif isinstance(a, tuple) and a and not isinstance(a[0], type):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a == b


def _weight(fmt, N, K, dev, E=None):
    if fmt == "mxfp4":
        w, s = synth.mxfp4_weight(N, K, seed=N + K, E=E)
        return w.to(dev), s.to(dev), None, 32, True
    if fmt == "nvfp4":
        w, s, z = synth.nvfp4_weight(N, K, seed=N + K, E=E)
        return w.to(dev), s.to(dev), z.view(torch.int32).to(dev), 16, True
    g = 64 if fmt == "asym64" else 128
    w, s, z = synth.int4_weight(N, K, g, seed=N + K, asym=fmt != "sym", scale_floor=1e-4, E=E)
    return w.to(dev), s.to(dev), None if z is None else z.to(dev), g, False


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["sym", "asym", "asym64", "mxfp4", "nvfp4"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_plain_calls_are_served_by_the_extension(kernels, dev, fmt, dtype):
    """What the comparisons below do not show, since a call that the extension leaves is the Python path's on
    both sides: it takes the calls it is there for."""
    m = pkg("_host").load()
    assert m is not pkg("_host")._Absent
    E, H, I = 8, 512, 256
    w, s, z, g, e2 = _weight(fmt, 96, H, dev)
    t = kernels.repack_w4(w, weight_is_e2m1=e2)
    w13, s13, z13, _, _ = _weight(fmt, 2 * I, H, dev, E=E)
    w2, s2, z2, _, _ = _weight(fmt, H, I, dev, E=E)
    t13, t2 = kernels.repack_w4(w13, e2), kernels.repack_w4(w2, e2)
    abi = pkg("_abi")
    for M in (1, 16, 17, 70):
        x = synth.activations(M, H, seed=M, dtype=dtype).to(dev)
        lg = synth.router_logits(M, E, seed=M).to(dev)
        q, sc = kernels.act_quant(x)
        out, arm = m.linear(x, t, s, z, g, e2, None, None, False, abi.KERNEL_AUTO)
        assert arm == (abi.KERNEL_DECODE if M <= 16 else abi.KERNEL_PREFILL)
        for call in (m.linear(x, t, s, z, g, e2, q, sc, False, abi.KERNEL_AUTO),
                     m.linear(x, torch.nn.Parameter(t, requires_grad=False), s, z, g, e2, None, None, False, abi.KERNEL_AUTO)):
            assert torch.equal(call[0], out)
        if M <= 16:
            assert m.linear(x, t, s, z, g, e2, None, None, True, abi.KERNEL_DECODE)[0].shape == (M, 48)
        assert m.rms_norm(x, None, 1e-6, False, None, False).shape == (M, H)
        assert len(m.rms_norm(x, x[0].clone(), 1e-6, False, x.clone(), True)) == 3
        bm = 16 if M <= 16 else 64
        assert m.moe(x, t13, s13, z13, t2, s2, z2, lg, 2, True, e2, bm, M == 1, True, True, M <= 16)[0].shape == (M, H)
    torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["sym", "asym", "asym64", "mxfp4", "nvfp4"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_forms(kernels, dev, monkeypatch, fmt, dtype):
    K, N = 512, 96
    w, s, z, g, e2 = _weight(fmt, N, K, dev)
    t = kernels.repack_w4(w, weight_is_e2m1=e2)
    eng = pkg("_hip_engage")
    for M in (0, 1, 5, 16, 17, 70):
        x = synth.activations(M, K, seed=M, dtype=dtype).to(dev)
        q, sc = kernels.act_quant(x)
        wide = torch.zeros(M, K + 8, dtype=dtype, device=dev)[:, :K].copy_(x)
        lin = lambda x=x, w=t, s=s, z=z, **k: kernels.w4a8_linear(x, w, s, z, g, weight_is_e2m1=e2, **k)  # noqa: E731
        forms = [lin, lambda: lin(x=wide), lambda: lin(w=w), lambda: lin(w=torch.nn.Parameter(t, requires_grad=False)),
                 lambda: lin(x_fp8=q, act_scales=sc), lambda: lin(x_fp8=q.view(torch.float8_e4m3fn), act_scales=sc),
                 lambda: lin(kernel="decode_gemv"), lambda: lin(kernel="wmma_tiled_tuned"),
                 lambda: lin(z=torch.empty(0, dtype=torch.int32, device=dev)),
                 # refused, or served by the Python path only
                 lambda: lin(x_fp8=q), lambda: lin(x_fp8=q[:, :64], act_scales=sc), lambda: lin(s=s.t()),
                 lambda: lin(s=s.float()), lambda: lin(x=x.float()), lambda: lin(x=x[None]), lambda: lin(kernel="nope"),
                 lambda: lin(x=x[:, :256]), lambda: lin(w=t[:, :2]), lambda: lin(s=s.t().contiguous().t()),
                 lambda: kernels.w4a8_linear_silu(x, t, s, z, g, weight_is_e2m1=e2),
                 lambda: kernels.w4a8_linear(x, t, s, z, 48, weight_is_e2m1=e2),
                 lambda: kernels.w4a8_linear(x, t, s, z, g, weight_is_e2m1=not e2)]
        if fmt == "nvfp4":
            forms += [lambda: lin(z=z.view(torch.float32)), lambda: lin(s=s.view(torch.uint8)), lambda: lin(z=None)]
        for i, f in enumerate(forms):
            n0 = eng.counts()
            a, b = _both(monkeypatch, f)
            _same(a, b)
            moved = eng.counts_delta(n0)
            assert all(v == 2 for v in moved.values()), (i, moved)  # the same ledger entry from either path


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["sym", "asym", "asym64", "mxfp4", "nvfp4"])
def test_moe_forms(kernels, dev, monkeypatch, fmt):
    E, H, I = 16, 512, 256
    w13, s13, z13, _, e2 = _weight(fmt, 2 * I, H, dev, E=E)
    w2, s2, z2, _, _ = _weight(fmt, H, I, dev, E=E)
    t13, t2 = kernels.repack_w4(w13, e2), kernels.repack_w4(w2, e2)
    eng = pkg("_hip_engage")
    for T in (0, 1, 4, 9, 20, 40, 200):
        x = synth.activations(T, H, seed=T).to(dev)
        lg = synth.router_logits(T, E, seed=T + 1).to(dev)
        moe = lambda x=x, w=t13, lg=lg, k=4, s=s13, **kw: kernels.w4a8_moe(  # noqa: E731
            x, w, s, z13, t2, s2, z2, lg, k, True, weight_is_e2m1=e2, **kw)
        tw, ids = kernels._moe_route(lg, 4, True, E) if T else (None, None)
        forms = [moe, lambda: moe(k=2), lambda: moe(block_m=16), lambda: moe(block_m=64), lambda: moe(block_m=128),
                 lambda: moe(lg=lg.float()), lambda: moe(w=w13), lambda: moe(activation="gelu"),
                 lambda: moe(topk_ids=ids, topk_weights=tw) if T else None,
                 lambda: moe(lg=lg[:, :8]), lambda: moe(lg=lg[:, :8].contiguous()), lambda: moe(x=x.float()),
                 lambda: moe(s=s13.transpose(1, 2)), lambda: moe(lg=None), lambda: moe(activation="relu"),
                 lambda: moe(act_scales=torch.ones(T, device=dev))]
        for i, f in enumerate(forms):
            n0 = eng.counts()
            a, b = _both(monkeypatch, f)
            _same(a, b)
            assert all(v % 2 == 0 for v in eng.counts_delta(n0).values()), i


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_norm_forms(dev, monkeypatch, dtype):
    norm = pkg("layers.norm")
    K = 768
    gain = (1 + 0.1 * synth.activations(1, K, seed=3)[0].float()).to(dtype).to(dev)
    for shape in ((1, K), (7, K), (2, 3, K), (K,), (0, K)):
        x = synth.activations(max(1, torch.Size(shape).numel() // K), K, seed=4, dtype=dtype).to(dev)
        x = x[:0] if 0 in shape else x.view(shape)
        res = (x * 0.5).contiguous()
        forms = [lambda: norm._rms_norm(x, gain, 1e-6), lambda: norm._rms_norm(x, None, 1e-6),
                 lambda: norm._rms_norm(x, gain, 1e-6, True), lambda: norm._rms_norm_quant(x, gain, 1e-6),
                 lambda: norm._rms_norm(x, gain.float(), 1e-6), lambda: norm._rms_norm_quant(x.float(), gain, 1e-6)]
        if x.dim() > 1:
            forms.append(lambda: norm._rms_norm_quant(x.transpose(0, 1), gain, 1e-6) if x.shape[0] == K else None)

        def add():
            r = res.clone()
            return (*norm._rms_norm_add_quant(x, r, gain, 1e-6), r, norm._rms_norm_add(x, res.clone(), gain, 1e-6))

        for f in forms + [add]:
            _same(*_both(monkeypatch, f))

"""The native host path of short launches (csrc/host.cpp) against the Python
path it stands in front of: the same bits, and the same calls refused."""
import pytest
import torch

DEV = "cuda"
DTYPES = [torch.float16, torch.bfloat16, torch.float32]


def _layer(n, k, seed=0):
    from quant_models import ops

    g = torch.Generator(device=DEV).manual_seed(seed)
    planes = [torch.randint(0, 256, (n, k // 4), generator=g, device=DEV, dtype=torch.uint8) for _ in range(4)]
    scale = [0.01 + 0.03 * torch.rand(n, 1, generator=g, device=DEV) for _ in range(4)]
    return ops.PackedWide.from_planes(planes, scale, scale, n, k), g


def _both(monkeypatch, f):
    """f() on the native path and on the Python path."""
    from quant_models import _native as N

    assert N.host() is not None
    native = f()
    with monkeypatch.context() as m:
        m.setattr(N, "_host", False)
        return native, f()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(1, 500, 384), (8, 48, 16), (17, 96, 96), (197, 384, 384), (600, 100, 64)])
def test_native_linear_equals_python_path(m, n, k, dtype, monkeypatch):
    pw, g = _layer(n, k)
    bias = torch.randn(2 * n, device=DEV, generator=g)
    ln = [torch.randn(2 * k, device=DEV, generator=g) for _ in range(2)]
    x = torch.randn(1, m, 2 * k, device=DEV, generator=g).to(dtype)
    for out in DTYPES:
        r = torch.randn(1, m, 2 * n, device=DEV, generator=g).to(out)
        for kw in ({}, {"residual": r}, {"gelu": True}):
            for b in (None, bias):
                a, c = _both(monkeypatch, lambda: pw.linear(x, b, out_dtype=out, **kw))
                assert a.shape == (1, m, 2 * n) and torch.equal(a, c)
    if pw.ln_fusable(m, dtype):
        assert torch.equal(*_both(monkeypatch, lambda: pw.layer_norm_linear(x, *ln, 1e-5, bias)))
        assert torch.equal(*_both(monkeypatch, lambda: pw.act_quant_linear(x, 4, bias)))


@pytest.mark.gpu
def test_native_path_leaves_other_calls_to_python(monkeypatch):
    """Strided, offset and other-dtype operands, empty inputs, and errors."""
    from quant_models import _native as N
    from quant_models import ops

    pw, g = _layer(48, 32)
    x = torch.randn(6, 64, device=DEV, generator=g).half()
    bias = torch.randn(96, device=DEV, generator=g)
    forms = [x.t().contiguous().t(), torch.cat((x, x), 1)[:, 64:], torch.zeros(385, device=DEV, dtype=torch.half)[1:].view(6, 64).copy_(x)]
    for f in forms:
        assert torch.equal(pw.linear(f, bias), pw.linear(x, bias))
    assert torch.equal(pw.linear(x, bias.double()), pw.linear(x, bias))
    assert torch.equal(pw.linear(x, bias, residual=torch.ones(6, 96, device=DEV)), pw.linear(x, bias, residual=torch.ones(6, 96, device=DEV).half()))
    assert pw.linear(x[:0], bias).shape == (0, 96)
    for bad in (lambda: pw.linear(x[:, :32]), lambda: pw.linear(x.cpu()), lambda: pw.linear(x, residual=x),
                lambda: pw.linear(x, residual=torch.ones(6, 96, device=DEV).half(), gelu=True)):
        with pytest.raises(ValueError):
            bad()
    with pytest.raises(TypeError):
        pw.linear(x.double())
    with pytest.raises(N.RPFQError):
        pw.linear(x, flags=N.FLAG_STREAM | N.FLAG_NO_STREAM)
    qkv = torch.randn(2, 20, 3 * 128, device=DEV, generator=g).half()
    assert torch.equal(*_both(monkeypatch, lambda: ops.attention(qkv, 2, 0.125)))
    with pytest.raises(N.RPFQError):
        ops.attention(qkv, 4, 0.125)


@pytest.mark.gpu
def test_native_path_runs_on_the_current_stream():
    pw, g = _layer(96, 96)
    x = torch.randn(4, 192, device=DEV, generator=g).half()
    ref = pw.linear(x)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        z = x.clone()
        for _ in range(50):
            z = z + 0
        y = pw.linear(z)
    s.synchronize()
    assert torch.equal(y, ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = pw.linear(x)
    for _ in range(3):
        x.mul_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, pw.linear(x))


@pytest.mark.gpu
def test_native_path_allocates_nothing_for_calls_it_leaves(monkeypatch):
    """A call that goes on to the Python path allocates what it allocates there."""
    from quant_models import _native as N

    pw, g = _layer(384, 384)
    x = torch.randn(1576, 768, device=DEV, generator=g).bfloat16()  # prescaled rows, the DMA kernel
    half = torch.randn(8, 768, device=DEV, generator=g).half()
    calls = [lambda: pw.linear(x), lambda: pw.linear(half, torch.ones(768, device=DEV).double()),
             lambda: pw.layer_norm_linear(half.expand(4, 8, 768).contiguous(), torch.ones(768, device=DEV).double(), None, 1e-5)]
    assert pw.kernel_for(1576, torch.float16, torch.bfloat16) == N.KERNEL_DMA

    def count(f):
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        f()
        return torch.cuda.memory_stats()["allocation.all.allocated"] - before

    for f in calls:
        f()
        native = count(f)
        with monkeypatch.context() as m:
            m.setattr(N, "_host", False)
            assert native == count(f)


@pytest.mark.gpu
def test_native_path_launches_without_the_interpreter_lock():
    """Every launch function of the native path replaced by the interpreter's
    own PyGILState_Check: 0 (the lock is free), read as success, or 1, read as
    a refused call."""
    import ctypes

    from quant_models import _native as N

    pw, g = _layer(384, 384)
    x = torch.randn(20, 768, device=DEV, generator=g).half()
    host, lib, d = N.host(), N.load(), ctypes.addressof(pw.desc)
    address = {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in host.CALLS}
    check = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    # these two choose a kernel and launch nothing
    chooses = ("rpfq_wide_linear_kernel", "rpfq_layer_norm_wide_linear_fusable")
    host.bind(tuple(address[name] if name in chooses else check for name in host.CALLS))
    try:
        taken = [host.linear(d, pw.blob, x, None, None, None, 0, 3), host.linear(d, pw.blob, x.float(), None, None, None, 0, 1),
                 host.layer_norm_linear(d, pw.blob, x, None, None, 1e-5, None, None, 0),
                 host.act_quant_linear(d, pw.blob, x, 4, None, None, None, 0),
                 host.attention(x.new_zeros(1, 5, 192), 1, 0.125)]
    finally:
        host.bind(tuple(address[name] for name in host.CALLS))
    assert pw.ln_fusable(20, torch.float16)
    assert all(t is not None for t in taken)


@pytest.mark.gpu
def test_native_path_from_several_threads():
    """Threads on their own streams get the results of one thread."""
    import threading

    from quant_models import ops

    pw, g = _layer(96, 96)
    xs = [torch.randn(1 + 3 * t, 192, device=DEV, generator=g).half() for t in range(4)]
    qkv = [torch.randn(1, 5 + 40 * t, 384, device=DEV, generator=g).half() for t in range(4)]
    want = [(pw.linear(x), ops.attention(q, 2, 0.125)) for x, q in zip(xs, qkv)]
    torch.cuda.synchronize()
    same = [False] * 4

    def work(t):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            got = [(pw.linear(xs[t]), ops.attention(qkv[t], 2, 0.125)) for _ in range(200)]
        s.synchronize()
        same[t] = all(torch.equal(a, b) for pair in got for a, b in zip(pair, want[t]))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(same)


def test_native_path_takes_device_tensors_only():
    from quant_models import _native as N

    host = N.host()
    assert host is not None, "quant_models/_host.so is not built"
    t = torch.zeros(4, 64, dtype=torch.half)
    assert host.linear(0, t, t, None, None, None, 0, 3) is None
    assert host.linear(t) is None
    assert host.attention(t, 1, 0.125) is None


def test_native_path_leaves_other_numbers_to_python():
    """Numbers of another kind (heads = 2.0) and too large ones are not taken,
    and leave no Python error behind."""
    from quant_models import _native as N

    host = N.host()
    t = torch.zeros(4, 64, dtype=torch.half)
    assert host.attention(t, 2.0, 0.125) is None
    assert host.attention(t, 2, "scale") is None
    assert host.linear(1 << 80, t, t, None, None, None, 0, 3) is None
    assert host.linear(0, t, t, None, None, None, 0.5, 3) is None
    assert host.linear(0, t, t, None, None, None, 1 << 80, 3) is None
    assert host.layer_norm_linear(0, t, t, None, None, None, None, None, 0) is None
    assert host.act_quant_linear(0, t, t, "4", None, None, None, 0) is None


def test_native_path_calls_the_library_that_was_loaded(tmp_path):
    """RPFQ_LIBRARY names another build: the default one is not loaded beside
    it, so every call of the process runs the named one."""
    import os
    import shutil
    import subprocess
    import sys

    from quant_models import _native as N

    other = tmp_path / "librpfq_other.so"
    shutil.copy(N.library_path(), other)
    code = ("from quant_models import _native as N; host = N.host(); assert host is not None; "
            "print(*sorted({l.split()[-1] for l in open('/proc/self/maps') if 'librpfq' in l}))")
    env = dict(os.environ, RPFQ_LIBRARY=str(other), PYTHONPATH=os.path.dirname(os.path.dirname(N.__file__)))
    out = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr
    assert out.stdout.split() == [str(other)]
    host = N.host()
    for bad in ((), (0,) * len(host.CALLS), (1 << 80,) * len(host.CALLS), [1]):
        with pytest.raises((ValueError, OverflowError)):
            host.bind(bad)


def test_native_path_is_built_for_the_installed_torch():
    """Another torch rebuilds it; without torch's headers the library is built
    and the native path left out."""
    import os
    import subprocess

    from quant_models import _native as N

    csrc = os.path.join(os.path.dirname(N.library_path()), "csrc")

    def plan(*args):
        out = subprocess.run(["make", "-n", "-C", csrc, *args], capture_output=True, text=True, timeout=120)
        assert out.returncode == 0, out.stderr
        return out.stdout

    assert "host.cpp" in plan("TORCH_VERSION=0.0.other")
    without = plan("-B", "TORCH=/nonexistent")
    assert "host.cpp" not in without and "librpfq.so" in without

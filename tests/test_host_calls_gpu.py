"""The ops' native bodies against their Python ones: the same launches, so the same bits
where both serve a call, and the Python body's answer or refusal everywhere else."""

from __future__ import annotations

import math
import struct
from contextlib import contextmanager

import pytest
import torch

from mini_vllm.kernels import extension as ext_module
from mini_vllm.kernels import ops
from mini_vllm import torch_path
from mini_vllm.workloads import build_batch

gpu = pytest.mark.gpu


@contextmanager
def python_bodies(ext):
    host, ext._host = ext._host, None
    try:
        yield
    finally:
        ext._host = host


def both(ext, call):
    """The op's result with the native body (its second call: the first may grow the
    workspace) and with the Python one, or the error each raises."""
    def run():
        try:
            return call()
        except (RuntimeError, TypeError) as e:
            return str(e)
    run()
    native = run()
    with python_bodies(ext):
        python = run()
    return native, python


def assert_same(native, python):
    if isinstance(python, torch.Tensor):
        assert isinstance(native, torch.Tensor) and native.dtype == python.dtype
        assert native.shape == python.shape and native.stride() == python.stride()
        assert torch.equal(native, python)
    elif isinstance(python, tuple):
        assert len(native) == len(python)
        for a, b in zip(native, python):
            assert_same(a, b)
    else:
        assert native == python


def test_the_built_module_matches_its_source():
    if not ext_module.HOST_PATH.exists():
        pytest.skip("the host module is not built")
    host = ext_module.open_host()  # None for a stale build
    assert host is not None and host.source_hash == ext_module.host_hash()
    x = torch.zeros(2, 64, dtype=torch.bfloat16)  # host memory: not a call it serves
    entries = host.entries(*[0] * 7)
    assert host.linear_swiglu(entries, {}, x, x, 32) is None
    assert host.paged_attention(entries, {}, *[x] * 12) is None
    assert host.paged_served(*[x] * 12) is False
    with pytest.raises(ValueError):
        host.linear_swiglu(x, {}, x, x, 32)  # not the library's entries


def test_the_module_has_no_thread_local_storage():
    """A late-loaded module with a TLS segment slows every other library's thread-local
    accesses (glibc before 2.39), and so every op that is not the module's."""
    if not ext_module.HOST_PATH.exists():
        pytest.skip("the host module is not built")
    elf = ext_module.HOST_PATH.read_bytes()
    at, = struct.unpack_from("<Q", elf, 32)  # the ELF64 header's e_phoff, e_phentsize, e_phnum
    size, count = struct.unpack_from("<HH", elf, 54)
    kinds = [struct.unpack_from("<I", elf, at + i * size)[0] for i in range(count)]
    assert 1 in kinds and 7 not in kinds  # PT_LOAD, PT_TLS


def test_a_module_that_is_not_this_build_is_left_alone(tmp_path, monkeypatch, capsys):
    """Other sources' or another torch's (told by its id, before it is loaded), or a file that
    does not load: no module and a warning, and the Python bodies serve, as where there is
    none."""
    if not ext_module.HOST_PATH.exists():
        pytest.skip("the host module is not built")
    built = ext_module.HOST_PATH.read_bytes()
    ident = b"mvllm-host-id:" + ext_module.host_hash().encode()
    assert built.count(ident) == 1
    path = tmp_path / "mvllm_host.so"
    monkeypatch.setattr(ext_module, "HOST_PATH", path)
    assert ext_module.open_host() is None and capsys.readouterr().err == ""  # not built
    for content in (built.replace(ident, b"mvllm-host-id:0123456789abcdef"), b"not a library",
                    b"not a library but " + ident):
        path.write_bytes(content)
        assert ext_module.open_host() is None
        assert "rebuilt" in capsys.readouterr().err


def test_no_host_compiler_is_no_build_error(tmp_path, monkeypatch, capsys):
    """Without one the module is left out, a stale one with it, and the library is built."""
    path = tmp_path / "mvllm_host.so"
    path.write_bytes(b"stale")
    monkeypatch.setattr(ext_module, "HOST_PATH", path)
    monkeypatch.setattr(ext_module, "CXX", "no-such-compiler")
    assert ext_module.build_host() is None and not path.exists()
    assert "no-such-compiler" in capsys.readouterr().err


@gpu
@pytest.mark.parametrize("contexts,lens,dtype,kv", [
    ([1], [1], torch.bfloat16, None),
    ([300, 17], [1, 1], torch.float32, None),
    ([400, 90, 33], [1, 1, 1], torch.bfloat16, torch.float8_e4m3fn),
    ([200, 70], [64, 1], torch.float16, None),
])
def test_paged_attention(extension, contexts, lens, dtype, kv):
    kwargs = {} if kv is None else {"kv_dtype": kv}
    b = build_batch(contexts, lens, dtype=dtype, seed=3, device="cuda:0", **kwargs)
    scales = dict(k_scale=b.k_scale, v_scale=b.v_scale)
    args = list(b.args())
    q, kp, vp, tables, cu, ctx, seq, mq, mc, *rest = args

    def op(*a, **kw):
        return lambda: ops.paged_attention(*a, use_cuda=True, **{**scales, **kw})
    served = extension._host.paged_served(q, kp, vp, tables, cu, ctx, seq, mq, mc, 0.1,
                                          b.k_scale, b.v_scale)
    assert served
    native, python = both(extension, op(*args))
    assert_same(native, python)
    own = extension._host.paged_attention(  # the native body itself, its workspace there by now
        extension._entries, extension._workspaces, q, kp, vp, tables, cu, ctx, seq, mq, mc,
        1.0 / math.sqrt(q.shape[-1]), b.k_scale, b.v_scale)
    assert own is not None
    assert_same(own, python)
    stream = torch.cuda.Stream()  # a workspace of its own, not there at the first call
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        assert_same(*both(extension, op(*args)))
    torch.cuda.current_stream().wait_stream(stream)
    odd = [
        (q, kp, vp, tables, cu, ctx.repeat_interleave(2)[::2], seq, mq, mc),  # strided lengths
        (q, kp, vp, tables, cu, ctx, seq, mq, 0),
        (q, kp, vp, tables, cu[:-1], ctx, seq, mq, mc),
        (q, kp, vp[:-1], tables, cu, ctx, seq, mq, mc),
        (q[:0], kp, vp, tables, cu, ctx, seq, mq, mc),
        (q[:, :-1].contiguous(), kp, vp, tables, cu, ctx, seq, mq, mc),
    ]
    for case in odd:
        assert_same(*both(extension, op(*case)))
    wrong = {"k_scale": None if kv is not None else torch.ones(1, device="cuda:0")}
    assert_same(*both(extension, op(*args, **wrong)))


@gpu
@pytest.mark.parametrize("m", [1, 33, 64, 65])
@pytest.mark.parametrize("k,n", [(64, 32), (1024, 3072), (3072, 1024), (3072, 1000)])
def test_projections(extension, m, k, n):
    gen = torch.Generator().manual_seed(m * k + n)

    def rand(*shape):
        return (torch.randn(*shape, generator=gen) / 8).to("cuda:0", torch.bfloat16)
    x, residual, norm = rand(m, k), rand(m, n), rand(n)
    w = ops.pack_weight(rand(n, k), use_cuda=True)
    wide = rand(m, 2 * k)[:, ::2]  # a strided input
    for a in (x, wide, x.half()):
        taken = a is x and m <= 64  # the calls that the native bodies are to serve
        def residual_norm(a=a):
            return ops.linear_residual_rmsnorm(a, w, residual, norm, 1e-6, use_cuda=True)
        native, python = both(extension, residual_norm)
        assert_same(native, python)
        own = extension.try_linear_residual_rmsnorm(a, w.packed, n, residual, norm, 1e-6)
        assert (own is not None) == (taken and k > 1024 and n % 512 == 0)
        if own is not None:
            assert_same(own, python)
        if n % 32 == 0 and a.dtype == x.dtype:
            native, python = both(extension, lambda a=a: ops.linear_swiglu(a, w, use_cuda=True))
            assert_same(native, python)
            own = extension.try_linear_swiglu(a, w.packed, n)
            assert (own is not None) == taken
            if own is not None:
                assert_same(own, python)
    with extension.recording_workspaces() as held:  # the buffers that a graph keeps alive
        ops.linear_residual_rmsnorm(x, w, residual, norm, 1e-6, use_cuda=True)
    assert bool(held) == (m <= 64 and k > 1024 and n % 512 == 0)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("contexts", [[1], [700, 16, 17, 250]])
def test_the_fused_decode_step(extension, contexts, dtype):
    seqs = len(contexts)
    b = build_batch(contexts, [1] * seqs, dtype=dtype, seed=5, device="cuda:0")
    q, kp, vp, tables, cu, ctx, seq, _, mc, *_ = b.args()
    hq, hk, d = q.shape[1], kp.shape[2], q.shape[2]
    gen = torch.Generator().manual_seed(9)

    def rand(*shape):
        return torch.randn(*shape, generator=gen).to("cuda:0", dtype)
    qkv = rand(seqs, (hq + 2 * hk) * d)
    views = [t.view(seqs, -1, d) for t in qkv.split([hq * d, hk * d, hk * d], dim=1)]
    qw, kw = rand(d), rand(d)
    cos, sin = torch_path.rope_tables(d, 1024, 1e6, device="cuda:0")

    def op(q, k, v, qw=qw, pools=(kp, vp), max_context=mc):
        def call():
            kp, vp = (p.clone() for p in pools)
            return ops.paged_decode_qk_norm_rope(
                q, k, v, qw, kw, cos, sin, 1e-6, kp, vp, tables, cu, ctx, seq, max_context,
                0.09, use_cuda=True), kp, vp
        return call
    def native_serves(q, k, v, qw=qw):
        kp2, vp2 = kp.clone(), vp.clone()
        out = extension.try_paged_decode_qk_norm_rope(q, k, v, qw, kw, cos, sin, 1e-6, kp2, vp2, tables,
                                                      cu, ctx, seq, mc, 0.09)
        return None if out is None else (out, kp2, vp2)
    for rows in (views, [t.contiguous() for t in views]):
        native, python = both(extension, op(*rows))
        assert_same(native, python)
        own = native_serves(*rows)
        assert own is not None
        assert_same(own, python)
    q, k, v = views
    assert native_serves(q, k[:, :-1], v) is None
    assert native_serves(q, k, v, qw=qw.float()) is None
    assert_same(*both(extension, op(q, k, v.contiguous())))       # k and v apart
    assert_same(*both(extension, op(q, k, v, qw=qw.float())))     # not the kernel's dtype
    assert_same(*both(extension, op(q, k[:, :-1], v)))
    assert_same(*both(extension, op(q, k, v, max_context=0)))

"""The wrappers' native host path (csrc/host_calls.cpp): on the GPU, every form
of call gives the same bits and the same errors with it as without it; on the
CPU, it declines whatever is not a GPU tensor."""
import ctypes
import shutil
import subprocess
import threading

import pytest
import torch

from vllm_apple_amd import _lib, backend, kernels

NAMES = ["norm", "silu", "epilogue", "topk", "gate_up", "linear", "kv_write", "decode",
         "step_decode", "step_prefill", "prefill", "no_cache"]
COUNTS = dict(norm=7, silu=4, epilogue=13, topk=6, gate_up=6, linear=5, kv_write=7, decode=14,
              step_decode=16, step_prefill=16, prefill=14, no_cache=13)


@pytest.mark.parametrize("name", NAMES)
def test_declines_other_objects(name):
    fn = getattr(_lib.host(), name)
    t = torch.zeros(4, 4, 8, dtype=torch.float16)
    for a in (None, t, t[0], 3, "x", 2.5, object()):
        assert fn(*[a] * COUNTS[name]) is False
    with pytest.raises(TypeError):
        fn(t)


# Entry points that only count their calls; every size query asks for 64 bytes.
_STUB = """
#include <stddef.h>
#include <unistd.h>
int calls, delay_ms, inside, version;
int vaa_abi_version() { return version; }
int vaa_topk_workspace_size(int t, int v, int k, size_t* n) { *n = 64; return 0; }
""" + "".join(f"size_t {f}() {{ return 64; }}\n" for f in (
    "decode_workspace", "prefill_workspace", "step_workspace", "gate_workspace",
    "linear_workspace", "no_cache_workspace")) + """
int launch() {
  ++calls;
  inside = 1;
  usleep(1000 * delay_ms);
  inside = 0;
  return 0;
}
"""
_STUB_NAMES = {
    "decode_workspace": ["vaa_paged_attention_decode_workspace_size"],
    "prefill_workspace": ["vaa_paged_attention_prefill_workspace_size"],
    "step_workspace": ["vaa_prefill_step_workspace_size"],
    "gate_workspace": ["vaa_gate_up_silu_workspace_size"],
    "linear_workspace": ["vaa_linear_workspace_size"],
    "no_cache_workspace": ["vaa_attention_no_cache_workspace_size"],
    "launch": ["vaa_kv_write_slots", "vaa_paged_attention_decode", "vaa_paged_attention_prefill",
               "vaa_paged_attention_prefill_split", "vaa_paged_attention_prefill_tiles",
               "vaa_prefill_step", "vaa_rmsnorm", "vaa_add_rmsnorm", "vaa_silu_mul",
               "vaa_qkv_epilogue", "vaa_topk_logits", "vaa_gate_up_silu_split", "vaa_linear",
               "vaa_attention_no_cache"]}


@pytest.fixture(scope="module")
def stub_lib(tmp_path_factory):
    if shutil.which("gcc") is None:
        pytest.skip("gcc not available")
    d = tmp_path_factory.mktemp("stub")
    so = d / "stub.so"
    (d / "stub.c").write_text(_STUB)
    alias = [f"-Wl,--defsym={n}={f}" for f, ns in _STUB_NAMES.items() for n in ns]
    subprocess.run(["gcc", "-shared", "-fPIC", str(d / "stub.c"), "-o", str(so), *alias],
                   check=True)
    lib = ctypes.CDLL(str(so))
    ctypes.c_int.in_dll(lib, "version").value = _lib.ABI_VERSION
    return lib


@pytest.fixture
def stub(stub_lib):
    """The native path bound to entry points that launch nothing."""
    host = _lib.host()
    host.bind(stub_lib._handle)
    yield host, ctypes.c_int.in_dll(stub_lib, "calls")
    ctypes.c_int.in_dll(stub_lib, "delay_ms").value = 0
    host.bind(_lib.load()._handle)


_memory = ctypes.create_string_buffer(1 << 20)


def _on(device, shape, dtype=torch.float16):
    """A tensor that says it lives on cuda:`device` (its memory is the host's
    and is never read)."""
    base = (ctypes.addressof(_memory) + 255) // 256 * 256
    storage = torch._C._construct_storage_from_data_pointer(
        base, torch.device("cuda", device), len(_memory) - 256)
    strides = [1] * len(shape)
    for i in range(len(shape) - 1, 0, -1):
        strides[i - 1] = strides[i] * shape[i]
    return torch._C._construct_CUDA_Tensor_From_Storage_And_Metadata(
        dict(dtype=dtype, device=torch.device("cuda", device), size=tuple(shape),
             stride=tuple(strides), storage_offset=0), storage)


def _apart(t, elements):
    """The same tensor `elements` further on in the memory."""
    return t.as_strided(t.shape, t.stride(), elements)


def _accepted(name, dev=lambda i: 0):
    """Arguments that `name` takes whole; dev(i): the device of argument i."""
    n, H, KV, D, i32, i64 = 4, 4, 2, 64, torch.int32, torch.int64

    def t(i, *shape, dtype=torch.float16):
        return _on(dev(i), shape, dtype)
    ws = lambda i: t(i, 64, dtype=torch.uint8)  # noqa: E731
    kv = lambda i: t(i, 8, 16, KV, D)  # noqa: E731
    if name == "norm":
        return [t(0, n, D), t(1, D), t(2, n, D), t(3, n, D), 1e-5, 0, False]
    if name == "silu":
        return [t(0, n, D), t(1, n, D), t(2, n, D), 0]
    if name == "epilogue":
        return [t(0, n, H, D), t(1, n, KV, D), t(2, n, KV, D), t(3, n, dtype=i32),
                t(4, 9, D // 2, dtype=torch.float32), t(5, 9, D // 2, dtype=torch.float32),
                t(6, n, dtype=i64), kv(7), kv(8), t(9, (H + 2 * KV) * D), D, True, 0]
    if name == "topk":
        return [t(0, n, 9000), 5, t(2, n, 5, dtype=i32), t(3, n, 5), ws(4), 0]
    if name == "gate_up":
        return [t(0, n, D), t(1, 128, D), t(2, 128, D), t(3, n, 128), ws(4), 0]
    if name == "linear":
        return [t(0, n, D), t(1, 128, D), t(2, n, 128), ws(3), 0]
    if name == "kv_write":
        return [t(0, n, KV, D), t(1, n, KV, D), kv(2), kv(3), t(4, n, dtype=i64), True, 0]
    if name == "decode":
        return [t(0, n, H, D), kv(1), kv(2), t(3, n, 3, dtype=i32), t(4, n, dtype=i32),
                t(5, n, H, D), t(6, n, KV, D), t(7, n, KV, D), True, 0.1, 40, 0, ws(12), 0]
    if name == "step_decode":
        return [t(0, n, H, D), t(1, n, KV, D), t(2, n, KV, D), t(3, 2, 8, 16, KV, D),
                t(4, n, H, D), t(5, n, 3, dtype=i32), t(6, n, dtype=i32), t(7, n, dtype=i64), n,
                True, D, 0.1, 40, 0, ws(14), 0]
    if name == "step_prefill":
        return [t(0, n, H, D), t(1, n, KV, D), t(2, n, KV, D), t(3, 2, 8, 16, KV, D),
                t(4, n, H, D), t(5, 2, 3, dtype=i32), t(6, 2, dtype=i32), t(7, n, dtype=i64),
                t(8, 3, dtype=i32), n, True, D, 0.1, True, ws(14), 0]
    if name == "prefill":
        return [t(0, n, H, D), kv(1), kv(2), t(3, 2, 3, dtype=i32), t(4, n, dtype=i32),
                t(5, n, dtype=i32), t(6, n, H, D), True, 0.1, t(9, 2, 2, dtype=i32), 64, 40,
                ws(12), 0]
    return [t(0, n, H, D), t(1, n, KV, D), t(2, n, KV, D), _apart(t(3, n, H, D), 4096),
            t(4, 3, dtype=i32), n, 2, D, 0.1, 3, False, ws(11), 0]


@pytest.mark.parametrize("name", NAMES)
def test_tensors_of_two_devices_are_declined(stub, name):
    """A call whose tensors are on one device is taken; with any one of them on
    another device nothing is launched."""
    host, calls = stub
    fn, args = getattr(host, name), _accepted(name)
    assert len(args) == COUNTS[name]
    assert fn(*args) is True
    for i, a in enumerate(args):
        if not isinstance(a, torch.Tensor):
            continue
        calls.value = 0
        done = fn(*_accepted(name, lambda j, i=i: int(j == i)))
        assert done is not True and calls.value == 0, f"argument {i}"
    assert fn(*_accepted(name, lambda j: 1)) is True


def test_product_is_left_to_torch_where_it_would_do_more(stub):
    """The product that stands in for torch.matmul(out=) declines what the
    library call refuses or hands on: a gradient to record, a dispatch mode.  It
    counts as a write to its output."""
    from torch.utils._python_dispatch import TorchDispatchMode

    host, calls = stub
    for i in range(3):
        args = _accepted("linear")
        args[i].requires_grad_()
        calls.value = 0
        assert host.linear(*args) is False and calls.value == 0
        with torch.no_grad():
            assert host.linear(*args) is True
    args = _accepted("linear")
    version = args[2]._version
    assert host.linear(*args) is True and args[2]._version == version + 1

    class Sees(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    args = _accepted("linear")
    with Sees():
        assert host.linear(*args) is False
    assert host.linear(*args) is True


def test_a_library_of_another_version_is_refused(stub, stub_lib, monkeypatch):
    """The host path calls entry points by the signatures it was built with: it
    binds to no library of another version, and loading one says so."""
    host, calls = stub
    version = ctypes.c_int.in_dll(stub_lib, "version")
    try:
        for other in (_lib.ABI_VERSION - 1, _lib.ABI_VERSION + 1):
            version.value = other
            with pytest.raises(RuntimeError, match="version"):
                host.bind(stub_lib._handle)
    finally:
        version.value = _lib.ABI_VERSION

    def refuse(handle):
        raise RuntimeError("ABI version mismatch")
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_host", None)
    from vllm_apple_amd import _host
    monkeypatch.setattr(_host, "bind", refuse)
    with pytest.raises(_lib.NativeLibraryError, match="build_library"):
        _lib.load()


@pytest.mark.parametrize("name", NAMES)
def test_launches_leave_the_interpreter_to_other_threads(stub, stub_lib, name):
    """While one thread's launch blocks (a full queue), another runs Python."""
    host, _ = stub
    ctypes.c_int.in_dll(stub_lib, "delay_ms").value = 150
    inside = ctypes.c_int.in_dll(stub_lib, "inside")
    done = []
    worker = threading.Thread(
        target=lambda: done.append(getattr(host, name)(*_accepted(name))))
    worker.start()
    seen = 0
    while not done:
        seen |= inside.value
    worker.join()
    assert done == [True] and seen == 1


class _Declines:
    """A native path that declines everything: the wrappers' own path runs."""

    def __getattr__(self, name):
        return lambda *a: False


def _both(monkeypatch, call):
    """call() with the native path and without it: (result or error) of each."""
    out, used = [], []
    real = _lib.host()

    class Spy:
        def __getattr__(self, name):
            f = getattr(real, name)
            return lambda *a: used.append(f(*a)) or used[-1]

    for host in (Spy(), _Declines()):
        monkeypatch.setattr(_lib, "host", lambda host=host: host)
        try:
            out.append(call())
        except Exception as e:  # noqa: BLE001
            out.append((type(e), str(e)))
        torch.cuda.synchronize()
    monkeypatch.undo()
    return out, True in used


def _same(a, b):
    if isinstance(a, torch.Tensor):
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
    elif isinstance(a, (list, tuple)) and not isinstance(a[0], type):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a == b


def _rand(*shape, dtype=torch.float16, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g).to(dtype).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_layer_ops(gpu, monkeypatch, dtype):
    wide = _rand(5, 192, dtype=dtype)
    forms = [(wide[:, :128], True), (wide[:, 1:129], True), (wide.t()[:128, :5], False),
             (wide[:0, :128], True), (wide[:, :128].float(), False)]
    w = _rand(128, dtype=dtype)
    for x, native in forms:
        def norm(x=x):
            out, res = torch.empty_like(x), x.clone()
            kernels.rms_norm(x, w[:x.shape[1]], 1e-5, residual=res, out=out)
            out2 = torch.empty_like(x)
            kernels.add_rms_norm(x, res, w[:x.shape[1]], 1e-5, out=out2)
            return out, out2, res
        (a, b), used = _both(monkeypatch, norm)
        _same(a, b)
        assert used is native

        def silu(x=x):
            return kernels.silu_mul(x.contiguous(), x.contiguous(),
                                    out=torch.empty(x.shape, dtype=x.dtype, device="cuda"))
        (a, b), _ = _both(monkeypatch, silu)
        _same(a, b)
    (a, b), used = _both(monkeypatch, lambda: kernels.rms_norm(wide, w, 1e-5, out=wide.clone()))
    _same(a, b)  # a weight of another length: the same error
    assert isinstance(a, tuple) and a[0] is ValueError and not used


@pytest.mark.gpu
@pytest.mark.parametrize("slots_dtype", [torch.int32, torch.int64, torch.int16])
@pytest.mark.parametrize("layout", ["kernel", "vllm", "other"])
def test_kv_write_and_epilogue(gpu, monkeypatch, layout, slots_dtype):
    T, H, KV, D = 6, 4, 2, 64
    qkv = _rand(T, (H + 2 * KV) * D)
    shape = (3, KV, 16, D) if layout == "kernel" else (3, 16, KV, D)
    slots = torch.tensor([0, 5, -1, 33, 47, 16], dtype=slots_dtype).cuda()
    cos, sin = kernels.rope_cos_sin_cache(D, 64, 1e4)
    pos = torch.arange(T, dtype=torch.int32).cuda()

    def run():
        kc, vc, x = torch.zeros(shape).half().cuda(), torch.zeros(shape).half().cuda(), qkv.clone()
        q, k, v = (t.view(T, -1, D) for t in x.split([H * D, KV * D, KV * D], 1))
        kernels.kv_write_slots(k, v, kc, vc, slots, layout=layout)
        kernels.qkv_epilogue(q, k, v, pos, cos, sin, slots, kc, vc, bias=qkv[0].clone(),
                             layout=layout)
        return kc, vc, x
    (a, b), used = _both(monkeypatch, run)
    _same(a, b)
    assert used is (layout != "other" and slots_dtype != torch.int16)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 20, 257])
def test_topk_and_mlp(gpu, monkeypatch, k):
    x = _rand(3, 9000)

    def topk():
        idx = torch.full((3, k), -1, dtype=torch.int32, device="cuda")
        val = torch.zeros(3, k, dtype=x.dtype, device="cuda")
        kernels.topk_logits(x, k, indices=idx, values=val)
        return idx, val
    (a, b), used = _both(monkeypatch, topk)
    _same(a, b)
    assert used is (k <= 256)
    for H, I in ((2048, 256), (96, 128)):  # a split product; a refused width
        h, w = _rand(7, H), _rand(2 * I, H)
        o = torch.zeros(7, I, dtype=h.dtype, device="cuda")
        (a, b), used = _both(monkeypatch, lambda: kernels.gate_up_silu(h, w, out=o).clone())
        _same(a, b)
        assert used is (H % 64 == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[1], [40, 3, 0, 700], [5000, 20]])
@pytest.mark.parametrize("cache_dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("new", [1, 9])
def test_backend_steps(gpu, monkeypatch, lens, cache_dtype, new):
    """Decode-only and prefill-only steps of the backend, with a padded query
    buffer, and a query type that differs from the cache's."""
    H, KV, D = 8, 2, 64
    lens = [max(n, new) if new > 1 else n for n in lens]
    S, nblk = len(lens), [max(1, -(-n // 16)) for n in lens]
    perm = torch.randperm(sum(nblk) + 2, generator=torch.Generator().manual_seed(1))
    bt = torch.full((S, max(nblk)), -1, dtype=torch.int32)
    off = 0
    for s, n in enumerate(nblk):
        bt[s, :n] = perm[off:off + n]
        off += n
    n = S * new
    tok = torch.arange(S).repeat_interleave(new)
    pos = torch.tensor([max(0, L - new + i) for L in lens for i in range(new)])
    slots = (bt[tok, pos // 16].long() * 16 + pos % 16).cuda()
    cache = _rand(2, sum(nblk) + 2, 16, KV, D, dtype=cache_dtype)
    q, k, v = (_rand(n + 3, h, D, seed=h) for h in (H, KV, KV))
    qsl = torch.arange(0, n + 1, new, dtype=torch.int32)
    md = backend.HipAttentionMetadata(
        n, new, qsl.cuda(), max(lens), torch.tensor(lens, dtype=torch.int32).cuda(), bt.cuda(),
        slots, num_decode_tokens=n if new == 1 else 0, _query_start_loc_cpu=qsl.tolist(),
        _seq_lens_cpu=lens)
    impl = backend.HipAttentionImpl(H, D, 0.125, KV, None, None, "auto")

    def run():
        c, out = cache.clone(), torch.full((n + 3, H, D), 7.0, dtype=q.dtype, device="cuda")
        impl.forward(None, q, k, v, c, md, output=out)
        return c, out
    (a, b), used = _both(monkeypatch, run)
    _same(a, b)
    assert used


@pytest.mark.gpu
def test_decode_wrapper(gpu, monkeypatch):
    """The fused and plain decode, strided queries, an explicit workspace that
    is too small, tables of another type."""
    H, KV, D, S = 4, 2, 64, 3
    kc, vc = _rand(40, KV, 16, D), _rand(40, KV, 16, D, seed=1)
    bt = torch.arange(36, dtype=torch.int32).view(3, 12).cuda()
    sl = torch.tensor([150, 1, 190], dtype=torch.int32).cuda()
    q = _rand(S, 3 * H, D)[:, ::3]
    nk, nv = _rand(S, KV, D, seed=2), _rand(S, KV, D, seed=3)
    tiny = torch.empty(16, dtype=torch.uint8, device="cuda")
    for kw, native in (({}, True), ({"partition_size": 128}, True), ({"partition_size": -1}, True),
                       ({"partition_size": 128, "workspace": tiny}, False),
                       ({"partition_size": 100}, False), ({"layout": "x"}, False)):
        for table in (bt, bt.long()):
            for new in (False, True):
                def run(kw=kw, table=table, new=new):
                    k2, v2 = kc.clone(), vc.clone()
                    o = torch.zeros(S, H, D, dtype=q.dtype, device="cuda")
                    kernels.paged_decode(q, k2, v2, table, sl, scale=0.125, max_seq_len=190,
                                         output=o, new_keys=nk if new else None,
                                         new_values=nv if new else None, **kw)
                    return o, k2, v2
                (a, b), used = _both(monkeypatch, run)
                _same(a, b)
                assert used is (native and table is bt), kw


@pytest.mark.gpu
def test_lazy_clones_are_not_written_through(gpu):
    """A lazy clone (torch._lazy_clone) shares its original's memory until one of
    the two is written: kernels that write a clone leave the original alone."""
    n, KV, D = 5, 2, 64
    x, w = _rand(n, D), _rand(D)
    base = torch.full((n, D), 7.0, dtype=x.dtype, device="cuda")
    out = torch._lazy_clone(base)
    assert torch._C._is_cow_tensor(out)
    kernels.rms_norm(x, w, 1e-5, out=out)
    _same(base, torch.full_like(base, 7.0))
    _same(out, kernels.rms_norm(x, w, 1e-5))
    cache = torch.zeros(2, 3, 16, KV, D, dtype=x.dtype, device="cuda")
    clone = torch._lazy_clone(cache)
    kv = _rand(n, KV, D)
    slots = torch.arange(n, device="cuda")
    kernels.kv_write_slots(kv, kv, clone[0], clone[1], slots, layout="vllm")
    torch.cuda.synchronize()
    assert not cache.any()
    _same(clone[:, 0, :n], kv.expand(2, n, KV, D))

"""The wrappers' native host path (csrc/host_calls.cpp): on the GPU, every form
of call gives the same bits and the same errors with it as without it; on the
CPU, it declines whatever is not a GPU tensor."""
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

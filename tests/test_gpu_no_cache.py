"""Encoder attention read in place from the caller's K/V (vaa_attention_no_cache)
against torch SDPA in fp32: sequence lengths around the 16-key group, the
64-key tile and the workgroup's token tile, empty sequences, more sequences
than are searched in LDS, packed QKV views, and the staged path that views the
kernels cannot read directly keep."""
import pytest
import torch
import torch.nn.functional as F

from helpers import CANARY, assert_close, assert_close_bf16, host

pytestmark = pytest.mark.gpu

CASES = [
    # lens, H, KV, D, dtype, causal
    ([1], 4, 4, 64, torch.float16, False),
    ([15, 16, 17, 0, 63, 64, 65], 12, 12, 64, torch.float16, False),
    ([127, 128, 129, 1], 8, 2, 128, torch.bfloat16, False),
    ([0, 33, 0, 200, 0], 6, 2, 96, torch.float16, True),
    ([300, 2, 31], 4, 2, 32, torch.float16, True),
    ([1, 2, 0, 3] * 300, 2, 2, 32, torch.float16, False),  # 1200 sequences
]


def reference(q, k, v, lens, causal, scale):
    ref = torch.zeros(q.shape)
    a = 0
    for n in lens:
        if n:
            qt, kt, vt = (t[a:a + n].float().transpose(0, 1) for t in (q, k, v))
            kt, vt = (t.repeat_interleave(q.shape[1] // k.shape[1], 0) for t in (kt, vt))
            ref[a:a + n] = F.scaled_dot_product_attention(qt, kt, vt, scale=scale,
                                                          is_causal=causal).transpose(0, 1)
        a += n
    return ref.numpy()


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("lens,H,KV,D,dtype,causal", CASES)
def test_in_place(gpu, lens, H, KV, D, dtype, causal, packed):
    from vllm_apple_amd.backend import AttentionType, HipAttentionImpl, HipAttentionMetadata
    from vllm_apple_amd import kernels

    g = torch.Generator().manual_seed(len(lens) + H)
    T, scale = sum(lens), D ** -0.5
    qkv = torch.randn(T, (H + 2 * KV) * D, generator=g).to(dtype)
    split = [H * D, KV * D, KV * D]
    ref = reference(*(t.reshape(T, -1, D) for t in qkv.split(split, 1)), lens, causal, scale)
    dev = qkv.cuda()
    q, k, v = (t.view(T, -1, D) if packed else t.reshape(T, -1, D).contiguous()
               for t in dev.split(split, 1))
    qsl = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    # Canary rows behind the output: nothing is written past the last token.
    buf = torch.full((T + 4, H, D), CANARY, dtype=torch.int16, device="cuda").view(dtype)
    calls = []
    inner = kernels.try_attention_no_cache
    kernels.try_attention_no_cache = lambda *a, **kw: (calls.append(inner(*a, **kw)), calls[-1])[1]
    try:
        impl = HipAttentionImpl(H, D, scale, KV, None, None, "auto",
                                attn_type=AttentionType.ENCODER_ONLY)
        md = HipAttentionMetadata(T, max(lens), qsl.cuda(), max(lens), None, None, None,
                                  _query_start_loc_cpu=qsl.tolist())
        impl._attention_no_cache(q, k, v, buf[:T], md, causal=causal)
    finally:
        kernels.try_attention_no_cache = inner
    torch.cuda.synchronize()
    assert calls == [True]
    check = assert_close if dtype == torch.float16 else assert_close_bf16
    check(host(buf[:T].float()), ref, what=f"lens={lens[:8]} packed={packed}")
    assert bool((buf[T:].view(torch.int16) == CANARY).all())


@pytest.mark.parametrize("why", ["unaligned", "overlap", "fewer_queries"])
def test_staged_path_kept(gpu, why):
    """K/V rows that are not 16-byte aligned, an output that shares memory with
    the keys, and fewer query rows than the sequences hold take the staged
    path, with the same results."""
    from vllm_apple_amd.backend import AttentionType, HipAttentionImpl, HipAttentionMetadata
    from vllm_apple_amd import kernels

    lens, H, D = [20, 50], 4, 64
    T, scale = sum(lens), D ** -0.5
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(T, H, D, generator=g).half() for _ in range(3))
    ref = reference(q, k, v, lens, False, scale)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    out, rows = torch.zeros_like(qd), T
    if why == "unaligned":
        base = torch.zeros(2, T * H * D + 8, dtype=torch.float16, device="cuda")
        for i, t in enumerate((kd, vd)):
            base[i, 1:1 + t.numel()] = t.reshape(-1)
        kd, vd = (base[i, 1:1 + T * H * D].view(T, H, D) for i in range(2))
    elif why == "overlap":
        out = kd
    else:
        rows = T - 1
    calls = []
    inner = kernels.try_attention_no_cache
    kernels.try_attention_no_cache = lambda *a, **kw: (calls.append(inner(*a, **kw)), calls[-1])[1]
    try:
        impl = HipAttentionImpl(H, D, scale, H, None, None, "auto",
                                attn_type=AttentionType.ENCODER_ONLY)
        qsl = [0, 20, 70]
        md = HipAttentionMetadata(T, 50, torch.tensor(qsl, dtype=torch.int32).cuda(), 50, None,
                                  None, None, _query_start_loc_cpu=qsl)
        impl._attention_no_cache(qd[:rows], kd, vd, out[:rows], md, causal=False)
    finally:
        kernels.try_attention_no_cache = inner
    torch.cuda.synchronize()
    assert True not in calls
    assert_close(host(out[:rows].float()), ref[:rows], what=why)

"""A prefill-only step in two launches (vaa_prefill_step) against the KV write,
index and prefill entry points in turn: the same bits of the cache and of every
row, with query tiles of one sequence each and of consecutive tokens, sequence
ends at the edges of the tiles, empty sequences, padded slots, K/V rows that are
not 16-byte aligned, no write, and more sequences than have tiles."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own", [0, 1])
@pytest.mark.parametrize("lens,prefix,H,KV,D", [
    ([1], 0, 8, 2, 64), ([31, 32, 33, 1, 64, 65], 5, 8, 2, 128), ([127, 128, 129, 0, 3], 0, 4, 4, 64),
    ([63, 0, 65, 64, 2], 40, 8, 4, 96), ([5, 200, 17], 100, 14, 2, 64), ([2] * 1100, 0, 4, 2, 32),
])
@pytest.mark.parametrize("write", ["aligned", "int32", "unaligned", "none"])
def test_step(gpu, lens, prefix, H, KV, D, own, write):
    from vllm_apple_amd import _lib, kernels

    S, T = len(lens), sum(lens)
    g = torch.Generator().manual_seed(T + H)
    total = [prefix + n if n else 0 for n in lens]
    nblk = [-(-n // 16) for n in total]
    bt = torch.full((S, max(nblk)), -1, dtype=torch.int32)
    perm = torch.randperm(sum(nblk) + 2, generator=g).int()
    off = 0
    for s, n in enumerate(nblk):
        bt[s, :n] = perm[off:off + n]
        off += n
    cache = torch.randn(2, sum(nblk) + 2, 16, KV, D, generator=g).half().cuda()
    q = torch.randn(T, H, D, generator=g).half().cuda()
    shift = 1 if write == "unaligned" else 0
    kv = torch.randn(2, T * KV * D + 8, generator=g).half().cuda()
    k, v = (kv[i, shift:shift + T * KV * D].view(T, KV, D) for i in range(2))
    qsl = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32).cuda()
    seq_lens = torch.tensor(total, dtype=torch.int32).cuda()
    bt = bt.cuda()
    tok, pos = kernels.build_token_index(qsl, seq_lens, T)
    slots = kernels.build_slot_mapping(bt, 16, tok, pos)
    slots[::7] = -1
    if write == "int32":
        slots = slots.int()
    ref_c, ref_o = cache.clone(), torch.full_like(q, 7.0)
    if write != "none":
        kernels.kv_write_slots(k, v, ref_c[0], ref_c[1], slots, layout="vllm")
    kernels.paged_prefill(q, ref_c[0], ref_c[1], bt, tok, pos, scale=0.1, layout="vllm",
                          output=ref_o)
    out = torch.full_like(q, 7.0)
    p = kernels.make_params(key_cache=cache[0], value_cache=cache[1], layout="vllm",
                            num_query_heads=H, scale=0.1, num_seqs=S,
                            max_blocks_per_seq=bt.shape[1], query=q, output=out, new_kv=k)
    n = _lib.load().vaa_prefill_step_workspace_size(ctypes.byref(p), T, S)
    ws = torch.full((n // 4 + 16,), -77, dtype=torch.int32, device="cuda")
    new = (k.data_ptr(), v.data_ptr(), slots.data_ptr()) if write != "none" else (None,) * 3
    _lib.call("vaa_prefill_step", ctypes.byref(p), q.data_ptr(), cache[0].data_ptr(),
              cache[1].data_ptr(), bt.data_ptr(), seq_lens.data_ptr(), qsl.data_ptr(), S, *new,
              _lib.VAA_INDEX_I32 if write == "int32" else _lib.VAA_INDEX_I64, out.data_ptr(), T,
              own, ws.data_ptr(), n, _lib.stream_handle())
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), ref_o.view(torch.int16))
    assert torch.equal(cache.view(torch.int16), ref_c.view(torch.int16))
    assert bool((ws[n // 4:] == -77).all()), "workspace overrun"


@pytest.mark.parametrize("split", [0, 64, 128])
@pytest.mark.parametrize("lens,H,KV,D", [
    ([33], 8, 2, 128), ([187, 1, 65, 0, 31], 32, 8, 128), ([127, 129, 3], 4, 4, 64),
    ([65, 63, 2], 8, 4, 96),
])
def test_tiles_behind_decodes(gpu, lens, H, KV, D, split):
    """The prefill of a mixed step's chunks over a tile table: the same bits as
    over consecutive tokens, the decodes' rows untouched."""
    from vllm_apple_amd import kernels

    nd, prefix = 5, 300
    new = [1] * nd + lens
    S, T = len(new), sum(new)
    g = torch.Generator().manual_seed(T)
    total = [prefix + 17 * i + n if n else 0 for i, n in enumerate(new)]
    nb = -(-max(total) // 16)
    bt = torch.randperm(S * nb, generator=g).int().view(S, nb).cuda()
    cache = torch.randn(2, S * nb, 16, KV, D, generator=g).half().cuda()
    q = torch.randn(T, H, D, generator=g).half().cuda()
    qsl = torch.tensor([0] + torch.tensor(new).cumsum(0).tolist(), dtype=torch.int32).cuda()
    sl = torch.tensor(total, dtype=torch.int32).cuda()
    tok, pos = kernels.build_token_index(qsl, sl, T)
    ref, out = torch.full_like(q, 7.0), torch.full_like(q, 7.0)
    kw = dict(scale=0.1, layout="vllm", split_keys=split, max_seq_len=max(total) if split else 0)
    kernels.paged_prefill(q[nd:], cache[0], cache[1], bt, tok[nd:], pos[nd:], output=ref[nd:], **kw)
    t, p, tiles = kernels.build_prefill_tiles(qsl[nd:], sl[nd:], nd, T - nd, H // KV)
    assert torch.equal(t + nd, tok[nd:]) and torch.equal(p, pos[nd:])
    per = kernels._prefill_tile_tokens(H // KV)
    want, at = [], 0
    for n in lens:
        want += [(at + i, min(per, n - i)) for i in range(0, n, per)]
        at += n
    want += [(0, 0)] * (tiles.shape[0] - len(want))
    assert [tuple(x) for x in tiles.tolist()] == want
    kernels.paged_prefill(q[nd:], cache[0], cache[1], bt[nd:], t, p, output=out[nd:], tiles=tiles,
                          **kw)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


def test_step_workspace_refused(gpu):
    from vllm_apple_amd import _lib

    p = _lib.VaaAttnParams()
    p.queries_per_kv = 4
    with pytest.raises(ValueError, match="workspace"):
        _lib.call("vaa_prefill_step", ctypes.byref(p), 16, 16, 16, 16, 16, 16, 2, None, None, None,
                  0, 16, 8, 1, None, 0, None)

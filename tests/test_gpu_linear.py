"""The plain product (vaa_linear) and the split gate/up product
(vaa_gate_up_silu_split) against fp64 products of the same 16-bit values:
token counts at the edges of the 32-token blocks, one to many splits with short
last splits, row strides that are and are not multiples of 4 KB (which walk
their steps from different starts), strided rows."""
import pytest
import torch

from helpers import assert_close, assert_close_bf16, host

import oracle.layer_ops as olo

pytestmark = pytest.mark.gpu


def _check(out, ref, dtype, what):
    if dtype == torch.float16:
        assert_close(host(out), ref, what=what)
    else:
        assert_close_bf16(out.cpu().double().numpy(), ref, what=what)


@pytest.mark.parametrize("T", [1, 31, 32, 33, 64, 65, 96, 97, 127, 128])
@pytest.mark.parametrize("K,N", [(64, 128), (1024, 256), (2048 + 64, 384), (8192, 128)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_linear_few_tokens(gpu, T, K, N, dtype):
    from vllm_apple_amd import kernels

    g = torch.Generator().manual_seed(T + K + N)
    x = torch.randn(T, K, generator=g).to(dtype)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(dtype)
    buf = torch.full((T + 1, N + 8), 7.0, dtype=dtype, device="cuda")
    out = buf[:T, :N]
    kernels.linear(x.cuda(), w.cuda(), out)
    torch.cuda.synchronize()
    _check(out, (x.double() @ w.double().T).numpy(), dtype, f"linear {T}x{K}x{N}")
    assert bool((buf[T:] == 7.0).all()) and bool((buf[:, N:] == 7.0).all()), "padding written"


@pytest.mark.parametrize("T", [129, 192, 193, 257, 384, 513, 1024])
@pytest.mark.parametrize("K,N", [(64, 256), (576, 512), (8192, 256), (2048, 2048)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_linear_wide(gpu, T, K, N, dtype):
    """Token counts at the edges of the 128-, 192- and 256-token tiles, one to
    many splits."""
    test_linear_few_tokens(gpu, T, K, N, dtype)


@pytest.mark.parametrize("T,I", [(300, 14336), (192, 14336), (384, 32768), (150, 38 * 128)])
def test_gate_up_silu_tile_heights(gpu, T, I):
    """Batches that pick 2, 3 and 4 token blocks per wave (by the columns), on
    rows and columns of the first, a middle and the last tiles."""
    from vllm_apple_amd import kernels

    H = 192
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, H, generator=g, device="cuda").half()
    w = (torch.randn(2 * I, H, generator=g, device="cuda") / H ** 0.5).half()
    out = kernels.gate_up_silu(x, w).double()
    gu = x.double() @ w.double().T
    ref = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
    assert bool(((out - ref).abs() <= 2e-3 + 1e-2 * ref.abs()).all())


@pytest.mark.parametrize("T", [1, 24, 33, 64, 100, 128])
@pytest.mark.parametrize("H,I", [(2048, 256), (1088, 128), (4096, 1024)])
def test_gate_up_silu_split(gpu, T, H, I):
    from vllm_apple_amd import _lib, kernels

    assert _lib.load().vaa_gate_up_silu_workspace_size(T, H, I) > 0
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g).half()
    w = (torch.randn(2 * I, H, generator=g) / H ** 0.5).half()
    out = kernels.gate_up_silu(x.cuda(), w.cuda())
    torch.cuda.synchronize()
    assert_close(host(out), olo.gate_up_silu(host(x), host(w)), what=f"gate_up {T}x{H}x{I}")


def test_linear_strided_rows_and_refusals(gpu):
    from vllm_apple_amd import kernels

    g = torch.Generator().manual_seed(4)
    xb = torch.randn(40, 576, generator=g).half()
    wb = (torch.randn(256, 640, generator=g) / 23).half()
    x, w = xb.cuda()[:, 64:576], wb.cuda()[:, 64:576]
    out = torch.empty(40, 256, dtype=torch.float16, device="cuda")
    kernels.linear(x, w, out)
    torch.cuda.synchronize()
    assert_close(host(out), (xb[:, 64:].double() @ wb[:, 64:576].double().T).numpy(), what="strided")
    z = torch.zeros(1025, 512, dtype=torch.float16, device="cuda")
    assert not kernels.linear_ok(z, w, torch.empty(1025, 256, dtype=z.dtype, device="cuda"))
    assert not kernels.linear_ok(z[:129], w[:128],
                                 torch.empty(129, 128, dtype=z.dtype, device="cuda"))
    assert not kernels.linear_ok(xb.cuda()[:, 1:513], w, out)      # unaligned rows
    assert not kernels.linear_ok(x, w[:200], out[:, :200])         # 200 columns
    assert not kernels.linear_ok(x.bfloat16(), w, out)             # two types
    with pytest.raises(ValueError):
        kernels.linear(x, w[:200], out[:, :200])


def test_split_products_on_a_stream_given_by_its_handle(gpu):
    """stream may be any object with the raw handle, as for the other wrappers,
    where the product needs scratch of that stream too."""
    from types import SimpleNamespace

    from vllm_apple_amd import kernels

    side = torch.cuda.Stream()
    by_handle = SimpleNamespace(cuda_stream=side.cuda_stream)
    x = (torch.arange(7 * 2048, device="cuda") % 13).view(7, 2048).half()
    w = (torch.arange(512 * 2048, device="cuda") % 7 / 2048).view(512, 2048).half()
    outs = []
    side.wait_stream(torch.cuda.current_stream())
    for s in (side, by_handle):
        act = torch.zeros(7, 256, dtype=x.dtype, device="cuda")
        lin = torch.zeros(7, 512, dtype=x.dtype, device="cuda")
        torch.cuda.synchronize()
        kernels.gate_up_silu(x, w, out=act, stream=s)
        kernels.linear(x, w, lin, stream=s)
        torch.cuda.synchronize()
        outs.append((act, lin))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert bool(outs[0][0].any()) and bool(outs[0][1].any())


@pytest.mark.parametrize("which", ["down_proj", "out"])
def test_mlp_refuses_gradients_as_the_library_product_does(gpu, which):
    """encode writes into a given buffer, which autograd cannot follow: a down
    projection or output that needs a gradient is refused while gradients are
    on, by the own product as by torch.matmul, and taken without them.  A
    forward-mode tangent goes to torch.matmul too, and the output's version
    moves either way."""
    import torch.autograd.forward_ad as fwd

    from vllm_apple_amd.engine import EngineMLP

    H, I, T = 256, 512, 5
    g = torch.Generator().manual_seed(3)
    x, w1, w2 = ((torch.randn(s, generator=g) * 0.1).half().cuda()
                 for s in ((T, H), (2 * I, H), (H, I)))
    out = torch.zeros(T, H, dtype=torch.float16, device="cuda")
    m = EngineMLP(None, H, I)
    m.set_weights(gate_up_proj=w1, down_proj=w2)
    m.encode(None, x, out, T)
    want, version = out.clone(), out._version
    m.encode(None, x, out, T)
    assert torch.equal(out, want) and out._version > version
    with fwd.dual_level():
        dual = fwd.make_dual(w2, torch.ones_like(w2))
        kinds = []
        m.set_weights(gate_up_proj=w1, down_proj=dual)
        act = torch.zeros(T, I, dtype=torch.float16, device="cuda")
        for call in (lambda: torch.matmul(act, dual.t(), out=out),
                     lambda: m.encode(None, x, out, T)):
            try:
                call()
                kinds.append(None)
            except Exception as e:  # noqa: BLE001
                kinds.append(type(e))
        assert kinds[0] == kinds[1]
    m.set_weights(gate_up_proj=w1, down_proj=w2)
    (w2 if which == "down_proj" else out).requires_grad_()
    with pytest.raises(RuntimeError, match="automatic differentiation"):
        m.encode(None, x, out, T)
    with torch.no_grad():
        m.encode(None, x, out, T)
    assert torch.equal(out.detach(), want)

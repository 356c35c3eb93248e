"""The small-batch matrix-core path (NWCWeight.linear_tokens, nwc_tokens): 2 to 64 BF16 tokens times a compressed matrix of
any layout and element type, every output rounded once, to nearest even, from a value within 1e-3 of the float64 product
on the decoded weights plus the fp32 summation bound (tests/helpers.py check_rne).  Shapes at the edges of its tiles: row
groups cut short, a last column block of one, eight or nine super-chunks, columns that make no whole 16-byte chunks, several
rounds of units per workgroup; token counts at the edges of 16, 32 and 64; streams in fixed slots, packed, and longer than
a slot (decoded from memory)."""
import pytest
import torch

from tests.helpers import bf16_matrix, check_rne, fp8_source

pytestmark = pytest.mark.gpu


def _weight(M, K, elem, layout, seed, heavy=False):
    from nwc_amd.nwc_torch import NWCWeight
    w = fp8_source(M, K, seed=seed) if elem == "fp8" else bf16_matrix(M, K, seed=seed, escapes=False)
    if heavy:                               # rows of one rare exponent each: escapes and exceptions throughout
        g = torch.Generator().manual_seed(seed)
        w[:24] = (torch.rand(24, K, generator=g) * 20 - 10).exp2().to(torch.bfloat16)
    return NWCWeight(w, device="cuda", elem=elem, layout=layout)


def _check(c, x, y, bias):
    wd = c.dequant().double()
    if c.scale is not None:
        wd = wd * c.scale.double()[:, None]
    ref = x.double() @ wd.t() + (0.0 if bias is None else bias.double())
    terms = x.double().abs() @ wd.abs().t()
    check_rne(y, ref.cpu().numpy(), (1e-3 * ref.abs() + 2.0 ** -20 * terms + 1e-6).cpu().numpy(), "tokens")


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("elem", ["bf16", "fp8"])
@pytest.mark.parametrize("M,K,T,with_bias", [
    (17, 48, 2, True),            # less than one column block; a row group of one row
    (1003, 1100, 16, False),      # ragged both ways, no whole 16-byte chunks of x
    (250, 768, 17, True),         # a last column block of eight super-chunks
    (250, 800, 33, False),        # of nine
    (4999, 3590, 11, True),       # of one, six columns wide
    (300, 520, 64, False),
    (20000, 512, 32, True),       # several rounds of row groups per workgroup
])
def test_tokens_match_float64(cuda, layout, elem, M, K, T, with_bias):
    print(f"tokens layout {layout} {elem} {M}x{K} T={T}", flush=True)
    c = _weight(M, K, elem, layout, seed=M + K + T)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, K, generator=g).to(torch.bfloat16).cuda()
    b = torch.randn(M, generator=g).to(torch.bfloat16).cuda() if with_bias else None
    y = c.linear_tokens(x, b)
    assert y.shape == (T, M) and y.dtype == torch.bfloat16
    _check(c, x, y, b)
    assert torch.equal(y, c.linear_tokens(x, b))                 # a fixed order of sums
    shifted = torch.empty(T * K + 1, dtype=torch.bfloat16, device="cuda")[1:].view(T, K)
    shifted.copy_(x)                                              # not 16-byte aligned
    assert torch.equal(y, c.linear_tokens(shifted, b))


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("slots", [True, False])
@pytest.mark.parametrize("K", [700, 1024])
def test_tokens_packed_and_long_streams(cuda, monkeypatch, layout, slots, K):
    """Packed streams, and blocks of escapes whose streams do not fit a slot next to ordinary ones."""
    import nwc_amd.nwc_torch as nt
    print(f"tokens streams layout {layout} slots {slots} K={K}", flush=True)
    monkeypatch.setattr(nt, "FIXED_SLOTS", slots)
    c = _weight(600, K, "bf16", layout, seed=K, heavy=not slots)
    x = torch.randn(9, K, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).cuda()
    _check(c, x, c.linear_tokens(x, None), None)


@pytest.mark.parametrize("layout", [0, 1, 2])
def test_nwclinear_routes(cuda, layout):
    """NWCLinear sends small batches of matrices of a million weights and more here, and keeps F.linear where a gradient
    to the input is wanted and for more tokens."""
    import nwc_amd.nwc_torch as nt
    print(f"tokens route layout {layout}", flush=True)
    M, K = 1024, 1040
    lin = nt.NWCLinear(w=_weight(M, K, "bf16", layout, seed=5), device="cuda")
    x = torch.randn(2, 10, K, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    assert torch.equal(lin(x), lin.w.linear_tokens(x.view(20, K), None).view(2, 10, M))
    few = x[0, :3]
    want = lin.w.linear_batch(few, None) if layout == 0 else lin.w.linear_tokens(few, None)
    assert torch.equal(lin(few), want)
    weight = lin.w.dequant()
    grad = x.clone().requires_grad_()
    y = lin(grad)
    assert torch.equal(y, torch.nn.functional.linear(x, weight))
    y.float().sum().backward()
    assert grad.grad.shape == x.shape
    many = torch.randn(65, K, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).cuda()
    assert torch.equal(lin(many), torch.nn.functional.linear(many, weight))


def test_tokens_replays(cuda):
    """A captured call replayed with the program's own work between the replays gives the eager bits."""
    print("tokens graph replays", flush=True)
    c = _weight(2560, 1536, "bf16", 0, seed=9)
    x = torch.randn(8, 1536, generator=torch.Generator().manual_seed(4)).to(torch.bfloat16).cuda()
    want = c.linear_tokens(x, None)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = c.linear_tokens(x, None)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        c.linear_tokens(x[:5].contiguous(), None)


def test_tokens_captured_without_an_index(cuda):
    """A matrix used with two tokens only so far has no row index; four tokens are still captured, by the batched kernel."""
    from nwc_amd.nwc_torch import NWCLinear
    print("tokens capture without a row index", flush=True)
    c = _weight(2560, 1536, "bf16", 0, seed=9)
    c._row_index = None
    lin = NWCLinear(w=c, device="cuda")
    x = torch.randn(4, 1536, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).cuda()
    lin(x[:2])
    want = c.linear_batch(x, None)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = lin(x)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)

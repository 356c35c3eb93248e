"""The encoder on the GPU (kern_encode.hip) against the host encoder, byte for byte: every stored tensor of a matrix placed
on the GPU equals that of the same matrix encoded on the host, for sources in host and GPU memory, contiguous or not, all
layouts and element types, shapes cut short in rows, columns and 16-byte pieces, rare symbols (escapes, exceptions), and
the host encoder's refusals."""
import pytest
import torch

from tests.helpers import bf16_matrix, fp8_source

pytestmark = pytest.mark.gpu


def _same(gpu, host):
    a, b = gpu.tensors(), host.tensors()
    assert a.keys() == b.keys() and gpu.bytes == host.bytes
    for name in a:
        assert a[name].dtype == b[name].dtype
        assert torch.equal(a[name].cpu().view(torch.uint8), b[name].cpu().view(torch.uint8)), name
    if gpu.layout <= 1:
        assert torch.equal(gpu.seq_table().cpu(), host.seq_table().cpu())


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("elem", ["bf16", "fp8"])
@pytest.mark.parametrize("M,K", [(24, 16), (40, 17), (7, 513), (300, 1000), (257, 1027), (33, 3597), (2560, 1536)])
def test_gpu_encoder_equals_host(cuda, layout, elem, M, K):
    from nwc_amd.nwc_torch import NWCWeight
    print(f"encode layout {layout} {elem} {M}x{K}", flush=True)
    w = fp8_source(M, K, seed=K) if elem == "fp8" else bf16_matrix(M, K, seed=K)
    host = NWCWeight(w, device="cpu", elem=elem, layout=layout)
    _same(NWCWeight(w, device="cuda", elem=elem, layout=layout), host)
    _same(NWCWeight(w.cuda(), device="cuda", elem=elem, layout=layout), host)
    wide = torch.zeros(M, K + 3, dtype=w.dtype, device="cuda")
    wide[:, 1:K + 1] = w
    _same(NWCWeight(wide[:, 1:K + 1], device="cuda", elem=elem, layout=layout), host)


@pytest.mark.parametrize("layout", [0, 1, 2])
def test_rare_symbols_and_given_fp8(cuda, layout):
    from nwc_amd.nwc_torch import NWCWeight, quantize_fp8
    print(f"encode rare layout {layout}", flush=True)
    g = torch.Generator().manual_seed(layout)
    w = bf16_matrix(200, 1100, seed=3, escapes=False)
    w[::9] = (torch.randn(23, 1100, generator=g) * (torch.rand(23, 1100, generator=g) * 12 - 6).exp()).to(torch.bfloat16)
    w[1, ::7], w[2, 5], w[3, 6], w[4, 7] = 0.0, float("inf"), float("nan"), -0.0
    _same(NWCWeight(w, device="cuda", layout=layout), NWCWeight(w, device="cpu", layout=layout))
    codes, scale = quantize_fp8(bf16_matrix(65, 700, seed=4, escapes=False))
    codes.view(torch.uint8)[5] = (torch.arange(700) % 127).to(torch.uint8)          # every finite code
    _same(NWCWeight(codes, device="cuda", elem="fp8", scale=scale, layout=layout),
          NWCWeight(codes, device="cpu", elem="fp8", scale=scale, layout=layout))


def test_refusals(cuda):
    """What the host encoder refuses, with its exceptions."""
    from nwc_amd.nwc_torch import NWCWeight
    print("encode refusals", flush=True)
    codes = torch.zeros(16, 64, dtype=torch.uint8)
    codes[3, 5] = 0x7F
    for device in ("cpu", "cuda"):
        with pytest.raises(ValueError, match="NaN"):
            NWCWeight(codes.view(torch.float8_e4m3fn), device=device, elem="fp8", scale=torch.ones(16))
        with pytest.raises(RuntimeError, match="-1"):            # filler streams past the encoder's capacity
            NWCWeight(bf16_matrix(300, 16, seed=1), device=device, layout=0)
        spread = torch.rand(16, 512, generator=torch.Generator().manual_seed(2)) * 200 - 100
        with pytest.raises(ValueError, match="255 exceptions"):
            w = torch.cat([spread.exp2().to(torch.bfloat16)] + [bf16_matrix(16, 512, seed=i, escapes=False) for i in range(40)])
            w[:16] = torch.tensor(1e30)                          # a symbol rarer than seven others in whole lanes
            w[16:600] = (2.0 ** (torch.arange(512) % 16 * 2 - 30.0)).to(torch.bfloat16)
            NWCWeight(w, device=device, layout=2)

"""The token path on activations that end inside a 16-byte piece: the kernels read K values and none past them.  NaN after
the last value must not reach the result, which stays the value of a zero-extended copy, within 1e-3 of float64 before
its rounding (tests/helpers.py check_rne).  K one past, one short of and inside the kernels' pieces of 8, 16 and 32 columns, in shapes
that take each launch plan: two to four half-waves a block, the split tail, several rounds, several items a half-wave,
rows of more than 32 column blocks, and the kernels without a row index."""
import pytest
import torch

from tests.helpers import bf16_matrix, check_rne, fp8_source, token_tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,elem,M,K,index", [
    *[(layout, elem, 300 if K > 64 else 24, K, True) for layout in (0, 1, 2) for elem in ("bf16", "fp8") for K in (16, 17, 31, 505, 1009, 1095)],
    (0, "bf16", 2560, 2055, True),        # one to two row groups per CU: the split tail
    (0, "bf16", 40000, 519, True),        # several rounds
    (0, "bf16", 24, 16901, True),         # 34 column blocks
    (0, "bf16", 700, 777, False),
    (1, "bf16", 500, 8201, True),         # more blocks than half-waves
    (1, "bf16", 9001, 333, True),
    (1, "bf16", 700, 777, False),
    (1, "fp8", 64, 16901, True),
    (2, "bf16", 9001, 3333, True),
    (2, "bf16", 24, 16901, True),
])
def test_nothing_past_the_last_activation(cuda, monkeypatch, layout, elem, M, K, index):
    import nwc_amd.nwc_torch as nt
    print(f"tail layout {layout} {elem} {M}x{K} index {index}", flush=True)
    monkeypatch.setattr(nt, "ROW_INDEX", index)
    w = fp8_source(M, K, seed=K) if elem == "fp8" else bf16_matrix(M, K, seed=K, escapes=False)
    c = nt.NWCWeight(w, device="cuda", elem=elem, layout=layout)
    held = torch.full((K + 64,), float("nan"), dtype=torch.bfloat16, device="cuda")
    held[:K] = torch.randn(K, generator=torch.Generator().manual_seed(K)).to(torch.bfloat16)
    x = held[:K]
    y = c.linear_bf16(x, None)
    padded = torch.zeros(K + 64, dtype=torch.bfloat16, device="cuda")
    padded[:K] = x
    assert torch.equal(y, c.linear_bf16(padded[:K], None))
    wd = c.dequant().double()
    if c.scale is not None:
        wd = wd * c.scale.double()[:, None]
    y64 = wd @ x.double()
    check_rne(y, y64.cpu().numpy(), token_tol(y64.cpu().numpy(), (wd.abs() @ x.double().abs()).cpu().numpy()))

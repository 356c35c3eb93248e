"""Which inputs may take a kernel called by address instead of F.linear (nwc_torch._plain; no GPU): ordinary tensors only.
An input that wants a gradient, is inside a functorch transform or a forward-mode level, under a dispatch mode, traced,
of a subclass, on another device, or under autocast to another type keeps F.linear."""
import torch
from torch.utils._python_dispatch import TorchDispatchMode


class _Sub(torch.Tensor):
    pass


class _Mode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_plain_inputs():
    from nwc_amd.nwc_torch import _plain
    x, cpu = torch.randn(3, 4).bfloat16(), torch.device("cpu")
    assert _plain(x, cpu) and _plain(x[1:], cpu)
    assert not _plain(x, torch.device("meta"))
    assert not _plain(x.as_subclass(_Sub), cpu)
    assert not _plain(x.clone().requires_grad_(), cpu)
    with torch.no_grad():
        assert _plain(x.clone().requires_grad_(), cpu)
    seen = []
    torch.vmap(lambda v: seen.append(_plain(v, cpu)) or v)(x)
    torch.func.jvp(lambda v: seen.append(_plain(v, cpu)) or v, (x,), (x,))
    with torch.autograd.forward_ad.dual_level():
        seen.append(_plain(x, cpu))
    with _Mode():
        seen.append(_plain(x, cpu))
    torch.jit.trace(lambda v: (seen.append(_plain(v, cpu)), v + 1)[1], x, check_trace=False)
    assert seen and not any(seen)

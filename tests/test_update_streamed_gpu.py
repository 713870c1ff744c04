"""The update of fp32 states beyond the last-level cache, which goes past it, against the same entries some at a time, which do not:
states and outputs to the bit, and the kernel by its name on both sides of the border."""
import pytest
import torch

from quamba_amd import ops
from tests import launched

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,P,N,lanes", [(57, 128, 64, 128, 8), (241, 61, 64, 64, 4), (55, 128, 64, 128, 8), (234, 61, 64, 64, 4)])
def test_streamed(dev, B, H, P, N, lanes):
    streamed = B * H * P * N * 4 >= 224 << 20
    assert abs(B * H * P * N * 4 / (224 << 20) - 1) < 0.03 and 20 * H * P * N * 4 < 224 << 20
    gen = torch.Generator(device=dev).manual_seed(B)
    ri = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device=dev, generator=gen)
    f = lambda *v: torch.tensor(v, device=dev)
    state, x, dt, z = torch.randn(B, H, P, N, device=dev, generator=gen), ri(B, H, P), ri(B, H), ri(B, H, P)
    Bq, Cq, A, D = ri(B, 1, N), ri(B, 1, N), ri(H).abs(), ri(H)
    bias = (torch.rand(H, device=dev, generator=gen) - 2).half()

    def run(st, b):
        n = st.shape[0]
        return ops.sscan_update(st, x[b], f(0.03), dt[b].unsqueeze(-1).expand(n, H, P), f(0.02), A.view(H, 1, 1).expand(H, P, N), f(0.01), None,
                                Bq[b], f(0.02), Cq[b], f(0.02), D.view(H, 1).expand(H, P), f(0.02), z[b], f(0.03), bias.view(H, 1).expand(H, P), None, True)

    many = state.clone()
    y, names = launched.kernels(lambda: run(many, slice(None)))
    kernel = f"ssm_update_kernel<{lanes}, true, true, false, true, "
    launched.expect(names, kernel + ("true>" if streamed else "false>"))
    assert not torch.equal(many, state)
    for b in range(0, B, 20):
        some = state[b:b + 20].clone()
        ys, names = launched.kernels(lambda: run(some, slice(b, b + 20)))
        launched.expect(names, kernel + "false>")
        assert torch.equal(some, many[b:b + 20]) and torch.equal(ys, y[b:b + 20])

"""The update of int8 states that walks several batch entries per workgroup (many entries) against the same entries one at a
time, which test_ssd_gpu.py holds to the oracle: states and outputs to the bit, entry counts that are no multiple of the walk's,
heads whose channels do not fill a workgroup."""
import pytest
import torch

from quamba_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,P,N,G,grouped", [(33, 64, 64, 128, 2, True), (70, 64, 48, 64, 1, False), (129, 16, 64, 128, 1, False), (1, 4, 20, 128, 1, False)])
def test_one_entry_at_a_time(dev, B, H, P, N, G, grouped):
    gen = torch.Generator(device=dev).manual_seed(B)
    ri = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device=dev, generator=gen)
    f = lambda *v: torch.tensor(v, device=dev)
    ranges = {}
    x_scale, B_s, C_s, st_s = f(0.03), f(0.02), f(0.02), f(0.05)
    if grouped:
        hr = (torch.arange(1, 5, dtype=torch.int32, device=dev) * (H // G // 4)).repeat(G, 1).contiguous()
        dr = (torch.arange(1, 5, dtype=torch.int32, device=dev) * (P // 4)).repeat(G, 4, 1).contiguous()
        ranges = dict(x_head_group_range=hr, x_dim_group_range=dr)
        x_scale = torch.rand(G, 4, 4, device=dev, generator=gen) * 0.02 + 0.02
        st_s = torch.rand(G, 4, 4, N, device=dev, generator=gen) * 0.02 + 0.03
        B_s, C_s = f(*[0.02] * G), f(*[0.03] * G)
    state, x, dt, z = ri(B, H, P, N), ri(B, H, P), ri(B, H), ri(B, H, P)
    Bq, Cq, A, D = ri(B, G, N), ri(B, G, N), ri(H).abs(), ri(H)
    bias = (torch.rand(H, device=dev, generator=gen) - 2).half()

    def run(st, b):
        n = st.shape[0]
        return ops.sscan_update(st, x[b], x_scale, dt[b].unsqueeze(-1).expand(n, H, P), f(0.02), A.view(H, 1, 1).expand(H, P, N), f(0.01), st_s,
                                Bq[b], B_s, Cq[b], C_s, D.view(H, 1).expand(H, P), f(0.02), z[b], f(0.03), bias.view(H, 1).expand(H, P), None, True, **ranges)

    many = state.clone()
    y = run(many, slice(None))
    assert int((many != state).sum()) > 0 and int(many.abs().max()) > 100
    for b in range(B):
        one = state[b:b + 1].clone()
        y1 = run(one, slice(b, b + 1))
        assert torch.equal(one[0], many[b]) and torch.equal(y1[0], y[b])

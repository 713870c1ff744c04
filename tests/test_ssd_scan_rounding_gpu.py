"""Which fp32 values of the SSD chunk scan are rounded, told apart by inputs with one term a sum: exp(-127) is zero in fp32, so that
nothing decays, and one step of the last chunk has a non-zero x, of code 1 and scale 1."""
import pytest
import torch

from quamba_amd import ops

pytestmark = pytest.mark.gpu


# a workgroup that walks the heads of a group, one per head, one that chains up the chunks' own sums; last chunks whole and ragged
@pytest.mark.parametrize("B,L,H,P,N,G,Q", [(16, 256, 128, 64, 128, 8, 256), (16, 700, 128, 64, 64, 8, 128), (32, 64, 128, 64, 128, 8, 64), (2, 256, 16, 64, 128, 2, 256),
                                           (1, 1280, 128, 64, 64, 8, 128), (1, 1024, 128, 64, 128, 8, 256), (1, 700, 128, 64, 64, 8, 128)])
def test_the_weight_on_the_diagonal_is_rounded_from_the_references_value(dev, B, L, H, P, N, G, Q):
    """((s_C s_B) (q_C . q_B) exp) dt (quamba/triton/quant_bmm_chunk.py:60-66, quant_chunk_scan.py:135-150), not (q_C . q_B) exp
    (s_C s_B dt): they differ in the last fp16 place where the first sits at a tie.  Compared over the rows that share a piece of
    32 steps with the non-zero one, where the decay is one exponential."""
    g = torch.Generator(device=dev).manual_seed(L + N)
    t0 = (L - 1) // Q * Q
    rows = differ = 0
    for turn in range(max(4, 60 // B)):
        x = torch.zeros(B, L, H, P, dtype=torch.int8, device=dev)
        q_B, q_C = (torch.randint(-128, 128, (B, L, G, N), dtype=torch.int8, device=dev, generator=g) for _ in range(2))
        dt = torch.rand(B, L, H, device=dev, generator=g) + 0.01
        one, (s_B, s_C) = torch.ones(1, device=dev), torch.rand(2, 1, device=dev, generator=g) * 0.02 + 0.01
        at = [t0 + 16 * ((turn + b) % ((L - t0 + 15) // 16)) for b in range(B)]
        for b in range(B):
            x[b, at[b]] = 1
        y = ops.ssd_chunk_scan_combined_fwd(x, one, dt, None, torch.full((H,), -127, dtype=torch.int8, device=dev), one, q_B, s_B, q_C, s_C, one, Q)[0]
        for b, k in enumerate(at):
            m = slice(k, min(t0 + (k - t0) // 32 * 32 + 32, L))
            cb = (q_C[b, m].double() * q_B[b, k].double()).sum(-1).float().repeat_interleave(H // G, 1)          # exact
            want = (((s_C * s_B) * cb) * dt[b, k]).half()
            rows += want.numel()
            differ += int((want != (cb * ((s_C * s_B) * dt[b, k])).half()).sum())
            assert torch.equal(y[b, m], want[:, :, None].expand(-1, -1, P))
    assert differ >= 2, (rows, "these inputs tell the two orders apart")


# (as above; without a term of the scan, and with skip weights per head and per channel)
@pytest.mark.parametrize("B,L,H,P,N,G,Q", [(4, 1100, 32, 64, 128, 1, 256), (2, 256, 16, 64, 128, 2, 256), (1, 700, 128, 64, 64, 8, 128), (2, 300, 8, 32, 128, 2, 256)])
@pytest.mark.parametrize("per_channel", [False, True])
def test_the_skip_term_is_rounded_as_the_reference_rounds_it(dev, B, L, H, P, N, G, Q, per_channel):
    """(s_x q_x) (s_D q_D) (quamba/triton/quant_chunk_scan.py:153-163), not q_x (s_x (s_D q_D))."""
    g = torch.Generator(device=dev).manual_seed(H)
    codes = torch.arange(-128, 128, device=dev).float()
    for _ in range(4):
        while True:                                               # scales that tell the two orders apart, and at which skip weights
            s_x, s_D = torch.rand(2, 1, device=dev, generator=g) * 0.02 + 0.01
            tells = (((s_x * codes[:, None]) * (s_D * codes)).half() != (codes[:, None] * (s_x * (s_D * codes))).half()).any(0).nonzero()[:, 0]
            if tells.numel():
                break
        x, q_B = (torch.randint(-128, 128, s, dtype=torch.int8, device=dev, generator=g) for s in ((B, L, H, P), (B, L, G, N)))
        q_D = tells[torch.randint(tells.numel(), (H, P) if per_channel else (H,), device=dev, generator=g)].sub(128).to(torch.int8)
        one = torch.ones(1, device=dev)
        y = ops.ssd_chunk_scan_combined_fwd(x, s_x, torch.ones(B, L, H, device=dev), None, torch.zeros(H, dtype=torch.int8, device=dev), one, q_B, one,
                                            torch.zeros_like(q_B), one, one, Q, q_D=q_D, D_scale=s_D)[0]
        D = s_D * (q_D if per_channel else q_D[:, None]).float()
        want = ((s_x * x.float()) * D).half()
        assert torch.equal(y, want) and not torch.equal(want, (x.float() * (s_x * D)).half())

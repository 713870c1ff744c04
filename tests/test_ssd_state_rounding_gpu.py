"""Which fp32 value the B operand of the SSD state product is rounded to fp16 from: (s_B q) w, as the reference has it
(quamba/triton/quant_chunk_state.py:76-89), not q (s_B w), which differs in the last fp16 place where the first sits at a tie.
A is exp(-127), zero in fp32, and only the last step has a non-zero x, of code 1 and scale 1: its weight is exp(0) dt, the
product with B is the one term of the sum, and the final state is that operand."""
import numpy as np
import pytest
import torch

from quamba_amd import ops

pytestmark = pytest.mark.gpu


# one workgroup per (batch, head) that walks the chunks, a workgroup per chunk (few heads), the general kernels; last chunks
# whole and ragged
@pytest.mark.parametrize("B,L,H,P,N,G,Q", [(16, 256, 128, 64, 128, 8, 256), (16, 192, 128, 64, 64, 8, 128), (32, 64, 128, 64, 128, 8, 64), (16, 300, 128, 64, 128, 8, 256),
                                           (1, 1024, 128, 64, 128, 8, 256), (1, 700, 128, 64, 64, 8, 128),
                                           (16, 256, 128, 32, 128, 8, 256), (16, 100, 64, 64, 96, 8, 100)])
def test_the_operand_is_rounded_from_the_references_value(dev, B, L, H, P, N, G, Q):
    g = torch.Generator(device=dev).manual_seed(L + N)
    differ = 0
    for _ in range(4 if B > 1 else 40):
        x = torch.zeros(B, L, H, P, dtype=torch.int8, device=dev)
        x[:, -1] = 1
        q_B = torch.randint(-128, 128, (B, L, G, N), dtype=torch.int8, device=dev, generator=g)
        dt = torch.rand(B, L, H, device=dev, generator=g) + 0.01
        one, s_B = torch.ones(1, device=dev), torch.rand(1, device=dev, generator=g) * 0.05 + 0.01
        _, final = ops.ssd_chunk_scan_combined_fwd(x, one, dt, None, torch.full((H,), -127, dtype=torch.int8, device=dev), one, q_B, s_B, q_B, one, one, Q,
                                                   final_state_dtype=torch.float32)
        q, w = q_B[:, -1].float().repeat_interleave(H // G, 1), dt[:, -1, :, None]
        want = ((s_B * q) * w).half().float()
        differ += int((want != (q * (s_B * w)).half().float()).sum())
        assert torch.equal(final, want[:, :, None, :].expand(B, H, P, N))
    assert differ >= 2, "these inputs tell the two orders apart"

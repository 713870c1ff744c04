"""The SSD scan with a workgroup per chunk and head (few heads in flight) and with one that walks the chunks (many): one batch
entry at a time takes the first, all together the second, and the values are the same."""
import numpy as np
import pytest
import torch

from quamba_amd import ops, synth

pytestmark = pytest.mark.gpu


# every chunk length and state count, last chunks of 1, 88, 116 and 64 steps
@pytest.mark.parametrize("B,L,N,G,Q", [(5, 513, 128, 1, 256), (9, 600, 64, 2, 256), (5, 500, 128, 2, 128), (5, 1024, 128, 1, 64)])
@pytest.mark.parametrize("final_dtype", [torch.float32, torch.int8])
def test_one_entry_at_a_time(dev, B, L, N, G, Q, final_dtype):
    d = synth.mamba2_ssd_inputs(B, L, 48, 64, N, G, seed=L)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    s = lambda v: torch.tensor(np.asarray(v, np.float32)).to(dev)
    grouped = d["head_range"] is not None
    state_scale = s(np.full((G, d["head_range"].shape[1], d["dim_range"].shape[2], N), 0.02) if grouped else 0.02)

    def run(sel):
        return ops.ssd_chunk_scan_combined_fwd(
            t(d["x"][sel]), s(d["x_scale"]), t(d["dt"][sel]), s(d["s_dt"]), t(d["A_log"]), s(d["s_A"]), t(d["B"][sel]), s(d["s_B"]),
            t(d["C"][sel]), s(d["s_C"]), state_scale, Q, q_D=t(d["D"]), D_scale=s(d["s_D"]), dt_bias=t(d["dt_bias"]), dt_softplus=True,
            x_head_group_range=t(d["head_range"]) if grouped else None, x_dim_group_range=t(d["dim_range"]) if grouped else None,
            final_state_dtype=final_dtype)

    y, final = run(slice(None))
    for b in range(B):
        y1, final1 = run(slice(b, b + 1))
        assert torch.equal(y1[0], y[b]) and torch.equal(final1[0], final[b])
    assert float(y.float().abs().max()) > 0.1


# the most chunks whose sums the scan chains up itself (8), and one more (the pass between the two); last chunks of 128 and 1 steps
@pytest.mark.parametrize("B,L,N,G,Q", [(5, 1024, 128, 1, 128), (5, 1025, 128, 2, 128), (5, 1025, 64, 1, 128), (5, 2050, 64, 1, 256)])
@pytest.mark.parametrize("final_dtype", [torch.float32, torch.int8])
def test_one_entry_at_a_time_eight_and_nine_chunks(dev, B, L, N, G, Q, final_dtype):
    test_one_entry_at_a_time(dev, B, L, N, G, Q, final_dtype)


# the step sizes by the chunks' own workgroups (an entry alone) and in a launch of their own (all together): 20 chunks, and one
@pytest.mark.parametrize("B,L,N,G,Q", [(2, 20 * 256 - 3, 128, 1, 256), (23, 256, 128, 1, 256), (23, 17, 64, 2, 64)])
@pytest.mark.parametrize("final_dtype", [torch.float32, torch.int8])
def test_one_entry_at_a_time_step_sizes(dev, B, L, N, G, Q, final_dtype):
    test_one_entry_at_a_time(dev, B, L, N, G, Q, final_dtype)


# with more heads in flight than the chip holds workgroups, a workgroup walks some heads of a (batch, chunk, group), the last one
# of a group fewer: every chunk length, heads of 64 and of 128 channels, with and without gate and skip weights per channel
@pytest.mark.parametrize("B,L,H,P,N,G,Q,per_channel", [(4, 1100, 27, 64, 128, 1, 256, False), (9, 300, 48, 64, 64, 3, 128, True),
                                                       (5, 500, 56, 64, 128, 2, 64, False), (16, 600, 13, 128, 128, 1, 256, True)])
def test_heads_walked_by_a_workgroup(dev, B, L, H, P, N, G, Q, per_channel):
    d = synth.mamba2_ssd_inputs(B, L, H, P, N, G, seed=H, with_z=per_channel)
    if per_channel:
        d["D"] = np.random.default_rng(1).integers(-128, 128, (H, P)).astype(np.int8)
    t = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    s = lambda v: None if v is None else torch.tensor(np.asarray(v, np.float32)).to(dev)

    def run(sel):
        return ops.ssd_chunk_scan_combined_fwd(
            t(d["x"][sel]), s(d["x_scale"]), t(d["dt"][sel]), s(d["s_dt"]), t(d["A_log"]), s(d["s_A"]), t(d["B"][sel]), s(d["s_B"]),
            t(d["C"][sel]), s(d["s_C"]), None, Q, q_D=t(d["D"]), D_scale=s(d["s_D"]), q_z=t(d["z"][sel]) if per_channel else None,
            z_scale=s(d["s_z"]), dt_bias=t(d["dt_bias"]), dt_softplus=True, final_state_dtype=torch.float32)[0]

    y = run(slice(None))
    for b in range(B):
        assert torch.equal(run(slice(b, b + 1))[0], y[b])
    assert float(y.float().abs().max()) > 0.1

"""qa_sscan_fwd on token-major inputs against the same scan on seqlen-major ones (which test_sscan_gpu.py holds to the
oracle): every lane mapping, channel counts that are no multiple of a workgroup's, tile remainders, segments."""
import ctypes as C

import pytest
import torch

from quamba_amd import _lib, ops
from tests import launched

pytestmark = pytest.mark.gpu


def _inputs(dev, batch, dim, seqlen, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    ri = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device=dev, generator=g)
    t = lambda v: torch.tensor([v], device=dev)
    d = dict(u=ri(batch, seqlen, dim), dt=ri(batch, seqlen, dim), z=ri(batch, seqlen, dim), bc=ri(batch, seqlen, 48), A=ri(dim, 16).abs(),
             D=ri(dim), db=ri(dim))
    s = dict(u=t(0.02), dt=t(0.03), A=t(0.02), B=t(0.02), C=t(0.02), D=t(0.01), db=t(0.03), z=t(0.03), st=t(0.05))
    return d, s


def _token_major(d, s, state_dtype, with_z, workspace_bytes, lanes=None, softplus=1, segments=0):
    batch, L, dim = d["u"].shape
    out = torch.empty((batch, L, dim), dtype=torch.float16, device=d["u"].device)
    state = torch.empty((batch, dim, 16), dtype=state_dtype, device=out.device)
    ws = torch.empty(max(workspace_bytes, 1), dtype=torch.uint8, device=out.device)
    p = _lib.QaSScanParams()
    p.batch, p.dim, p.seqlen, p.dstate, p.n_groups, p.delta_softplus, p.token_major = batch, dim, L, 16, 1, softplus, 1
    p.u_batch_stride = p.delta_batch_stride = p.z_batch_stride = p.out_batch_stride = L * dim
    p.u_l_stride = p.delta_l_stride = p.z_l_stride = p.out_l_stride = dim
    p.u_d_stride = p.delta_d_stride = p.z_d_stride = p.out_d_stride = 1
    p.B_batch_stride = p.C_batch_stride = L * 48
    p.B_l_stride = p.C_l_stride = 48
    p.B_dstate_stride = p.C_dstate_stride = 1
    p.A_d_stride, p.A_dstate_stride = 16, 1
    p.u, p.delta, p.A_log, p.D, p.delta_bias = (d[k].data_ptr() for k in ("u", "dt", "A", "D", "db"))
    p.B, p.C = d["bc"].data_ptr() + 8, d["bc"].data_ptr() + 24
    p.z = d["z"].data_ptr() if with_z else None
    for name, k in (("u", "u"), ("delta", "dt"), ("A", "A"), ("B", "B"), ("C", "C"), ("D", "D"), ("delta_bias", "db"), ("z", "z"), ("ssm_state", "st")):
        setattr(p, "scale_" + name, s[k].data_ptr())
    p.out = out.data_ptr()
    setattr(p, "last_state_i8" if state_dtype == torch.int8 else "last_state_f32", state.data_ptr())
    p.workspace, p.workspace_bytes = ws.data_ptr(), workspace_bytes
    p.mapping, p.segments = 0 if lanes is None else 0x40000000 | lanes << 20, segments
    _lib.check(_lib.lib().qa_sscan_fwd(C.byref(p), _lib.current_stream(out.device)), "sscan_fwd")
    return out, state


@pytest.mark.parametrize("batch,dim,seqlen,dtype,with_z,ws", [
    (1, 64, 1, torch.int8, True, 0), (2, 36, 31, torch.float32, True, 0), (3, 1036, 33, torch.int8, False, 0),      # few channels
    (32, 1280, 40, torch.float32, True, 0), (32, 1280, 65, torch.int8, False, 0),                                   # two kinds of workgroup
    (40, 1024, 40, torch.float32, True, 0), (40, 1024, 65, torch.int8, False, 0),                                   # four lanes
    (48, 1024, 37, torch.float32, True, 0), (48, 1028, 64, torch.int8, False, 0),
    (1, 512, 256, torch.float32, True, 1 << 22), (2, 1540, 515, torch.int8, True, 1 << 22), (1, 96, 2049, torch.float32, False, 1 << 22)])
def test_token_major(dev, batch, dim, seqlen, dtype, with_z, ws):
    # (lanes 16: the library's own choice of waves)
    _against_seqlen_major(dev, batch, dim, seqlen, dtype, with_z, [dict(lanes=n) for n in ((None,) if ws else (None, 4, 8, 16))], ws)


# cut into segments by name, whatever the library's rule would choose: two, a ragged last one, as many as there are tiles
@pytest.mark.parametrize("batch,dim,seqlen,dtype,with_z", [(1, 512, 256, torch.float32, True), (2, 1540, 515, torch.int8, True), (1, 96, 2049, torch.float32, False),
                                                           (2, 512, 1300, torch.float32, True), (5, 36, 97, torch.int8, False), (1, 5120, 700, torch.float32, True)])
def test_segments(dev, batch, dim, seqlen, dtype, with_z):
    ways = [dict(lanes=8, segments=n) for n in sorted({2, 3, 7, (seqlen + 31) // 32})]
    names = _against_seqlen_major(dev, batch, dim, seqlen, dtype, with_z, ways, 1 << 28)
    for ran in names:
        launched.expect(ran, "scan_tm_kernel<8, false, false, 0>", f"scan_tm_kernel<8, {'true' if with_z else 'false'}, true, 0>")


def _against_seqlen_major(dev, batch, dim, seqlen, dtype, with_z, ways, ws):
    d, s = _inputs(dev, batch, dim, seqlen, seed=dim + seqlen)
    rows = lambda a: a.transpose(1, 2).contiguous()
    B, Cm = rows(d["bc"][:, :, 8:24])[:, None], rows(d["bc"][:, :, 24:40])[:, None]
    want, st = ops.sscan_fwd(rows(d["u"]), s["u"], rows(d["dt"]), s["dt"], d["A"], s["A"], B, s["B"], Cm, s["C"], s["st"], d["D"], s["D"],
                             rows(d["z"]) if with_z else None, s["z"] if with_z else None, d["db"], s["db"], True, state_dtype=dtype)
    names = []
    for way in ways:
        (out, state), ran = launched.kernels(lambda: _token_major(d, s, dtype, with_z, ws, **way))
        names.append(ran)
        diff = (out.float() - want.float()).abs()
        assert bool((diff <= 1e-3 + 2e-3 * want.float().abs()).all())
        a, b = state.float(), st[:, :, 0].float()
        if dtype == torch.int8:
            assert float((a - b).abs().max()) <= 1
        else:
            assert float((a - b).abs().max()) <= 1e-4 * float(b.abs().max())
    return names

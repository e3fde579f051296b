"""The backward with q, k, v and their gradients in rows of projections (vig_gla_bidir_bwd_rows): bit for bit what vig_gla_bidir_bwd gives on head-major tensors,
at the edges of its tiles, with sequences beyond the matrix-core kernel's gate range too, and nothing written between the columns."""
import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Dk", [32, 64])
@pytest.mark.parametrize("B,H,L", [(1, 1, 1), (2, 3, 33), (3, 2, 64), (2, 3, 65), (2, 3, 96), (5, 2, 128), (2, 3, 129), (100, 6, 196), (3, 3, 224), (2, 2, 225), (2, 3, 256)])
def test_bit_for_bit(B, H, L, Dk):
    announce(f"bwd rows B{B} H{H} L{L} Dk{Dk}")
    lib, g = _lib.load(), torch.Generator().manual_seed(L)
    K, V = H * Dk, H * 64
    ld, dld = 2 * K + V + 24, 2 * K + V + 104
    bf = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    z, do = bf(B, L, ld), bf(B, H, L, 64)
    gates = -torch.rand(2, B, H, L, Dk, generator=g).cuda()
    gates[0, 0, 0] *= 40  # out of range there: the recurrent kernel's
    if B > 2:
        gates[1, 2, H - 1] *= 40
    gates = gates.bfloat16()
    q, k, v = (t.reshape(B, L, H, -1).transpose(1, 2).contiguous() for t in (z[..., :K], z[..., K:2 * K], z[..., 2 * K:2 * K + V]))
    need = lib.vig_gla_bidir_bwd_workspace_for(B, H, L, Dk, 64, 1, 1, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    st, tail = torch.cuda.current_stream().cuda_stream, (B, H, L, Dk, 64, Dk ** -0.5, 0.5, 1, 1)
    dq, dk, dv, dg = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), torch.empty_like(gates)
    p = lambda t, n=0: t.data_ptr() + 2 * n  # noqa: E731
    assert lib.vig_gla_bidir_bwd(p(q), p(k), p(v), p(gates[0]), p(gates[1]), p(do), p(dq), p(dk), p(dv), p(dg[0]), p(dg[1]), ws.data_ptr(), need, *tail, st) == 0
    dz, dg2 = torch.full((B, L, dld), 7.0, dtype=torch.bfloat16, device="cuda"), torch.empty_like(gates)
    ws.fill_(255)
    assert lib.vig_gla_bidir_bwd_rows(p(z), p(z, K), p(z, 2 * K), ld, p(gates[0]), p(gates[1]), p(do), p(dz), p(dz, K), p(dz, 2 * K), dld, p(dg2[0]), p(dg2[1]),
                                      ws.data_ptr(), need, *tail, st) == 0
    want = torch.cat([t.transpose(1, 2).reshape(B, L, -1) for t in (dq, dk, dv)], -1)
    assert torch.equal(dz[..., :2 * K + V], want) and torch.equal(dg2, dg) and (dz[..., 2 * K + V:] == 7).all()


def test_refused():
    announce("bwd rows: calls it refuses")
    lib = _lib.load()
    t = torch.zeros(1 << 16, dtype=torch.bfloat16, device="cuda")
    p, st = t.data_ptr(), torch.cuda.current_stream().cuda_stream

    def run(ld=256, dld=256, L=8, Dk=32, Dv=64, io=1, need=1 << 17, at=0, gb=p):
        return lib.vig_gla_bidir_bwd_rows(p + at, p, p, ld, p, gb, p, p, p, p, dld, p, p, p, need, 1, 2, L, Dk, Dv, 1.0, 1.0, io, 1, st)

    assert all(run(**a) == -95 for a in (dict(L=257), dict(Dk=16, Dv=32), dict(Dv=32), dict(io=0)))
    assert all(run(**a) == -22 for a in (dict(ld=120), dict(dld=120), dict(ld=257), dict(dld=(1 << 20) + 8), dict(at=2), dict(gb=None)))
    assert run(need=64) == -28

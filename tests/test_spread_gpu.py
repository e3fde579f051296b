"""Few sequences of the bf16 forward, a workgroup a query tile: tile edges, both key widths, gates made inside, inputs that leave the fp16
form's range in one tile, and the smallest size that goes to a workgroup a sequence, against the fp32 recurrence."""
import ctypes

import pytest
import torch

import vig_amd
from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


def _inputs(B, H, L, Dk, gen):
    r = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    q, k, v = r(B, H, L, Dk), r(B, H, L, Dk) * Dk ** -0.5, r(B, H, L, 64)
    g = torch.nn.functional.logsigmoid(r(2, B, H, L, Dk)) / 16
    return [t.bfloat16().cuda() for t in (q, k, v, g)]


def _run(fn, q, k, v, g):
    B, H, L, Dk = q.shape
    o, ws = torch.full_like(v, float("nan")), torch.empty(4 * v.numel() + 4096, device="cuda")  # (the recurrence parks its first direction's sums)
    rc = fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), o.data_ptr(), ws.data_ptr(), ws.numel() * 4, B, H, L, Dk, 64, Dk ** -0.5, 0.25,
            1, 1, torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.VIG_OK
    return o.float()


def _close(got, want):
    """bf16 outputs: the rounding of either side (2^-9 each), and operands and score tiles of 11-bit significands: 1e-3 of the rms."""
    rms = want.pow(2).mean().sqrt()
    assert torch.isfinite(got).all()
    assert ((got - want).abs() <= 2.0 ** -7 * want.abs() + 0.01 * rms).all(), ((got - want).abs() / rms).max()
    assert (got - want).norm() <= 4e-3 * want.norm()


@pytest.mark.parametrize("B,H,L,Dk", [(1, 1, 129, 32), (2, 3, 160, 64), (1, 3, 196, 32), (1, 2, 225, 64), (1, 3, 256, 32), (32, 1, 256, 64),
                                      (36, 1, 197, 64), (37, 1, 197, 32)])
def test_against_recurrence(B, H, L, Dk):
    announce(f"spread forward B{B} H{H} L{L} Dk{Dk}")
    lib, x = _lib.load(), _inputs(B, H, L, Dk, torch.Generator().manual_seed(L))
    got = _run(lib.vig_gla_bidir_fwd, *x)
    _close(got, _run(lib.vig_gla_bidir_fwd_exact, *x))
    assert torch.equal(got, _run(lib.vig_gla_bidir_fwd, *x))


@pytest.mark.parametrize("what,tile", [("gf", 0), ("gf", 3), ("gb", 2), ("gb", 6), ("q", 4), ("k", 1), ("v", 5), ("all", 0)])
@pytest.mark.parametrize("Dk", [32, 64])
def test_outside_the_range(what, tile, Dk):
    announce(f"spread forward, {what} of tile {tile} outside the fp16 form, Dk{Dk}")
    lib, (q, k, v, g) = _lib.load(), _inputs(1, 2, 197, Dk, torch.Generator().manual_seed(3))
    rows = slice(32 * tile, 32 * tile + 9)
    if what in ("gf", "gb"):
        g["gf gb".split().index(what)][:, 1, rows, 3] = -2.0
    elif what == "all":
        g.fill_(-1.0)
    else:
        {"q": q, "k": k, "v": v}[what][:, 1, rows] *= {"q": 300.0, "k": 300.0, "v": 30000.0}[what]
    got, want = _run(lib.vig_gla_bidir_fwd, q, k, v, g), _run(lib.vig_gla_bidir_fwd_exact, q, k, v, g)
    if what in ("q", "k", "v"):  # rows of their own magnitude
        rms = want.pow(2).mean(-1, keepdim=True).sqrt()
        assert ((got - want).abs() <= 0.02 * rms + 2.0 ** -7 * want.abs()).all()
    else:
        _close(got, want)


@pytest.mark.parametrize("B,H,L", [(1, 3, 196), (2, 6, 129), (4, 1, 256)])
def test_gates_made_inside(B, H, L):
    """Against the same gates made by their own kernel and handed to the op."""
    announce(f"spread forward from low-rank gates B{B} H{H} L{L}")
    gen = torch.Generator().manual_seed(B)
    ld, K = H * 192 + 16, H * 32
    z = torch.randn(B, L, ld, generator=gen).bfloat16().cuda()
    up, bias = (torch.randn(2 * K, 16, generator=gen) / 4).bfloat16().cuda(), torch.randn(2 * K, generator=gen).bfloat16().cuda()
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    row = lambda n: (ctypes.c_longlong * 3)(L * ld, n, ld)  # noqa: E731
    o, g = torch.full((B, H, L, 64), float("nan"), dtype=z.dtype, device="cuda"), torch.empty(2, B, H, L, 32, dtype=z.dtype, device="cuda")
    p = z.data_ptr()
    assert lib.vig_gla_lowrank_fwd(p, p + 2 * K, p + 4 * K, p + 2 * H * 192, ld, up.data_ptr(), bias.data_ptr(), o.data_ptr(), None, 0, B, H, L, 32,
                                   64, row(32), row(32), row(64), 1 / 16, float("-inf"), 32 ** -0.5, 0.25, 1, st) == _lib.VIG_OK
    assert lib.vig_dirgate_lowrank_fwd(p + 2 * H * 192, ld, up.data_ptr(), bias.data_ptr(), g.data_ptr(), B, L, H, 32, 16, 1 / 16, float("-inf"), 1, 1,
                                       st) == _lib.VIG_OK
    q, k, v = (z[..., a:a + n].reshape(B, L, H, -1).transpose(1, 2).contiguous() for a, n in ((0, K), (K, K), (2 * K, 2 * K)))
    _close(o.float(), _run(lib.vig_gla_bidir_fwd_exact, q, k, v, g))
    assert torch.equal(o.float(), _run(lib.vig_gla_bidir_fwd, q, k, v, g))  # the same operands, one form


def test_one_sequence_in_a_batch():
    """A sequence's outputs as a workgroup a query tile gives them and as a workgroup a sequence does."""
    q, k, v, g = _inputs(1, 2, 196, 64, torch.Generator().manual_seed(9))
    one = vig_amd.batch_bid_fused_chunk_gla(q, k, v, g.flatten(0, 1))[0].float()
    many = [t.repeat(30, 1, 1, 1) for t in (q, k, v)]
    batch = vig_amd.batch_bid_fused_chunk_gla(*many, g.repeat_interleave(30, 1).flatten(0, 1))[0].float()
    assert torch.equal(batch[0], batch[29])
    _close(one[0], batch[0])


@pytest.mark.parametrize("L,Dk,keys", [(129, 32, 1.0), (160, 64, 1.0), (196, 32, 1.0), (197, 64, 1.0), (225, 32, 1.0), (256, 64, 1.0), (256, 32, 30.0), (196, 32, 1e-3),
                                       (196, 32, 1e-4), (256, 64, 3e-4)])
def test_one_sequence_among_sixty(L, Dk, keys):
    """A sequence's outputs as a workgroup a query tile gives them and as a workgroup a sequence does: the same bits, keys in fp16's subnormals
    once decayed among them."""
    announce(f"spread forward, one sequence and sixty L{L} Dk{Dk} keys x {keys}")
    q, k, v, g = _inputs(1, 2, L, Dk, torch.Generator().manual_seed(9))
    k = k * keys
    one = vig_amd.batch_bid_fused_chunk_gla(q, k, v, g.flatten(0, 1))[0]
    many = [t.repeat(30, 1, 1, 1) for t in (q, k, v)]
    batch = vig_amd.batch_bid_fused_chunk_gla(*many, g.repeat_interleave(30, 1).flatten(0, 1))[0]
    assert torch.equal(batch[0], batch[29]) and torch.equal(one[0], batch[0])


@pytest.mark.parametrize("L,Dk,over", [(129, 32, "v"), (196, 32, "v"), (256, 32, "v"), (196, 64, "q"), (197, 64, "k"), (256, 64, "v"), (225, 64, "gf"), (160, 64, "gb")])
def test_output_over_an_input(L, Dk, over):
    """A sequence's outputs written over one of its inputs, as a workgroup that has read the sequence may."""
    announce(f"few sequences, output over {over} L{L} Dk{Dk}")
    q, k, v, g = _inputs(1, 3, L, Dk, torch.Generator().manual_seed(L + 1))
    want = vig_amd.gla_bidir_forward(q, k, v, g[0], g[1])
    names = dict(q=q, k=k, v=v, gf=g[0].clone(), gb=g[1].clone())
    o = vig_amd.gla_bidir_forward(*names.values(), out=names[over])
    assert o.data_ptr() == names[over].data_ptr() and torch.equal(o, want)


@pytest.mark.parametrize("Dk", [32, 64])
def test_gated_output_over_the_values(Dk):
    announce(f"few sequences, gated output over v Dk{Dk}")
    gen = torch.Generator().manual_seed(Dk)
    (q, k, v, g), w = _inputs(2, 3, 196, Dk, gen), (torch.randn(192, 9, generator=gen) / 3).cuda()
    want = vig_amd.gla_bidir_locality_gate(q, k, v, g[0], g[1], w.view(-1, 1, 3, 3), (14, 14))
    rc = _lib.load().vig_gla_bidir_locgate_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), w.data_ptr(), v.data_ptr(), 2, 3, 196,
                                               Dk, 64, 14, 14, Dk ** -0.5, 1.0, 1, 1, torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.VIG_OK and torch.equal(v, want)


def test_output_over_the_rows_of_the_values():
    """One sequence whose values lie in wider rows, the output inside their span."""
    announce("one sequence, output over the values' rows")
    q, k, v, g = _inputs(1, 1, 196, 64, torch.Generator().manual_seed(5))
    want = vig_amd.gla_bidir_forward(q, k, v, g[0], g[1])
    rows = torch.cat([v[0, 0], v[0, 0]], 1).contiguous()
    s, sv = (ctypes.c_longlong * 3)(196 * 64, 196 * 64, 64), (ctypes.c_longlong * 3)(196 * 128, 64, 128)
    rc = _lib.load().vig_gla_bidir_fwd_strided(q.data_ptr(), k.data_ptr(), rows.data_ptr() + 128, g[0].data_ptr(), g[1].data_ptr(), rows.data_ptr(), 1, 1, 196, 64,
                                               64, s, s, sv, 0.125, 1.0, 1, 1, torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.VIG_OK and torch.equal(rows.view(-1)[:196 * 64].view(196, 64), want[0, 0])


@pytest.mark.parametrize("B,H,hw,Dk", [(1, 3, (14, 14), 32), (2, 2, (2, 126), 64), (1, 2, (256, 1), 32), (3, 1, (11, 12), 64)])
def test_locality_gate_behind_it(B, H, hw, Dk):
    announce(f"spread forward with the locality gate B{B} H{H} {hw} Dk{Dk}")
    gen = torch.Generator().manual_seed(hw[0])
    q, k, v, g = _inputs(B, H, hw[0] * hw[1], Dk, gen)
    w = (torch.randn(H * 64, 1, 3, 3, generator=gen) / 3).cuda()
    want = vig_amd.locality_gate(vig_amd.gla_bidir_forward(q, k, v, g[0], g[1]), w, hw)
    assert torch.equal(vig_amd.gla_bidir_locality_gate(q, k, v, g[0], g[1], w, hw), want)

"""The paged decode on small head groups (H no multiple of 128, or few queries
or positions): every head group (32, 64, 96) with and without splits, at tile and split edges, against
the oracle; calls on several streams and inside a graph.

Tolerance: max-abs 1e-2, the bf16 output's and the bf16 probabilities' rounding
at outputs of magnitude O(0.1) (as the other decode tests).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(amd, t, Q, H, S, page):
    qn, qp, cache, pt, lg, pps = t
    out = torch.empty((Q, H, 512), dtype=torch.int16, device="cuda")
    amd.dsa_decode_bf16_paged(qn, qp, cache, pt, lg, out, amd.dsa_config(Q, H, 512, 64, S, page, cache.shape[0]), pps)
    return out


SHAPES = [
    (1, 32, 1, 64),       # the smallest call
    (2, 32, 33, 64),      # a tile and one position
    (3, 64, 257, 512),    # 32-head groups, splits
    (2, 96, 300, 512),
    (1, 160, 1000, 2048),  # 5 groups of 32
    (1, 64, 4096, 8192),  # the largest selection, many splits
    (40, 64, 1024, 1024),  # 64-head groups, 6 splits
    (70, 96, 600, 1024),  # 96-head groups
    (300, 32, 64, 256),   # more groups than CUs, one split each
    (130, 64, 2050, 4096),  # one split of more than 2048 positions
    (130, 96, 3072, 4096), (130, 96, 3073, 4096), (131, 96, 4096, 4096),  # 96-head groups: rounds of 1536 positions
    (1, 128, 2048, 4096), (3, 256, 65, 256), (64, 128, 64, 256), (1, 384, 4096, 8192),  # H a multiple of 128
    (1, 128, 4097, 8192),  # past the small groups' positions: 128 heads
    (257, 32, 65, 128), (260, 32, 96, 128), (257, 32, 97, 128), (260, 32, 160, 192),  # two token groups from 4 tiles on
    (257, 32, 3072, 3072), (257, 32, 3073, 3136),  # their most positions, and past it
    (64, 96, 512, 1024), (32, 192, 512, 1024),
]


@pytest.mark.parametrize("Q,H,S,ctx", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_decode_head_groups(amd, orc, Q, H, S, ctx):
    import synth
    print("decode", Q, H, S, ctx, flush=True)
    page = 64
    t = synth.dsa_paged(Q, H, 512, 64, S, page, ctx, seed=Q + H + S)
    lg = t[4].cpu().numpy()
    lg[0, : S // 2] = -1  # a query with whole tiles invalid
    lg[-1, -1] = ctx
    t = t[:4] + (torch.from_numpy(lg).cuda(), t[5])
    out = _call(amd, t, Q, H, S, page)
    torch.cuda.synchronize()
    h = lambda v: v.cpu().numpy().view(np.uint16)
    qs = sorted({0, Q // 2, Q - 1})
    ref = orc.dsa_decode_bf16_paged(h(t[0][qs]), h(t[1][qs]), h(t[2]), t[3][qs].cpu().numpy(), lg[qs], 512, page)
    got = orc.bf16_to_f32(h(out[qs]))
    assert np.abs(got - ref).max() < 1e-2


def _sets(H, n=3):
    import synth
    Q, S, page = 3, 900, 64
    return Q, S, page, [synth.dsa_paged(Q, H, 512, 64, S, page, 1024, seed=s) for s in range(n)]


@pytest.mark.parametrize("n", [10, 280])
def test_decode_groups_streams(amd, n):
    """Calls in flight on several streams at once, up to more than there are
    scratch buffers, give the bits of a call alone."""
    import ctypes
    H = 64
    Q, S, page, sets = _sets(H)
    ref = [_call(amd, t, Q, H, S, page).cpu() for t in sets]
    lib = amd.load()
    raw = [ctypes.c_void_p() for _ in range(n)]
    for p in raw:
        assert lib.hipStreamCreateWithFlags(ctypes.byref(p), 1) == 0  # non-blocking
    streams = [torch.cuda.ExternalStream(p.value) for p in raw]
    outs = [torch.empty_like(ref[0], device="cuda") for _ in range(3 * n)]
    cfg = amd.dsa_config(Q, H, 512, 64, S, page, sets[0][2].shape[0])
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        t = sets[i % 3]
        amd.dsa_decode_bf16_paged(*t[:5], out, cfg, t[5], streams[i % n])
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        assert torch.equal(o.cpu(), ref[i % 3]), i
    for p in raw:
        assert lib.hipStreamDestroy(p) == 0


def test_decode_groups_in_turn(amd):
    """H a multiple of 128: calls of changing inputs and sizes one after the
    other on one stream, which share their scratch."""
    import synth
    shapes = [(3, 128, 900), (1, 128, 2048), (64, 128, 64), (2, 256, 513), (40, 128, 700)]
    ts = [(q, h, s, synth.dsa_paged(q, h, 512, 64, s, 64, 2048, seed=q + s)) for q, h, s in shapes]
    ref = []
    for q, h, s, t in ts:
        ref.append(_call(amd, t, q, h, s, 64).cpu())
        torch.cuda.synchronize()
    order = [0, 1, 0, 2, 1, 3, 4, 3, 0, 4, 2, 1]
    outs = [_call(amd, ts[i][3], *ts[i][:3], 64) for i in order]
    torch.cuda.synchronize()
    for i, o in zip(order, outs):
        assert torch.equal(o.cpu(), ref[i]), i


@pytest.mark.parametrize("H", [64, 128])
def test_decode_groups_graph(amd, H):
    """A captured call: H a multiple of 128 runs the eager call's plan, with the
    same bits; otherwise one split (no scratch), the same sums in another order."""
    Q, S, page, sets = _sets(H)
    ref = _call(amd, sets[0], Q, H, S, page).cpu()
    out = torch.empty_like(ref, device="cuda")
    cfg = amd.dsa_config(Q, H, 512, 64, S, page, sets[0][2].shape[0])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        amd.dsa_decode_bf16_paged(*sets[0][:5], out, cfg, sets[0][5])
    for _ in range(4):
        out.zero_()
        _call(amd, sets[1], Q, H, S, page)
        g.replay()
        torch.cuda.synchronize()
        if H % 128 == 0:
            assert torch.equal(out.cpu(), ref)
        d = (out.cpu().view(torch.bfloat16).float() - ref.view(torch.bfloat16).float()).abs().max()
        assert d < 1e-2

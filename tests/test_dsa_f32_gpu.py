"""The fp32 sparse attention's chunked kernels at the sizes where they change
form: chunk and tile edges, ragged head and column counts, unaligned rows, the
split and the one-launch form, calls on several streams and inside a graph.

Tolerance: the oracle sums sequentially in fp32; outputs are averages of
values in [-0.3, 0.3], and sums of n such terms in another order differ by a
few ulps of the partial sums, so 1e-6 (the reference cases' bar) holds.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(Q, H, Dc, Dp, S, N, seed):
    rng = np.random.default_rng(seed)
    u = lambda *s: rng.uniform(-0.3, 0.3, s).astype(np.float32)
    idx = np.stack([rng.choice(N, S, replace=S > N) for _ in range(Q)]).astype(np.int32)
    return u(Q, H, Dc), u(Q, H, Dp), u(N, Dc), u(N, Dp), u(N, Dc), idx


def _run(amd, t, shape):
    Q, H, Dc, Dp, S, N = shape
    out = torch.full((Q, H, Dc), float("nan"), device="cuda")
    amd.dsa_forward_f32(*t, out, amd.dsa_config(Q, H, Dc, Dp, S, 16, N))
    return out


SHAPES = [
    (1, 1, 1, 0, 1, 1),          # the smallest call
    (3, 2, 1, 0, 45, 64), (2, 3, 30, 6, 33, 64), (3, 2, 64, 16, 17, 64), (2, 2, 120, 4, 1, 8),  # a wave per row
    (5, 40, 32, 4, 8, 64), (2, 2, 320, 4, 3, 8), (3, 2, 1, 0, 70, 100), (3, 2, 64, 16, 60, 64),  # and chunks
    (256, 1, 32, 8, 129, 256), (300, 2, 31, 5, 300, 512), (600, 1, 100, 20, 1025, 2048),  # many rows
    (3, 5, 30, 6, 15, 40),       # unaligned rows, one partial tile
    (2, 16, 64, 16, 128, 300),   # the largest single chunk
    (2, 17, 100, 12, 129, 300),  # two head tiles, the first two-chunk row
    (1, 3, 516, 4, 1025, 2048),  # more than 8 blocks of 64 dims, chunk 48
    (2, 2, 7, 3, 2049, 4096),    # scalar loads, chunk 80
    (1, 20, 512, 64, 1000, 2048),
    (65, 64, 40, 8, 140, 256),   # 260 head tiles: the one-launch form
    (1, 2, 48, 8, 9000, 9500),   # chunks of 256
]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_dsa_f32_shapes(amd, orc, shape):
    print("dsa_f32", shape, flush=True)
    a = _inputs(*shape, seed=sum(shape))
    a[5][0, : shape[4] // 3] = -1  # invalid positions before, between and after valid ones
    a[5][-1, -1] = shape[5]
    out = _run(amd, [torch.from_numpy(x).cuda() for x in a], shape)
    torch.cuda.synchronize()
    for q in range(shape[0]):
        v = a[5][q][(a[5][q] >= 0) & (a[5][q] < shape[5])]
        if len(v) == 0:
            assert (out[q] == 0).all()
            continue
        ref = orc.dsa_forward_f32(a[0][q:q + 1], a[1][q:q + 1], a[2], a[3], a[4], v[None].astype(np.int32))
        assert np.abs(out[q].cpu().numpy() - ref[0]).max() < 1e-6


def test_dsa_f32_unaligned_base(amd, orc):
    """A cache that starts 4 bytes past a 16-byte boundary."""
    shape = (2, 4, 64, 16, 200, 512)
    a = _inputs(*shape, seed=9)
    t = [torch.from_numpy(x).cuda() for x in a]
    kc = torch.empty(t[2].numel() + 1, device="cuda")[1:].view_as(t[2])
    kc.copy_(t[2])
    ref = _run(amd, t, shape)
    t[2] = kc
    out = _run(amd, t, shape)
    torch.cuda.synchronize()
    assert (out - ref).abs().max() < 1e-6


def test_dsa_f32_streams_and_graph(amd):
    """Calls in flight on several streams at once and a captured call (which
    has no scratch and runs the one-launch form) give the same bits."""
    shape = (4, 8, 128, 32, 700, 2048)
    sets = [[torch.from_numpy(x).cuda() for x in _inputs(*shape, seed=s)] for s in range(4)]
    ref = [_run(amd, t, shape).cpu() for t in sets]
    streams = [torch.cuda.Stream() for _ in range(10)]
    torch.cuda.synchronize()
    outs = []
    for i in range(40):
        with torch.cuda.stream(streams[i % 10]):
            outs.append(_run(amd, sets[i % 4], shape))
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        assert torch.equal(o.cpu(), ref[i % 4]), i
    out = torch.empty_like(outs[0])
    cfg = amd.dsa_config(*shape[:5], 16, shape[5])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        amd.dsa_forward_f32(*sets[0], out, cfg)
    for i in range(4):
        out.zero_()
        _run(amd, sets[1], shape)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), ref[0])


@pytest.mark.parametrize("shape", [(1, 2, 64, 16, 100, 256), (2, 4, 64, 16, 300, 512), (1, 2, 7, 3, 1500, 2000),
                                   (65, 64, 40, 8, 140, 256)], ids=["chunk", "split", "split-scalar", "loop"])
def test_dsa_f32_largest_values(amd, orc, shape):
    """V near the largest float: the output is an average of its rows (the
    reference divides the probabilities before it sums), so it is finite.  5e-6
    of it: the probabilities' and the sums' rounding."""
    a = list(_inputs(*shape, seed=11))
    a[4] = (np.float32(3.3e38) * np.sign(a[4][:1]) * (1.0 - np.abs(a[4]) / 10)).astype(np.float32)
    ref = orc.dsa_forward_f32(*a)
    assert np.isfinite(ref).all()
    out = _run(amd, [torch.from_numpy(x).cuda() for x in a], shape).cpu().numpy()
    assert np.abs(out / ref - 1.0).max() < 5e-6


@pytest.mark.parametrize("shape,valid", [((1, 1, 8, 4, 5000, 5000), "all"), ((260, 1, 8, 4, 5000, 5000), "all"),
                                         ((260, 1, 8, 4, 5000, 5000), "tail"), ((260, 1, 8, 4, 5000, 5000), "sparse"),
                                         ((260, 1, 8, 4, 20000, 20000), "gaps"), ((2, 1, 8, 4, 20000, 20000), "gaps")],
                         ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_dsa_f32_long_lists(amd, orc, shape, valid):
    """Selections of many chunks (the windows' cursor): every position, only the
    last ones, one in 7, and lists with whole segments invalid."""
    Q, H, Dc, Dp, S, N = shape
    a = list(_inputs(*shape, seed=S + Q))
    a[5][:] = np.arange(S)[None]
    keep = np.zeros(S, bool)
    if valid == "all":
        keep[:] = True
    elif valid == "tail":
        keep[S - 700:] = True
    elif valid == "sparse":
        keep[3::7] = True
    else:
        keep[:64] = keep[S // 8 - 1: S // 8 + 70] = keep[S // 2: S // 2 + 3000] = keep[-1:] = True
    a[5][:, ~keep] = -1
    out = _run(amd, [torch.from_numpy(x).cuda() for x in a], shape).cpu().numpy()
    for q in sorted({0, Q // 2, Q - 1}):
        ref = orc.dsa_forward_f32(a[0][q:q + 1], a[1][q:q + 1], a[2], a[3], a[4], a[5][q:q + 1][:, keep])
        assert np.abs(out[q] - ref[0]).max() < 1e-6


@pytest.mark.parametrize("n", [12, 70])
def test_dsa_f32_many_streams(amd, n):
    """Streams in turn, up to more than there are scratch buffers: the same bits,
    and once each has had its first call none waits for the device."""
    import ctypes
    shape = (2, 8, 64, 16, 500, 1024)
    t = [torch.from_numpy(x).cuda() for x in _inputs(*shape, seed=4)]
    ref = _run(amd, t, shape).cpu()
    lib = amd.load()
    raw = []
    for _ in range(n):
        p = ctypes.c_void_p()
        assert lib.hipStreamCreateWithFlags(ctypes.byref(p), 1) == 0  # non-blocking
        raw.append(p)
    streams = [torch.cuda.ExternalStream(p.value) for p in raw]
    cfg = amd.dsa_config(*shape[:5], 16, shape[5])
    outs = [torch.empty_like(t[0]) for _ in streams]
    side, done = torch.cuda.Stream(), torch.cuda.Event()
    torch.cuda.synchronize()
    for turn in range(3):
        if turn == 1:  # every stream has had a call
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                torch.cuda._sleep(200_000_000)
                done.record()
        for s, out in zip(streams, outs):
            amd.dsa_forward_f32(*t, out, cfg, s)
    assert not done.query()
    torch.cuda.synchronize()
    for out in outs:
        assert torch.equal(out.cpu(), ref)
    for p in raw:
        assert lib.hipStreamDestroy(p) == 0


@pytest.mark.parametrize("S", [6, 60])
def test_dsa_f32_small_non_finite(amd, S):
    """The same rules in the kernel of the smallest calls and in the next one."""
    shape = (4, 2, 32, 4, S, 256)
    a = list(_inputs(*shape, seed=6))
    a[5][:] = np.arange(S) + 64 * np.arange(4)[:, None]
    a[2][:, 0] = np.abs(a[2][:, 0]) + 0.1
    a[2][2, 1] = np.nan       # one NaN score in query 0
    a[0][1, 0, 0] = np.inf    # every score of a head
    a[0][2, 1, 0] = -np.inf
    a[5][3, S - 2:] = [-1, 256]
    a[4][64 * 3 + S - 2:] = np.inf
    out = _run(amd, [torch.from_numpy(x).cuda() for x in a], shape).cpu()
    assert torch.isnan(out[0]).all()
    assert torch.isnan(out[1, 0]).all() and torch.isfinite(out[1, 1]).all()
    assert torch.isfinite(out[2, 0]).all() and (out[2, 1] == 0).all()
    assert torch.isfinite(out[3]).all()


def test_dsa_f32_non_finite(amd):
    """As in the reference's loops: a NaN or +inf score makes its head NaN, a
    head without a score above -inf (all -inf, or all NaN) gives 0; an infinity
    in a V row past the valid positions does not reach the sums."""
    shape = (5, 2, 64, 16, 300, 1024)
    a = list(_inputs(*shape, seed=3))
    a[5][:] = np.arange(300)
    a[5][1:] += 300
    a[5][4, :] += 300
    a[5][4, 250:] = -1
    a[2][:, 0] = np.abs(a[2][:, 0]) + 0.1
    a[2][5, 1] = np.nan       # one NaN score in query 0
    a[0][1, 0, 0] = np.inf    # every score of a head
    a[0][2, :, 0] = -np.inf
    a[0][3, 1, 0] = np.nan
    a[4][850:] = np.inf
    out = _run(amd, [torch.from_numpy(x).cuda() for x in a], shape).cpu()
    assert torch.isnan(out[0]).all()
    assert torch.isnan(out[1, 0]).all() and torch.isfinite(out[1, 1]).all()
    assert (out[2] == 0).all()
    assert torch.isfinite(out[3, 0]).all() and (out[3, 1] == 0).all()
    assert torch.isfinite(out[4]).all()

"""The fp32 gate for few experts (a lane per token) at the edges of its tiles:
indices and weights against the oracle, whose sums and order it reproduces
(indices exactly, weights within 2e-6: device expf against glibc's)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # T, E, K, D
    (1, 1, 1, 1), (3, 2, 1, 3), (64, 1, 1, 7), (65, 1, 1, 130), (5, 3, 4, 31), (21, 3, 3, 33),
    (11, 6, 2, 500), (10, 6, 2, 513), (16, 4, 2, 64), (13, 5, 4, 1030), (9, 7, 3, 2049),
    (4, 16, 4, 1000), (7, 31, 4, 129), (2, 32, 2, 1028), (33, 2, 2, 512), (40, 8, 2, 512),
    (40, 8, 4, 256), (9, 16, 3, 768),
    (6, 33, 4, 200), (6, 8, 5, 100),  # one past: the wave forms
    (70, 31, 4, 129), (33, 32, 2, 1028), (45, 7, 3, 2049), (130, 1, 1, 5), (200, 24, 4, 36), (129, 5, 1, 261),
    (1, 32, 2, 4096), (1, 6, 4, 1000), (2, 16, 4, 512), (1, 16, 2, 1024),  # a token or two
]


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16x"])
@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_gate_few_experts(amd, orc, shape, bf16):
    T, E, K, D = shape
    print("gate", shape, bf16, flush=True)
    r = np.random.default_rng(sum(shape))
    x = torch.from_numpy(r.standard_normal((T, D)).astype(np.float32))
    wg = (r.standard_normal((E, D)) / D ** 0.5).astype(np.float32)
    wg[E // 2] = wg[0]  # equal logits: ties go to the first
    if bf16:
        x = x.to(torch.bfloat16)
    xf = x.float().numpy()
    if T > 2:
        xf[1] = np.nan
        x[1] = float("nan")
    I = 1
    ridx, rw = orc.moe_forward_f32(xf, wg, np.zeros((E, 2 * I, D), np.float32), np.zeros((E, D, I), np.float32), K)[:2]
    idx = torch.full((T, K), -7, dtype=torch.int32, device="cuda")
    w = torch.full((T, K), -7.0, device="cuda")
    cfg = amd.moe_config(T, E, K, D, I)
    g = torch.from_numpy(wg).cuda()
    if bf16:
        amd.moe_gate_bf16x(x.view(torch.int16).cuda(), g, None, idx, w, cfg)
    else:
        amd.moe_gate_f32(x.cuda(), g, idx, w, cfg)
    torch.cuda.synchronize()
    assert np.array_equal(idx.cpu().numpy(), ridx)
    got = w.cpu().numpy()
    ok = ridx >= 0
    assert np.abs(got[ok] - rw[ok]).max(initial=0) < 2e-6
    assert np.array_equal(got[~ok], rw[~ok])

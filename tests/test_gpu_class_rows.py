"""A group whose class sums need several launches (more than 256 MiB of them): the
same bits as the requests alone, and a kernel time that covers every launch of
the group.  The allocation-free entry point, whose class sums take what its workspace
leaves: the same bits at few requests and at the most it takes."""
import numpy as np
import pytest

import ekgsim_amd as E
from ekgsim_amd import synth as S

pytestmark = pytest.mark.gpu


def _requests(n, L, B, s0):
    ks, ps = [], []
    for b in range(B):
        x = S.random_params(3, L, s0 + b)
        ks.append(S.layer_k_from_params(x, 3))
        ps.append(E.move_leads(S.lead_positions(n, L), S.displacements(x, 3, L)))
    return np.stack(ks), np.stack(ps)


def test_rows_in_several_launches():
    # 96^3, 16 leads: a row of class sums per request, about 3,800 lines of 128 B (0.49 MB)
    ctx = E.Context(0)
    n, L, B, T = 96, 16, 900, 24.0
    h = S.make_heart(n, seed=1)
    g = E.Heart(ctx, h.layer, h.seed)
    g.excite_delay(h.delay)
    k, p = _requests(n, L, 12, 40)
    k, p = np.resize(k, (B,) + k.shape[1:]), np.resize(p, (B,) + p.shape[1:])
    ctx.set_profiling(True)

    def timed(b):
        best = np.inf
        for _ in range(4):
            ctx.reset_profiling()
            out = g.simulate_batch(k[:b], p[:b], "3D4", 30.0, T, 1.0)
            groups, ms = ctx.kernel_time()
            assert groups == 1
            best = min(best, ms)
        return out, best

    whole, t_whole = timed(B)
    half, t_half = timed(B // 2)  # one launch
    print(f"{B} requests {t_whole:.3f} ms, {B // 2} requests {t_half:.3f} ms")
    assert np.array_equal(whole[:B // 2], half)
    for b in range(12):
        alone = g.simulate(k[b], p[b], "3D4", 30.0, T, 1.0)
        for q in range(b, B, 12):
            assert np.array_equal(whole[q], alone)
    assert t_whole >= 0.85 * 2 * t_half
    g.close()
    ctx.close()


def test_allocation_free_batches_up_to_the_limit():
    import torch
    ctx = E.Context(0)
    n, L, T = 128, 12, 600
    h = S.make_heart(n, seed=1)
    g = E.Heart(ctx, h.layer, h.seed)
    g.excite_delay(h.delay)
    g.layout_info("3D4")
    k8, p8 = _requests(n, L, 8, 90)
    for B in (1, 8, 440):  # 440: the most requests of this shape
        print(f"allocation-free batch of {B}", flush=True)
        k = torch.from_numpy(np.resize(k8, (B,) + k8.shape[1:])).cuda()
        p = torch.from_numpy(np.resize(p8, (B,) + p8.shape[1:])).cuda()
        ref = torch.zeros((B, L, T), dtype=torch.float64, device="cuda")
        got = torch.full((B, L, T), float("nan"), dtype=torch.float64, device="cuda")
        args = (B, 3, L, "3D4", 0.0, float(T), 1.0)
        g.simulate_batch_device(k.data_ptr(), p.data_ptr(), ref.data_ptr(), *args)
        ctx.synchronize()
        g.simulate_batch_device_noalloc(k.data_ptr(), p.data_ptr(), got.data_ptr(), *args)
        ctx.synchronize()
        assert torch.equal(got.view(torch.int64), ref.view(torch.int64))
    g.close()
    ctx.close()

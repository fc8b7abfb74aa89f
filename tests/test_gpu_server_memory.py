"""Device memory of server groups against what they are accounted as: a heart whose class
layout an excitation dropped (it is sized before the layout exists again), and budgets that held a
request before class sums were kept per region."""
import numpy as np
import pytest

import ekgsim_amd as E
from ekgsim_amd import synth as S

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def test_request_of_a_reexcited_heart_takes_what_is_accounted():
    import torch
    n, layers, L, T = 112, 24, 12, 40.0
    h = S.make_heart(n, seed=1, n_layers=layers)
    k = S.layer_k_from_params(S.random_params(layers, 1, 11), layers)
    pos = S.lead_positions(n, L)
    ecg, used, peak = [], [], []
    for reexcite in (False, False, True):  # the first run loads what a process loads once
        ctx = E.Context(0)
        g = E.Heart(ctx, h.layer, h.seed)
        g.excite_delay(h.delay)
        srv = E.Server(ctx, n_streams=1)
        hid = srv.add_heart(g)
        if reexcite:
            g.excite_delay(h.delay)  # the layout is built again inside the request
        ctx.synchronize()
        free = torch.cuda.mem_get_info(0)[0]
        ecg.append(srv.wait(srv.submit(hid, k, pos, "3D4", 20.0, T, 1.0))[0])
        used.append(free - torch.cuda.mem_get_info(0)[0])
        peak.append(srv.stats()["peak_bytes"])
        print(f"re-excited {reexcite}: {used[-1] / MIB:.1f} MiB taken, {peak[-1] / MIB:.1f} MiB accounted", flush=True)
        srv.close()
        g.close()
        ctx.close()
    assert np.array_equal(ecg[2], ecg[1])
    # the same buffers but for the class sums: what is accounted less is taken less (the
    # allocator rounds to 2 MiB)
    assert used[2] <= used[1] - (peak[1] - peak[2]) + 4 * MIB


# Bytes of one request of 200 steps on these hearts as they were accounted when a class took
# three sums per lead slot and piece of a window of classes: grid, leads, budget.
BUDGETS = [(24, 2, 88848), (24, 12, 240128), (24, 16, 314144), (48, 2, 95136), (48, 12, 258512), (48, 16, 338576),
           (96, 2, 105320), (96, 12, 287064), (96, 16, 376312)]


@pytest.mark.parametrize("n,leads,budget", BUDGETS)
def test_budget_that_held_a_request_still_does(n, leads, budget):
    ctx = E.Context(0)
    h = S.make_heart(n, seed=1)
    g = E.Heart(ctx, h.layer, h.seed)
    g.excite_delay(h.delay)
    k = S.layer_k_from_params(S.random_params(3, 1, 11), 3)
    pos = S.lead_positions(n, leads)
    ref = g.simulate(k, pos, "3D4", 0.0, 200.0, 1.0)
    srv = E.Server(ctx, hbm_budget_bytes=budget)
    hid = srv.add_heart(g)
    tickets = [srv.submit(hid, k, pos, "3D4", 0.0, 200.0, 1.0) for _ in range(3)]
    for t in tickets:
        assert np.array_equal(srv.wait(t)[0], ref)
    print(f"{n}^3, {leads} leads: budget {budget}, peak {srv.stats()['peak_bytes']}")
    assert srv.stats()["peak_bytes"] <= budget
    srv.close()
    # a budget too small for the request without its class sums is refused, as before
    srv = E.Server(ctx, hbm_budget_bytes=budget // 2)
    hid = srv.add_heart(g)
    with pytest.raises(E.EkgError) as e:
        srv.wait(srv.submit(hid, k, pos, "3D4", 0.0, 200.0, 1.0))
    assert e.value.code == 2  # EKG_ENOMEM
    srv.close()
    g.close()
    ctx.close()


def test_budget_that_held_a_request_with_one_class_still_does():
    ctx = E.Context(0)
    n, budget = 64, 9086976  # one small class among 363 chunks
    h = S.make_heart(n, seed=1)
    g = E.Heart(ctx, h.layer, h.seed)
    g.excite_transfer(S.layered_transfer(3, 5, diag=1.03, off=1.57))
    k = S.layer_k_from_params(S.random_params(3, 1, 11), 3)
    srv = E.Server(ctx, hbm_budget_bytes=budget)
    hid = srv.add_heart(g)
    srv.wait(srv.submit(hid, k, S.lead_positions(n, 12), "3D4", 0.0, 200.0, 1.0))
    assert srv.stats()["peak_bytes"] <= budget
    srv.close()
    g.close()
    ctx.close()

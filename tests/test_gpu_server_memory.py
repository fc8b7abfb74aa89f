"""Device memory of server groups against what they are accounted as: a heart whose class
layout an excitation dropped (it is sized before the layout exists again)."""
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

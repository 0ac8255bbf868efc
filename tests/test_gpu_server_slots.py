"""Slots a server gets by default: as many workgroups as the kernels' registers and
LDS let share a CU.  (The counts are this library's own figures for gfx950; a
kernel that takes a few registers more loses a half or a third of its slots.)"""
import pytest

import ddp_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("engine,heur,block,per_cu", [
    (ddp_amd.ENGINE_PILES, ddp_amd.H_EUCLID, 1024, 1), (ddp_amd.ENGINE_PILES, ddp_amd.H_EUCLID, 512, 2),
    (ddp_amd.ENGINE_PILES, ddp_amd.H_EUCLID, 256, 3), (ddp_amd.ENGINE_PILES, ddp_amd.H_ZERO, 512, 2),
    (ddp_amd.ENGINE_PILES, ddp_amd.H_ZERO, 256, 4), (ddp_amd.ENGINE_PILES, ddp_amd.H_ZERO, 128, 8),
    (ddp_amd.ENGINE_BIDI, ddp_amd.H_ZERO, 512, 2), (ddp_amd.ENGINE_BIDI, ddp_amd.H_MANHATTAN, 512, 2),
    (ddp_amd.ENGINE_BIDI, ddp_amd.H_EUCLID, 512, 1), (ddp_amd.ENGINE_HEAPS, ddp_amd.H_EUCLID, 256, 3),
    (ddp_amd.ENGINE_HEAPS, ddp_amd.H_EUCLID, 128, 4), (ddp_amd.ENGINE_HEAPS, ddp_amd.H_ZERO, 512, 1)])
def test_slots_per_cu(ctx, engine, heur, block, per_cu):
    if heur == ddp_amd.H_MANHATTAN:
        hg = ddp_amd.HostGraph.grid_maze(40, 40, 200, 1)
    else:
        hg = ddp_amd.HostGraph.geometric(1500, 8, 1000, 1)
    dg = ddp_amd.DeviceGraph(ctx, hg, reverse=True)
    if heur == ddp_amd.H_MANHATTAN:
        dg.set_grid(40)
    sv = ddp_amd.Server(ctx, dg, heur=heur, block=block, engine=engine, idle_ms=5)
    slots = sv.info()["slots"]
    sv.close()
    dg.close()
    print(engine, heur, block, slots, flush=True)
    assert slots >= per_cu * ctx.device_info()["compute_units"]

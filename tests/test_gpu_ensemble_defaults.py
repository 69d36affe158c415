"""Default tile shape of an ensemble: 32 x 8 points for sbp42 in FP64 where 32 x 16 tiles give more than 1450 blocks,
else 32 x 16.  The sizes lie on both sides of the line; on the upper one 32 members of C64, whose 898,560 stored
points take 164 us a step in 32 x 16 tiles and 151 us in 32 x 8."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ns,order,bits,rows", [
    ((64,) * 32, 42, 64, 8), ((64,) * 16, 42, 64, 8), ((32,) * 64, 42, 64, 8), ((144,) * 4, 42, 64, 16), ((96,) * 8, 42, 64, 16),
    ((32, 40, 48, 64), 42, 64, 16), ((64,) * 32, 42, 32, 16), ((64,) * 32, 43, 64, 16), ((64,) * 32, 63, 64, 16)])
def test_default_tile(Ns, order, bits, rows):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[ensemble default {len(Ns)} x {Ns[0]} {order} {bits}]", flush=True)
    ops = [swm.create_swm_operator(N, **swm.operator_names(order), precision=bits) for N in Ns]
    ens = swm.Ensemble(ops, [swm.create_stvec_swm(op) for op in ops])
    assert ens.get_tiling() == {"tile_cols": 32, "tile_rows": rows, "metric_on_the_fly": bits == 64, "blocks_per_slot": 0}

"""The form of the RK4 step that the benchmark prices is the one that the library runs.

Steps go by slopes where their four states, rows padded to multiples of 8 points, take more than 36 MB (64 MB for
FP32 and sbp63).  The sizes lie on either side of the line, some of them where the unpadded size lies on the
other.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,bits,N,slopes", [(42, 64, 247, False), (42, 64, 248, True), (42, 64, 249, True), (42, 64, 384, True),
                                                 (21, 64, 247, False), (21, 64, 248, True), (63, 64, 329, False),
                                                 (63, 64, 330, True), (42, 32, 463, False), (42, 32, 472, True)])
def test_bench_asks_the_library(order, bits, N, slopes):
    import bench
    import cubedsphere_sbp_swm_amd as swm
    print(f"[rk4 form {order} {bits} {N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names(order), precision=bits)
    assert bench.by_slopes(op) is slopes

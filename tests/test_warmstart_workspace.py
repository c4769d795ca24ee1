"""The warm-start network's workspace holds what its kernels write and no more per node: the
five activations, two gradients in turn and one product, 64 floats each."""
import pytest


@pytest.mark.parametrize("n", [1, 64, 65, 130_804, 8_388_608])
def test_floats_per_node(ND, n):
    blocks = min(1024, (n + 63) // 64)
    assert ND._abi.lib().nd_mp_workspace_floats(n) <= 8 * 64 * n + 64 * 256 + 8192 * (blocks + 2)

"""kernels.prefill_pieces where rows see no keys on average: causal attention of more rows than keys is not cut."""
import pytest

from omni_npu_amd import kernels as K


@pytest.mark.parametrize("seen", [-63, 0, 1])
def test_rows_without_keys_are_not_cut(seen):
    assert K.prefill_pieces(129, 2, 65, 3, seen) == 1

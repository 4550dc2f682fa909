"""kernels.prefill_pieces where there is nothing to cut: rows that see no keys on average (causal attention of more rows than keys), and no
rows at all.  The native host side's copy says the same."""
import pytest

from omni_npu_amd import _host, kernels as K


@pytest.mark.parametrize("seen", [-63, 0, 1])
def test_rows_without_keys_are_not_cut(seen):
    assert K.prefill_pieces(129, 2, 65, 3, seen) == 1


@pytest.mark.parametrize("max_q_len", [0, 1, 5, 300])
@pytest.mark.parametrize("batch", [0, 1, 3])
def test_no_rows_are_not_cut(batch, max_q_len):
    for rule in (K.prefill_pieces, _host.load().prefill_pieces):
        assert rule(0, batch, max_q_len, 16, 100) == 1

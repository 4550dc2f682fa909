"""The native host side shapes a prefill as the general path does (kernels.py has the rules and their reasons)."""
from omni_npu_amd import _host, kernels as K


def test_rules_are_those_of_the_general_path():
    ext = _host.load()
    assert ext.PREFILL_RULES == (K._PREFILL_RESIDENT, K._PREFILL_QUEUE_WORDS, K._PREFILL_LONG_KEYS)
    for tokens in (1, 2, 100, 127, 128, 129, 256, 700, 1017, 1024, 1100, 2048, 4095, 8192, 70000):
        for batch in (1, 2, 7, 64, 65):
            for heads in (1, 8, 16, 20, 32, 64, 128):
                assert ext.prefill_long_rows(tokens, batch, heads) == K._prefill_long_rows(tokens, batch, heads)
                for max_q in {1, min(tokens, 129), tokens}:
                    args = (tokens, batch, max_q, heads)
                    assert ext.prefill_blocks(*args) == K._prefill_blocks(*args), args
                    wants = batch <= 64 and heads % 8 == 0 and (K._prefill_blocks(*args) > K._PREFILL_RESIDENT or
                                                                 K._prefill_long_rows(tokens, batch, heads))
                    assert ext.prefill_wants_queue(*args) == wants, args
                    for seen in (0, 1, 64, 358, 5000, 30000, 10 ** 6):
                        assert ext.prefill_pieces(*args, seen) == K.prefill_pieces(*args, seen), (*args, seen)

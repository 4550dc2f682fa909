"""The split count of the sparse decode over row lists (kernels.list_splits), and its native copy."""
import math

from omni_npu_amd import kernels as K


def test_chunks_are_whole_passes_for_few_tokens_and_the_rule_by_length_for_many():
    from omni_npu_amd import _host
    ext = _host.load()
    for tokens in [*range(1, 70), 255, 256, 257, 1000]:
        for heads in (1, 16, 17, 32, 33, 64, 128):
            groups = tokens * math.ceil(heads / 32)
            for k in (1, 31, 32, 33, 512, 1000, 2048, 4096):
                s = K.list_splits(tokens, heads, k)
                assert s == ext.list_splits(tokens, heads, k) and s >= 1, (tokens, heads, k)
                if groups > 32:
                    assert s == K.launch_splits(tokens, 1, heads, k)
                    continue
                assert s * groups <= 256                       # no CU has two of them
                units = math.ceil(k / 32) + 8
                chunk = math.ceil(units / (256 // groups))
                assert s == math.ceil(units / (2 * math.ceil(chunk / 2)))

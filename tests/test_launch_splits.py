"""The split count of a decode launch (kernels.launch_splits): few rows and short contexts are cut into whole passes."""
import math

import torch

from omni_npu_amd import _lib, kernels as K


def test_chunks_are_whole_passes_where_cus_would_stand_idle_and_as_long_as_before_elsewhere():
    for batch in [*range(1, 70), 255, 256, 257, 1000]:
        for q_len, heads in ((1, 1), (1, 16), (2, 16), (1, 33), (1, 64), (1, 128), (2, 128)):
            groups = batch * math.ceil(q_len * heads / 32)
            for length in (1, 31, 32, 33, 512, 1000, 2048, 4096, 16384, 131072):
                s, base = K.launch_splits(batch, q_len, heads, length, full=True), K.default_num_splits(batch, q_len, heads, length)
                assert s >= 1
                if groups > 32 or base * groups > 256:
                    assert base <= s <= max(base, 256 // (4 * batch * math.ceil(q_len * heads / 128)))
                    continue
                assert s * groups <= 256                       # no CU has two of them
                units = math.ceil(length / 32) + 8
                assert s == math.ceil(units / (2 * math.ceil(math.ceil(units / (256 // groups)) / 2)))


def test_requests_that_may_be_shorter_keep_the_cut_by_length_where_they_would_go_through_more_passes():
    for batch, q_len, heads, length, by_length, passes in ((2, 2, 128, 2000, 16, 12), (5, 1, 128, 1495, 12, 10), (6, 1, 128, 486, 10, 6),
                                                           (3, 2, 128, 2000, 10, 9)):
        assert K.launch_splits(batch, q_len, heads, length) == by_length
        assert K.launch_splits(batch, q_len, heads, length, full=True) == passes
    # as many passes for them too, or more chunks than by length, or one sequence
    for args, splits in (((3, 1, 128, 2000), 18), ((8, 1, 32, 2000), 18), ((1, 2, 128, 2000), 18)):
        assert K.launch_splits(*args) == K.launch_splits(*args, full=True) == splits


def test_a_caller_s_workspace_for_the_cut_by_length_holds_what_is_launched():
    lib = _lib.load()
    for batch in (1, 2, 5, 12, 27, 64, 300):
        for q_len, heads in ((1, 16), (2, 16), (1, 32), (1, 128), (2, 128)):
            for length in (1, 300, 1495, 2048, 3300, 14000, 65536):
                for full in (False, True):
                    args = (batch, q_len, heads, length)
                    whole, by_length = K.launch_splits(*args, full=full), K._length_splits(*args)
                    need = [lib.mla_decode_workspace_bytes(batch, q_len, heads, s) for s in (whole, by_length)]
                    assert K._splits_within(lib, None, *args, full) == whole
                    assert K._splits_within(lib, torch.empty(max(need), dtype=torch.uint8, device="meta"), *args, full) == whole
                    small = K._splits_within(lib, torch.empty(need[1] // 2, dtype=torch.float16, device="meta"), *args, full)
                    assert small == min(whole, by_length)

"""The second look at the kernel of a forward launch (faster_rows): where the kernel that the modelled dispatch prefers was measured to be slower the
first choice stays, and where it is faster by far it is taken."""
import pytest

import lightron_amd as la


def _kernel(D, B, Hq, Hkv, rows, ranks, rank, layout, chunks=None):
    """Forward kernel of one rank of a ring, its chunks up to its last row (or the two halves of one step's chunk)."""
    if layout == "zigzag":
        h = rows // 2
        pos, split = (rank * h, (2 * ranks - 1 - rank) * h), h
        table = [i * h for i in (chunks or range(2 * ranks)) if i * h < pos[1] + h]
    else:
        h, split, pos = rows, None, rank * rows
        table = [i * h for i in range(rank + 1)]
    plan = la.attn_plan(B, Hq, Hkv, D, rows, [h] * len(table), table, pos, split, True)["fwd"]
    return plan["kernel"].replace("fwd_bf16_", "")


# us of the kernel named / of the one that the dispatch model prefers
@pytest.mark.parametrize("problem,kernel", [
    ((128, 8, 32, 32, 192, 16, 0, "zigzag"), "kernel<128, 1>"),                          # 99 / 170, four shares
    ((96, 8, 16, 16, 922, 16, 2, "zigzag"), "pad_kernel<128, 1>"),                       # 656 / 860, four shares
    ((96, 4, 12, 12, 2468, 16, 3, "zigzag"), "pad_kernel<128, 2>"),                      # 1427 / 1781, four shares
    ((64, 8, 32, 32, 1492, 2, 1, "contiguous"), "kernel<64, 1>"),                        # 262 / 336, 512 rows in pairs
    ((64, 1, 8, 8, 8152, 4, 1, "zigzag"), "shares_kernel<64, 2>"),                       # 435 / 474, four waves
    ((128, 8, 16, 16, 602, 8, 6, "zigzag"), "kernel<128, 1>"),                           # 121 / 145, four waves
    ((128, 4, 16, 4, 1284, 16, 4, "zigzag"), "kernel<128, 1>"),                          # 479 / 556, four waves, long blocks
    ((128, 8, 8, 8, 2126, 16, 7, "zigzag"), "kernel<128, 1>"),                           # 1306 / 1581, two shares
])
def test_the_first_choice_stays(problem, kernel):
    assert _kernel(*problem) == kernel


@pytest.mark.parametrize("problem,kernel", [
    ((128, 1, 32, 32, 1194, 8, 0, "zigzag"), "shares_kernel<128, 2>"),                   # 140 for 194 of four shares
    ((64, 8, 12, 12, 132, 4, 3, "contiguous"), "shares_kernel<64, 2>"),                  # 15 for 24 of four shares
    ((64, 2, 12, 12, 2498, 8, 0, "zigzag"), "shares_kernel<64, 4>"),                     # 239 for 340 of two shares
    ((64, 8, 32, 32, 558, 16, 2, "zigzag"), "w4_kernel<64>"),                            # 282 for 456 of 256 rows
    ((128, 4, 12, 12, 5066, 8, 0, "zigzag"), "w4_kernel<128>"),                          # 2583 for 4055 of 256 rows
])
def test_another_kernel_is_taken(problem, kernel):
    assert _kernel(*problem) == kernel

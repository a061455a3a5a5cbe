"""The attention's choice of a kernel, which needs no GPU."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hands-on-mlir_amd", "csrc")
WAYS = ("prefetch", "wide", "whole", "split")  # in the order of AttentionWay


def answers(tmp_path, expressions):
    """What these calls of attention_way.h return."""
    source, program = tmp_path / "ways.cpp", tmp_path / "ways"
    calls = "".join(f'printf("%d\\n", int(hom::{e}));' for e in expressions)
    source.write_text(f'#include "attention_way.h"\n#include <stdio.h>\nint main() {{ {calls} }}\n')
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(source), "-o", str(program)], check=True, timeout=60)
    out = subprocess.run([str(program)], capture_output=True, text=True, check=True, timeout=10).stdout.split()
    return list(map(int, out))


def ways(tmp_path, problems):
    """The way of each (batch, seq, heads, head size, fragment order) on a chip of 256 CUs."""
    return [WAYS[w] for w in answers(tmp_path, (f"attentionWay({b * h}, {s}, {d}, {int(packed)}, 256)"
                                                for b, s, h, d, packed in problems))]


# Sizes (batch, seq, heads) timed on an MI355X both ways with eight draws of lengths, uniform from a quarter of the
# sequence on; the other way took 5 % more at least in the mean, in fragment order 0.7 % of a request of six layers.
TIMED = {
    (64, False): {"split": [(4, 135, 16), (6, 223, 8), (2, 345, 16), (1, 706, 16), (5, 150, 16), (7, 307, 8), (4, 543, 12),
                            (11, 157, 16), (8, 294, 12), (3, 776, 16), (19, 132, 12), (16, 290, 8), (6, 300, 12)],
                  "whole": [(10, 150, 12), (7, 195, 16), (11, 193, 16), (26, 251, 8), (16, 380, 8), (5, 749, 12),
                            (30, 171, 8), (21, 228, 12), (11, 258, 16), (16, 442, 8)]},
    (128, False): {"split": [(8, 153, 8), (8, 220, 8), (4, 307, 8), (1, 706, 16), (10, 165, 8), (12, 147, 12), (12, 362, 8),
                             (6, 754, 8), (23, 159, 8), (9, 260, 16), (4, 656, 16)],
                   "whole": [(10, 150, 12), (15, 210, 8), (5, 329, 16), (3, 557, 12), (12, 198, 12), (24, 256, 8),
                             (5, 710, 12), (16, 185, 16), (21, 228, 12), (10, 304, 16), (13, 601, 8)]},
    (64, True): {"split": [(5, 256, 16), (5, 384, 16), (4, 450, 16), (6, 180, 16), (6, 220, 16), (15, 140, 12), (13, 165, 16),
                           (7, 400, 16), (19, 130, 12), (21, 130, 12)],
                 "whole": [(11, 200, 16), (12, 256, 12), (15, 200, 12), (16, 220, 12), (11, 384, 12), (8, 512, 12),
                           (6, 512, 16), (13, 270, 12), (14, 320, 12)]},
}


@pytest.mark.parametrize("d,packed", TIMED)
def test_attention_takes_the_faster_way(tmp_path, d, packed):
    want = [(size, way) for way, sizes in TIMED[d, packed].items() for size in sizes]
    got = ways(tmp_path, [(*size, d, packed) for size, _ in want])
    assert [(size, g) for (size, _), g in zip(want, got)] == want


# (batch, seq, heads) of split keys at head size 128 with all first query tiles first: 5 % faster or slower at least
@pytest.mark.parametrize("faster,sizes", [(True, [(3, 356, 16), (6, 335, 8), (2, 596, 16), (10, 203, 8), (1, 700, 12),
                                                  (7, 466, 12), (5, 522, 12), (11, 200, 12)]),
                                          (False, [(8, 620, 8), (4, 582, 16), (4, 575, 16), (4, 700, 12), (6, 384, 16)])])
def test_order_of_the_query_tiles(tmp_path, faster, sizes):
    assert answers(tmp_path, (f"attentionTilesOutside({b * h}, {-(-s // 64)})" for b, s, h in sizes)) == [faster] * len(sizes)


# (head size, seq) -> scores under the softmax: where both were timed, at the ends of the ranges
def test_lengths_with_scores_under_the_softmax(tmp_path):
    want = {(64, 129): 0, (64, 192): 0, (64, 193): 1, (64, 720): 1, (128, 64): 0, (128, 80): 1, (128, 720): 1, (256, 65): 0,
            (256, 192): 0, (256, 256): 1, (256, 720): 1}
    assert answers(tmp_path, (f"attentionOverlapsScores({d}, {s})" for d, s in want)) == list(want.values())


# Sizes (batch, seq, heads, head size, fragment order) that tests of the kernels use for each way
@pytest.mark.parametrize("way,sizes", [
    ("prefetch", [(3, 100, 4, 64, False), (5, 99, 16, 64, True)]),
    ("wide", [(44, 100, 12, 64, False), (48, 100, 11, 64, False), (44, 100, 12, 64, True), (48, 200, 2, 256, False)]),
    ("whole", [(30, 128, 12, 64, False), (24, 128, 12, 64, True), (40, 200, 8, 64, True), (48, 200, 2, 128, False),
               (13, 200, 11, 64, False), (13, 200, 5, 192, False)]),
    ("split", [(13, 160, 11, 64, False), (13, 160, 11, 128, False), (2, 300, 4, 64, True), (13, 200, 2, 128, False),
               (16, 100, 8, 192, False), (10, 192, 2, 256, False)])])
def test_sizes_that_stand_for_a_way(tmp_path, way, sizes):
    assert ways(tmp_path, sizes) == [way] * len(sizes)

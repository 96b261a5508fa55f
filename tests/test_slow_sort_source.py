"""The slow path's sort keeps its waves' counts as 16-bit words and clears two
with one store.  Nothing on a GPU shows whether the compiler may move that
store past the next round's reads, so the source itself is checked: the
clearing store has a type that may alias, and the wave synchronises between
it and the next round."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "llm-rs_amd", "csrc", "llmk_device.h")


def _sort_body():
    src = re.sub(r"//[^\n]*", "", open(SRC).read())
    at = src.index("void radix_sort_keys(")
    i = j = src.index("{", at)
    depth = 0
    while True:
        depth += {"{": 1, "}": -1}.get(src[j], 0)
        j += 1
        if depth == 0:
            return src[i:j]


def test_the_counts_are_cleared_through_a_type_that_may_alias():
    body = _sort_body()
    assert "(LDS uint32_t*)mine" not in body and "(LDS uint32_t*)wc" not in body
    typed = re.search(r"typedef uint32_t __attribute__\(\(may_alias\)\) (\w+);", body)
    assert typed
    assert re.search(r"LDS %s\* pairs = \(LDS %s\*\)mine;" % (typed[1], typed[1]), body)


def test_the_wave_synchronises_between_the_clear_and_the_next_round():
    body = _sort_body()
    clear = [m.end() for m in re.finditer(r"pairs\[[^\]]*\] = 0;", body)]
    assert len(clear) == 2  # before the histogram's barrier, and at a round's end
    assert re.match(r"\s*for \(.*?\) hist\[j\] = 0;\s*__syncthreads\(\);", body[clear[0]:])
    assert re.match(r"\s*WaveSync::sync\(\);\s*}", body[clear[1]:])

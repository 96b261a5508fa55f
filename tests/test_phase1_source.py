"""Phase 1's window 0 arrives as soon as its waves have published, whatever
the rest of its own walk takes: a walk in front of the arrival makes window 0
the last to arrive on some calls and not on others, depending on where the
code happens to lie, and those calls cost 2.8 us more.  The order is a matter
of the source, so it is checked there."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "llm-rs_amd", "csrc", "llmk_sampler.hip")


def _publish_to_walker():
    src = open(SRC).read()
    i = src.index("// ---- publish the segment: header, pairs, count, terms, runs")
    before = src[src.index("void xs_phase()"):i]
    return tuple(re.sub(r"//[^\n]*", "", s) for s in (before, src[i:src.index("// ---- the walker:")]))


def test_no_walk_before_the_segments_are_published():
    before, _ = _publish_to_walker()
    assert "runs_walk<" not in before and "xs_walk(" not in before


def test_window_0_counts_its_waves_before_it_walks():
    _, tail = _publish_to_walker()
    own = re.search(r"if \(own_walk\) \{(.*?)\} else \{\s*__syncthreads\(\);\s*\}\s*if \(tid == \(own_walk "
                    r"\? \(uint32_t\)\(NT - WAVE\) : 0u\)\)\s*sm\[70\] = __hip_atomic_fetch_add", tail, re.S)
    assert own, "the arrival follows the count, from a wave that does not walk"
    body = own[1]
    assert "__syncthreads" not in body
    count = body.index("__hip_atomic_fetch_add(&sm[73]")
    assert body.index("wait_stores();") < count < body.index("runs_walk<") < body.index("xs_walk(")
    # every wave adds to the count before any wave waits for it
    assert "if" not in body[:body.index("wait_stores();")]
    assert count < body.index("while (__hip_atomic_load(&sm[73]")

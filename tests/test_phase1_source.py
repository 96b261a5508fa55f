"""Phase 1's window 0 (of several) is never the workgroup that finishes the
row.  As the last window to arrive it would walk its own segments before it
could load anything, and whether it was the last hung on a few hundred
nanoseconds: calls cost 2.4 us more or not as their code happened to lie.
The order is a matter of the source, so it is checked there."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "llm-rs_amd", "csrc", "llmk_sampler.hip")


def _xs_phase():
    src = open(SRC).read()
    i = src.index("void xs_phase() {")
    return re.sub(r"//[^\n]*", "", src[i:src.index("\n}\n", i)])


def test_window_0_of_several_does_not_arrive():
    body = _xs_phase()
    own = body.index("if (own_walk) {")
    other = body.index("} else {", body.index("we = NW;", own))
    arrive = body.index("__hip_atomic_fetch_add(&w.xs_ctl[2 + j]")
    assert own < other < arrive < body.index("if (!sm[70]) return;")
    assert body.count("__hip_atomic_fetch_add(&w.xs_ctl[2 + j]") == 1
    assert "own_walk = k == 0 && nwin > 1;" in body
    assert "arrivals = nwin > 1 ? nwin - 1u : 1u;" in body
    # its walk publishes the sum the walker waits for, and it goes
    walk = body.index("xs_walk(")
    assert walk < body.index("__hip_atomic_store(own_sum + 1, tag", walk) < body.index("if (own_walk) return;")


def test_flags_and_sums_carry_the_calls_tag():
    """Nothing resets the windows' flags (window 0 may still be at work when
    the row is finished by other means), so they are told from those of an
    earlier call by the tag, and the entry point whose calls all have one
    tag clears them."""
    body = _xs_phase()
    assert "__hip_atomic_store(&wflag[k], tag, __ATOMIC_RELEASE" in body
    assert re.search(r"__hip_atomic_load\(&wflag\[i\], __ATOMIC_ACQUIRE, \w+\) == tag", body)
    src = open(SRC).read()
    clear = src[src.index("void static_clear_kernel("):]
    assert "xs_flag[i] = 0" in clear[:clear.index("\n}\n")]
    assert "ws.xs_wflag, XS_JOBS * ws.xs_maxw" in src

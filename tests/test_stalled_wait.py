"""A wait of the speculative kernel that passes its bound ends the launch with slots committed
but not yet booked: they are booked before the counters, the log and the controllers are
stored, so that these tell the state that the chain is in.

The bound (2^20 polls) is never reached in a sound run; this reads the order of the
launch's last statements."""
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "chromo_amd" / "csrc"


def test_committed_slots_are_booked_at_the_end():
    src = (CSRC / "chromo_spec.hpp").read_text()
    end = src[src.index("void spec_run("):]
    end = end[end.rindex("__syncthreads();"):]
    book = end.index("book_to<RING>(R, g, sctrl, sK, L, ctl->resolved)")
    assert book < end.index("R->ctrl[i] = sctrl[i]") and book < end.index("counters_store(")

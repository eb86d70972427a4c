"""Memory that a context's kernels read is not cleared on another stream: a
context's stream is non-blocking, so it does not wait for the null stream's
hipMemset, which may return before its work is done.  The allocations of
ctx_init are followed by copies that do wait; nothing follows the set-up of the
reciprocal sums."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "mdff_amd" / "csrc"


def test_scratch_is_cleared_on_the_contexts_stream():
    for name in ("mesh.hip", "recip.hip", "nlist.hip", "efg.hip", "realspace.hip"):
        src = (CSRC / name).read_text()
        assert not re.search(r"\bhipMemset\s*\(", src), name
        for call in re.findall(r"hipMemsetAsync\((.*)\)\)?;", src):
            assert call.split("//")[0].rstrip(")").endswith("c->stream"), (name, call)


def test_ctx_init_copies_after_its_last_clear():
    src = (CSRC / "mdff_gpu.hip").read_text()
    body = src[src.index("static int ctx_init("):]
    body = body[:body.index("\n}\n")]
    assert body.rindex("hipMemcpy(") > body.rindex("DMALLOC(")
    assert body.index("recip_setup(") > body.rindex("hipMemcpy(")

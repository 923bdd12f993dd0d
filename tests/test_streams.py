"""Every stream that a context owns is waited for before its buffers go
(csrc/s2g_api.hip).  Read from the source, so it runs without a GPU."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = open(os.path.join(ROOT, "sphtogrid.jl_amd", "csrc", "s2g_api.hip")).read()


def _body(head):
    b = SRC[SRC.index(head):]
    return b[:b.index("\n}")]


def test_destroy_waits_for_every_stream_before_it_frees():
    streams = re.findall(r"hipStream_t (\w+) = nullptr;", _body("struct s2g_ctx {"))
    assert {"stream", "side", "side2"} <= set(streams)
    body = _body("void s2g_destroy(s2g_ctx *c)")
    waits = body[:body.index(".release()")]
    for s in streams:
        assert f"hipStreamSynchronize(c->{s})" in waits, s
        assert f"hipStreamDestroy(c->{s})" in body, s


def test_forked_passes_wait_if_they_fail():
    """A pass that hands work to the side streams guards it from its fork on."""
    for head in ("void deposit2d_pass(", "void deposit3d_device("):
        body = _body(head)
        fork = body.index("hipEventRecord(c->fork, s)")
        assert -1 < body.find("ForkGuard forked{c, s};") < fork
        assert body.rindex("forked.joined = true;") > body.rindex("hipStreamSynchronize(s)") > fork
    guard = _body("struct ForkGuard {")
    assert all(q in guard for q in ("c->side,", "c->side2", "hipStreamSynchronize"))

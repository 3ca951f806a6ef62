"""CPU: the passes that a Net records, over a stand-in for the C ABI (fake_capi.cpp): replays are made where they should be, never of
what a pass could not do again, and never over a convolution that has been destroyed."""
import pytest

from test_net_units import run

NET = r"""
DEEPER = range(11, 21)  # layers behind the ones that a test is about: passes of fewer launches are not recorded
def deeper(g, last):
    for k in DEEPER: last = g.conv(k, last)
    return last
def deep(expr):
    for k in DEEPER: expr = "c%d(%s)" % (k, expr)
    return expr
def net():
    g = Graph()
    assert deeper(g, g.conv(2, g.conv(1, "data", True))) == OUT
    return g.ready()
OUT = "c%d" % DEEPER[-1]
def count(what): return fake.fake_count(what.encode())
def passes(s, want, n, replays):
    for _ in range(n):
        before = count("replay")
        s.run()
        assert fetched(s) == want, (fetched(s), want)
        assert count("replay") - before == replays
W = lambda v: (np.full((CH, CH, 1, 1), v, np.int8), None, np.full(CH, 50, np.float32), 20.0, 10.0)
"""


def test_passes_are_replayed_from_the_third_on(tmp_path):
    run(tmp_path, NET + r"""
g = net()
s = g.net.session("data", blob(), OUT)
passes(s, deep("c2(c1(x))"), 2, 0)
passes(s, deep("c2(c1(x))"), 4, 1)
assert count("record") == 1
for k in range(6):
    x = blob()
    x.reshape(-1)[:2].view(np.int64)[0] = fake.fake_number(b"y%d" % k)
    before = count("replay")
    assert expr_of(g.net.eval({"data": x}, OUT)) == deep("c2(c1(y%d))" % k)
    assert count("replay") - before == (k >= 3), k  # (the first asks for the size alone)
""")


def test_a_convolution_that_could_not_be_made_again_is_not_replayed(tmp_path):
    run(tmp_path, NET + r"""
g = net()
s = g.net.session("data", blob(), OUT)
for _ in range(4): s.run()
fake.fake_set(b"no_conv", 1)
try:
    g.net.set_conv("c1", *W(7))
    raise SystemExit("no error")
except hostnet.HostError:
    pass
for f in (s.run, lambda: g.net.eval({"data": blob()}, OUT)):
    for _ in range(4):
        try:
            f()
            raise SystemExit("a pass without its layer")
        except hostnet.HostError:
            pass
fake.fake_set(b"no_conv", 0)
g.net.set_conv("c1", *W(8))
passes(s, deep("c2(c8(x))"), 2, 0)
passes(s, deep("c2(c8(x))"), 3, 1)
assert count("dead") == 0
""")


def test_a_pipeline_that_the_program_builds_anew_is_recorded_anew(tmp_path):
    run(tmp_path, NET + r"""
g = net()
s = g.net.session("data", blob(), OUT)
for _ in range(4): s.run()
program = C.CDLL(sys.argv[2])
assert program.program_rebuild(g.net.h, b"c1") == 0
passes(s, deep("c2(c1(x))"), 2, 0)
passes(s, deep("c2(c1(x))"), 3, 1)
assert count("dead") == 0 and count("record") == 2
""", program=True)


@pytest.mark.parametrize("own_convolution", [0, 1])
def test_a_net_with_a_layer_of_the_program_is_not_recorded(tmp_path, own_convolution):
    run(tmp_path, NET + r"""
own = %d
program = C.CDLL(sys.argv[2])
Graph().net.close()  # (the library's layers are there)
program.program_register(own)
g = Graph()
out = deeper(g, g.conv(2, g.conv(1, "data", True)))
if not own: out = g.add("twice", "", type="Doubled", input=out)
g.ready()
s = g.net.session("data", blob(), out)
s.run()
want = fetched(s)
if own: assert want.startswith("sum(c20(sum(") and "c2(sum(c1(x),c1(x)))" in want
else: assert want == "sum(%%s,%%s)" %% ((deep("c2(c1(x))"),) * 2)
passes(s, want, 6, 0)
for k in range(6):
    x = blob()
    x.reshape(-1)[:2].view(np.int64)[0] = fake.fake_number(b"y%%d" %% k)
    assert expr_of(g.net.eval({"data": x}, out)) == want.replace("(x)", "(y%%d)" %% k), k
assert count("record") == 0
""" % own_convolution, program=True)


def test_passes_go_on_after_memory_ran_out_while_one_was_recorded(tmp_path):
    run(tmp_path, NET + r"""
g = net()
s = g.net.session("data", blob(), OUT)
passes(s, deep("c2(c1(x))"), 2, 0)
other = g.net.session("data", blob(), OUT)  # (its input takes the blob that the first pass has given back)
fake.fake_set(b"no_memory", 1)
try:
    s.run()
    raise SystemExit("a pass without its blobs")
except hostnet.HostError:
    pass
fake.fake_set(b"no_memory", 0)
assert hostnet.recording_counts() == (0, 0, 1)
passes(s, deep("c2(c1(x))"), 4, 0)
g.net.set_conv("c1", *W(5))  # (recorded again once the net has changed)
passes(s, deep("c2(c5(x))"), 2, 0)
passes(s, deep("c2(c5(x))"), 2, 1)
""")


def test_short_passes_are_recorded_only_where_the_host_waits(tmp_path):
    run(tmp_path, NET + r"""
g = Graph()
g.conv(4, g.conv(3, g.conv(2, g.conv(1, "data"))))
g.ready()
s = g.net.session("data", blob(), "c4")
passes(s, "c4(c3(c2(c1(x))))", 6, 0)
assert hostnet.recording_counts()[0] == 0
for k in range(6): assert expr_of(g.net.eval({"data": blob()}, "c4")) == "c4(c3(c2(c1(x))))"
assert hostnet.recording_counts()[0] == 1
""")

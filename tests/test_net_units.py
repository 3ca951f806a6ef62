"""CPU: the launches that a Net makes of several layers (pairs of pointwise layers, ShuffleNetV2 units, sums, blocks, pooled tails),
over a stand-in for the C ABI whose blobs hold the expression that they were computed from (fake_capi.cpp): whatever the forms of the
launches, in light mode or not, through a session or through eval, a pass gives the layers' own expression and runs every layer once."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

SCRIPT = r"""
import ctypes as C, sys
import numpy as np
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # (in front of the library that the host layer names)
fake.fake_number.restype = fake.fake_count.restype = C.c_long
fake.fake_expr.restype = C.c_char_p
from tensor_amd import hostnet

N, SIDE, CH = 1, 26, 88

class Graph:
    def __init__(self, light=True):
        self.net = hostnet.Net(lightmode=light)
        self.net.add_layer(type="Input", name="data", batchsize=N, channel=CH, height=SIDE, width=SIDE)
        self.expr, self.convs = {"data": "x"}, []
    def add(self, name, expr, **options):
        self.net.add_layer(name=name, **options)
        self.expr[name] = expr
        return name
    def conv(self, number, src, int8=False, dw=False):
        name = "c%d" % number
        opts = dict(kernel=3, padding=1, groups=CH, int8_scale_term=1) if dw else dict(kernel=1, int8_scale_term=2)
        opts["int8_scale_term"] += 100 if int8 else 0
        self.convs.append((number, dw))
        return self.add(name, "%s(%s)" % (name, self.expr[src]), type="Convolution", input=src, out_channels=CH, **opts)
    def sum(self, name, a, b):
        return self.add(name, "sum(%s,%s)" % tuple(sorted([self.expr[a], self.expr[b]])), type="Eltwise", input=a + "," + b)
    def shuffle(self, name, a, b):
        self.add(name + "_cat", "cat(%s,%s)" % (self.expr[a], self.expr[b]), type="Concat", input=a + "," + b)
        return self.add(name, "shuffle(%s)" % self.expr[name + "_cat"], type="ChannelShuffle", input=name + "_cat", groups=2)
    def halves(self, name, src):
        return [self.add(name + "_" + w, "half%d(%s)" % (k, self.expr[src]), type="Crop", input=src, start=k * CH, end=(k + 1) * CH)
                for k, w in enumerate(("lo", "hi"))]
    def mean(self, name, src):
        return self.add(name, "mean(%s)" % self.expr[src], type="GlobalAvgPool", input=src)
    def unit(self, name, other, branch):
        return self.halves(name, self.shuffle(name + "_sh", other, branch))
    def ready(self):
        self.net.compile()
        for number, dw in self.convs:
            w = np.full((CH, 1, 3, 3) if dw else (CH, CH, 1, 1), number, np.int8)
            self.net.set_conv("c%d" % number, w, None, np.full(CH, 50, np.float32), 20.0, 10.0)
        return self

def blob():
    x = np.zeros((N, CH, SIDE, SIDE), np.float32)
    x.reshape(-1)[:2].view(np.int64)[0] = fake.fake_number(b"x")
    return x
def expr_of(a):
    return fake.fake_expr(C.c_long(int(np.frombuffer(a.tobytes()[:8], np.int64)[0]))).decode()
def fetched(session):
    return expr_of(session.fetch((2 * N * CH * SIDE * SIDE,), np.float32))

def head(g):  # a unit's two halves
    return g.unit("u", g.conv(1, "data"), g.conv(3, g.conv(2, "data", True)))

# tails behind a unit: the blob that is asked for, and whether the unit's last layer and the next unit's first run as a pair
def sum_with_first_half(g):
    lo, hi = head(g)
    return g.sum("out", lo, g.conv(4, hi)), False
def sum_with_first_half_turned(g):
    lo, hi = head(g)
    return g.sum("out", g.conv(4, hi), lo), False
def sum_from_elsewhere(g):
    lo, hi = head(g)
    return g.sum("out", g.conv(5, lo), g.conv(4, hi)), False
def shuffle_again(g):
    lo, hi = head(g)
    return g.shuffle("out", lo, g.conv(4, hi)), False
def shuffle_again_turned(g):
    lo, hi = head(g)
    return g.shuffle("out", g.conv(4, hi), lo), False
def units_of_one_layer(g):
    lo, hi = head(g)
    lo, hi = g.unit("v", lo, g.conv(4, hi))
    return g.shuffle("out", lo, g.conv(6, g.conv(5, hi, True))), True
def pooled(g):
    lo, hi = head(g)
    g.conv(5, lo)
    return g.mean("out", g.conv(4, hi)), False
def next_unit(g):
    lo, hi = head(g)
    lo, hi = g.unit("v", lo, g.conv(6, g.conv(5, g.conv(4, hi, True), True, True)))
    return g.shuffle("out", lo, g.conv(9, g.conv(8, g.conv(7, hi, True), True, True))), True
def block_with_first_half(g):
    lo, hi = head(g)
    return g.sum("out", lo, g.conv(6, g.conv(5, g.conv(4, hi, True), True, True))), True
def block_with_first_half_turned(g):
    lo, hi = head(g)
    return g.sum("out", g.conv(6, g.conv(5, g.conv(4, hi, True), True, True)), lo), True
def another_pointwise(g):
    lo, hi = head(g)
    return g.sum("out", lo, g.conv(5, g.conv(4, hi, True))), True
def three_pointwise(g):
    lo, hi = head(g)
    return g.sum("out", g.conv(6, g.conv(5, g.conv(4, hi, True), True)), g.conv(7, lo)), True
TAILS = [sum_with_first_half, sum_with_first_half_turned, sum_from_elsewhere, shuffle_again, shuffle_again_turned, units_of_one_layer, pooled,
         next_unit, block_with_first_half, block_with_first_half_turned, another_pointwise, three_pointwise]

def ran(g):
    return [int(fake.fake_count(b"c%d" % n)) for n, _ in g.convs]
"""


def run(tmp_path, script, program=False):
    so, prog, lib = str(tmp_path / "libfake.so"), str(tmp_path / "libprogram.so"), os.path.join(os.path.dirname(HERE), "tensor_amd", "lib")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", os.path.join(HERE, "fake_capi.cpp"), "-o", so])
    if program:
        subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", os.path.join(HERE, "net_program.cpp"), "-L" + lib, "-lotter_hip_host",
                               "-Wl,-rpath," + lib, "-o", prog])
    r = subprocess.run([sys.executable, "-c", SCRIPT + script, so, prog], capture_output=True, text=True, timeout=120, cwd=os.path.dirname(HERE))
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("light", [True, False])
def test_every_tail_of_a_unit(tmp_path, light):
    run(tmp_path, r"""
for form in (3, 2, 1):
    for join in (1, 0):
        for pair in (1, 0):
            for what, v in ((b"form", form), (b"join", join), (b"pair", pair), (b"avgpool", join)): fake.fake_set(what, v)
            for tail in TAILS:
                g = Graph(%s)
                out, pairs = tail(g)
                where = (tail.__name__, form, join, pair)
                g.ready()
                s = g.net.session("data", blob(), out)
                before, pairs0 = ran(g), fake.fake_count(b"pair")
                s.run()
                assert fetched(s) == g.expr[out], (where, fetched(s))
                once = [b - a for a, b in zip(before, ran(g))]
                if tail is pooled: del once[3]  # (nobody asks for that one)
                assert max(once) == 1 and min(once) == 1, (where, once)
                if pairs and pair and join and form == 3: assert fake.fake_count(b"pair") > pairs0, where
                for _ in range(5):  # (recorded from the third on)
                    s.run()
                    assert fetched(s) == g.expr[out], where
                    assert expr_of(g.net.eval({"data": blob()}, out)) == g.expr[out], where
                s.close()
                g.net.close()
""" % light)


def test_a_second_half_that_is_asked_for_is_there(tmp_path):
    run(tmp_path, r"""
for tail in (next_unit, sum_with_first_half, another_pointwise):
    for ask in ("u_hi", "u_lo", "c4", "u_hi,out", "out,u_hi", "u_lo,c4,out"):
        g = Graph(light=ask != "out,u_hi")  # (in light mode a pass lets go of what it has read)
        tail(g)
        g.ready()
        s = g.net.session("data", blob(), ask)
        for _ in range(5):
            s.run()
            assert fetched(s) == g.expr[ask.split(",")[-1]], (tail.__name__, ask, fetched(s))
        if "," not in ask:
            for _ in range(5): assert expr_of(g.net.eval({"data": blob()}, ask)) == g.expr[ask], (tail.__name__, ask)
        s.close()
        g.net.close()
program = C.CDLL(sys.argv[2])
program.program_extract.restype = C.c_long
for tail in (next_unit, another_pointwise):  # not one of those that the program said it would ask for
    g = Graph()
    tail(g)
    g.ready()
    n = program.program_extract(g.net.h, b"data", blob().ctypes.data_as(C.c_void_p), CH, SIDE, SIDE, b"out", b"u_hi")
    assert n >= 0 and fake.fake_expr(C.c_long(n)).decode() in (g.expr["u_hi"], "q(%s)" % g.expr["u_hi"]), n
    g.net.close()
""", program=True)


def test_layers_in_front_of_a_concat_write_their_slices(tmp_path):
    """A Concat that an int8 convolution reads, of a pointwise layer and the depthwise one behind it (a ghost module), of an upsampling and
    a pointwise layer, and of what has to stay as it is."""
    run(tmp_path, r"""
def up(g, name, src):
    return g.add(name, "up(%s)" % g.expr[src], type="Upsample", input=src, stride=1)
def cat(g, name, *src):
    return g.add(name, "cat(%s)" % ",".join(g.expr[s] for s in src), type="Concat", input=",".join(src))
def wide(g, number, src):  # a pointwise layer over a concatenation
    name = "c%d" % number
    g.wide = getattr(g, "wide", []) + [(number, 0)]
    return g.add(name, "%s(%s)" % (name, g.expr[src]), type="Convolution", input=src, out_channels=CH, kernel=1, int8_scale_term=2)
def ghost(g, a=3, b=2):  # 3: the pointwise layer's channels come first
    first = g.conv(2, g.conv(1, "data"))
    second = g.conv(3, first, dw=True)
    return wide(g, 4, cat(g, "cat", *((first, second) if a > b else (second, first))))
def ghost_turned(g):
    return ghost(g, 2, 3)
def lateral(g):
    x = g.conv(1, "data")
    return wide(g, 4, cat(g, "cat", up(g, "up", x), g.conv(2, x)))
def three(g):
    x = g.conv(1, "data")
    p = g.conv(2, x)
    return wide(g, 4, cat(g, "cat", p, up(g, "up", x), g.conv(3, p, dw=True)))
def two_readers(g):  # (beside the Concat a depthwise and a pointwise layer)
    p = g.conv(2, g.conv(1, "data"))
    out = wide(g, 4, cat(g, "cat", p, g.conv(3, p, dw=True)))
    return g.sum("out", out, g.conv(5, p))
def read_by_a_sum(g):
    p = g.conv(2, g.conv(1, "data"))
    return g.sum("out", wide(g, 4, cat(g, "cat", p, g.conv(3, p, dw=True))), p)
def read_twice(g):
    p = g.conv(2, g.conv(1, "data"))
    c = cat(g, "cat", p, g.conv(3, p, dw=True))
    return g.sum("out", wide(g, 4, c), wide(g, 5, c))
def read_in_fp32(g):
    x = g.conv(1, "data")
    return up(g, "out", cat(g, "cat", up(g, "up", x), g.conv(2, x)))
def the_same_twice(g):
    p = g.conv(2, g.conv(1, "data"))
    return wide(g, 4, cat(g, "cat", p, p))
for light in (True, False):
  for on in (1, 0):
    fake.fake_set(b"slice", on)
    for tail, slices in ((ghost, 2), (ghost_turned, 2), (lateral, 2), (three, 3), (two_readers, 2), (read_by_a_sum, 0), (read_twice, 2), (read_in_fp32, 0), (the_same_twice, 0)):
        for ask in (None, "c2", "cat", "c3"):
            if ask == "c3" and tail in (lateral, read_in_fp32, the_same_twice): continue
            g = Graph(light)
            out = tail(g)
            g.ready()
            for number, _ in getattr(g, "wide", []):
                g.net.set_conv("c%d" % number, np.full((CH, (3 if tail is three else 2) * CH, 1, 1), number, np.int8), None, np.full(CH, 50, np.float32), 20.0, 10.0)
            names = out if ask is None else ask + "," + out
            s = g.net.session("data", blob(), names)
            g.convs += getattr(g, "wide", [])
            for k in range(5):
                before, made = ran(g), fake.fake_count(b"slice")
                s.run()
                where = (tail.__name__, light, on, ask, k)
                assert fetched(s) == g.expr[out], (where, fetched(s))
                assert all(b - a == 1 for a, b in zip(before, ran(g))) or (light and ask), where
                if not light or ask is None:
                    assert (fake.fake_count(b"slice") - made == slices) or ask or not on, where
                if not on or ask in ("cat", "c2"): assert fake.fake_count(b"slice") == made, where
            if ask is None or not light:
                assert expr_of(g.net.eval({"data": blob()}, out)) == g.expr[out], where
            s.close()
            g.net.close()
""")


def test_a_convolution_of_the_program_runs_its_own_forward(tmp_path):
    """Two pointwise layers that would be a pair, of a class that the program has put in the place of the library's."""
    run(tmp_path, r"""
program = C.CDLL(sys.argv[2])
for own in (0, 1):
    if own:
        program.program_register(1)
    g = Graph()
    out = g.conv(3, g.conv(2, g.conv(1, "data", True, dw=True), True))
    g.ready()
    s = g.net.session("data", blob(), out)
    pairs = fake.fake_count(b"pair")
    s.run()
    twice = lambda e: "sum(%s,%s)" % (e, e) if own else e
    assert fetched(s) == twice("c3(%s)" % twice("c2(%s)" % twice("c1(x)"))), fetched(s)
    assert fake.fake_count(b"pair") - pairs == (not own)
    s.close()
    g.net.close()
""", program=True)


BEHIND = r"""
def residual_blocks(g):  # the sum of one block is read by the next one's first layer and by its sum
    s = g.conv(1, "data")
    for k in (2, 5):
        s = g.sum("s%d" % k, s, g.conv(k + 2, g.conv(k + 1, g.conv(k, s, True), True, True)))
    return g.mean("out", g.conv(8, s))
def without_a_sum(g):  # an fp32 result that the next block's first layer and its sum read
    s = g.conv(3, g.conv(2, g.conv(1, "data", True), True, True))
    return g.sum("out", s, g.conv(6, g.conv(5, g.conv(4, s, True), True, True)))
def head_of_three(g):
    return g.conv(4, g.conv(3, g.conv(2, g.conv(1, "data", True), True, True), True))
def two_readers(g):  # the depthwise result has another reader
    d = g.conv(2, g.conv(1, "data", True), True, True)
    return g.sum("out", g.conv(3, d), g.conv(4, d))
MORE = [residual_blocks, without_a_sum, head_of_three, two_readers]
def set_all(**kw):
    for k, v in kw.items(): fake.fake_set(k.encode(), v)
"""


@pytest.mark.parametrize("light", [True, False])
def test_depthwise_layers_in_the_launch_of_their_reader(tmp_path, light):
    run(tmp_path, BEHIND + r"""
seen = {}
for form in (3, 1):
    for join, pair, alone, behind in ((1, 1, 1, 1), (1, 1, 1, 0), (1, 1, 0, 1), (0, 1, 1, 1), (1, 0, 1, 0), (1, 1, 0, 0)):
        set_all(form=form, join=join, pair=pair, dwpw=alone, dwpw_next=behind)
        for tail in TAILS + MORE:
            g = Graph(%s)
            made = tail(g)
            out = made[0] if isinstance(made, tuple) else made
            where = (tail.__name__, form, join, pair, alone, behind)
            g.ready()
            s = g.net.session("data", blob(), out)
            before, launches = ran(g), [fake.fake_count(k) for k in (b"dwpw", b"dwpw_next")]
            s.run()
            assert fetched(s) == g.expr[out], (where, fetched(s))
            once = [b - a for a, b in zip(before, ran(g))]
            if tail is pooled: del once[3]  # (nobody asks for that one)
            assert max(once) == 1 and min(once) == 1, (where, once)
            took = [fake.fake_count(k) - n for k, n in zip((b"dwpw", b"dwpw_next"), launches)]
            assert (alone or not took[0]) and (behind or not took[1]), where
            if form == 3 and join: seen[(tail.__name__, alone, behind)] = took
            for _ in range(5):  # (recorded from the third on)
                s.run()
                assert fetched(s) == g.expr[out], where
                assert expr_of(g.net.eval({"data": blob()}, out)) == g.expr[out], where
            s.close()
            g.net.close()
assert seen["residual_blocks", 1, 1] == [1, 1] and seen["residual_blocks", 1, 0] == [2, 0], seen  # (the second block's sum has no such reader)
assert seen["without_a_sum", 1, 1] == [1, 1] and seen["head_of_three", 1, 1] == [0, 1] and seen["next_unit", 1, 1][1] == 1, seen
assert seen["two_readers", 1, 1] == [0, 0], seen
""" % light)


def test_what_is_inside_such_a_launch_is_there_when_asked_for(tmp_path):
    run(tmp_path, BEHIND + r"""
for form in (3, 1):
    set_all(form=form)
    for tail, asks in ((residual_blocks, ("c3", "c4", "s2", "c5", "c6", "s2,out", "c3,out", "out,c3", "c5,out", "out,s2")),
                       (without_a_sum, ("c2", "c3", "c4", "c5", "c3,out", "c4,out", "c5,out", "out,c3")), (head_of_three, ("c2", "c3", "c2,c4", "c4,c3"))):
        for ask in asks:
            for light in (True, False) if ask.split(",")[0] not in ("out", asks[-1].split(",")[0]) else (False,):  # (light: a pass lets go of what it has read)
                g = Graph(light)
                tail(g)
                g.ready()
                s = g.net.session("data", blob(), ask)
                for _ in range(5):
                    s.run()
                    got, want = fetched(s), g.expr[ask.split(",")[-1]]
                    assert got == want, (tail.__name__, ask, light, got)
                s.close()
                g.net.close()
""")


def test_a_blob_in_front_of_such_a_launch_is_there_unannounced(tmp_path):
    """A program says that it will ask for the last blob, and asks for one whose only reader would run in the launch that makes it."""
    run(tmp_path, BEHIND + r"""
program = C.CDLL(sys.argv[2])
program.program_extract.restype = C.c_long
def read_by_one(g):
    s = g.sum("s", g.conv(1, "data"), g.conv(4, g.conv(3, g.conv(2, "data", True), True, True)))
    return g.conv(5, s)
def without_a_sum(g):
    return g.conv(4, g.conv(3, g.conv(2, g.conv(1, "data", True), True, True)))
for light in (True, False):
    for tail, asked in ((read_by_one, "s"), (without_a_sum, "c3")):
        g = Graph(light)
        out = tail(g)
        g.ready()
        n = program.program_extract(g.net.h, b"data", blob().ctypes.data_as(C.c_void_p), CH, SIDE, SIDE, out.encode(), asked.encode())
        assert n >= 0 and fake.fake_expr(C.c_long(n)).decode() in (g.expr[asked], "q(%s)" % g.expr[asked]), (tail.__name__, light, n)
        g.net.close()
""", program=True)


@pytest.mark.parametrize("light", [True, False])
def test_no_layer_runs_that_nobody_asked_for(tmp_path, light):
    """A blob in front of a layer that could run in the same launch, and one on another way through the net."""
    run(tmp_path, BEHIND + r"""
import re
def two_heads(g):  # c5 reads the sum of a block, and so does a mean
    s = g.sum("s", g.conv(1, "data"), g.conv(4, g.conv(3, g.conv(2, "data", True), True, True)))
    g.mean("m", s)
    return g.conv(5, s)
for form in (3, 1):
    for join, pair, behind in ((1, 1, 1), (1, 1, 0), (0, 1, 1), (1, 0, 1)):
        set_all(form=form, join=join, pair=pair, dwpw_next=behind)
        for tail in TAILS + MORE + [two_heads]:
            probe = Graph(%s)
            tail(probe)
            asks = sorted(n for n in probe.expr if n != "data" and "_" not in n or n in ("u_lo", "u_hi", "v_lo", "v_hi"))
            probe.ready().net.close()
            for ask in asks:
                g = Graph(%s)
                tail(g)
                g.ready()
                s = g.net.session("data", blob(), ask)
                before = ran(g)
                s.run()
                got, want = fetched(s), g.expr[ask]
                assert got == want, (tail.__name__, ask, got)
                used = set(re.findall(r"c(\d+)\(", want))
                once = {n: b - a for (n, _), a, b in zip(g.convs, before, ran(g))}
                assert once == {n: int(str(n) in used) for n, _ in g.convs}, (tail.__name__, form, join, pair, behind, ask, once)
                s.close()
                g.net.close()
set_all(form=3, join=1, pair=1, dwpw_next=1)
for asks, launches in (("m", 0), ("m,c5", 1), ("c5", 1)):  # (wanted later in the pass: run now)
    g = Graph(%s)
    two_heads(g)
    g.ready()
    s = g.net.session("data", blob(), asks)
    before, made = ran(g), fake.fake_count(b"dwpw_next")
    s.run()
    assert fetched(s) == g.expr[asks.split(",")[-1]]
    assert fake.fake_count(b"dwpw_next") - made == launches, asks
    assert [b - a for a, b in zip(before, ran(g))] == [1, 1, 1, 1, launches], asks
    s.close()
    g.net.close()
""" % (light, light, light))


@pytest.mark.parametrize("light", [True, False])
def test_a_max_pooling_in_the_launch_of_an_image_stem(tmp_path, light):
    run(tmp_path, r"""
CH3 = 3
for on in (1, 0):
    for ask in ("out", "pool", "c1", "pool,out", "c1,out", "out,c1"):
        if %s and ask == "out,c1": continue  # (in light mode a pass lets go of what it has read)
        fake.fake_set(b"stem_pool", on)
        net = hostnet.Net(lightmode=%s)
        net.add_layer(type="Input", name="data", batchsize=1, channel=3, height=16, width=16)
        net.add_layer(type="Convolution", name="c1", input="data", out_channels=8, kernel=3, stride=2, padding=1, int8_scale_term=2)
        net.add_layer(type="MaxPool", name="pool", input="c1", kernel=3, stride=2, padding=1)
        net.add_layer(type="Convolution", name="c2", input="pool", out_channels=8, kernel=1, int8_scale_term=2)
        net.add_layer(type="Convolution", name="c3", input="pool", out_channels=8, kernel=1, int8_scale_term=2)
        net.add_layer(type="Eltwise", name="out", input="c2,c3")
        net.compile()
        net.set_conv("c1", np.full((8, 3, 3, 3), 1, np.int8), None, np.full(8, 50, np.float32), 20.0, 10.0)
        for n in (2, 3): net.set_conv("c%%d" %% n, np.full((8, 8, 1, 1), n, np.int8), None, np.full(8, 50, np.float32), 20.0, 10.0)
        x = np.zeros((1, 3, 16, 16), np.float32)
        x.reshape(-1)[:2].view(np.int64)[0] = fake.fake_number(b"x")
        expr = dict(c1="c1(x)", pool="maxpool(c1(x))")
        expr["out"] = "sum(c2(%%s),c3(%%s))" %% (expr["pool"], expr["pool"])
        s = net.session("data", x, ask)
        launches = fake.fake_count(b"stem_pool")
        for _ in range(5):
            s.run()
            got, want = expr_of(s.fetch((2 * 8 * 64,), np.float32)), expr[ask.split(",")[-1]]
            assert got == want, (on, ask, got)
        assert (fake.fake_count(b"stem_pool") > launches) == (on and "c1" not in ask), (on, ask)
        s.close()
        net.close()
""" % (light, light))

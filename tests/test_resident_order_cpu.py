"""The resident decode kernels hand values on through words that are written over without asking (decode_resident_order.h).  Every read and
write of some steps as a graph: a barrier of a workgroup lies behind the one in front of it and behind the puts of all words read
between them, a put behind its workgroup's last barrier and behind the words its threads read for it.  A put is in order if every reader of
the place's last value has a barrier behind that read from which a path leads to the put.  Workgroups of an XCD: three stand for 32."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zig_gpt2_amd", "csrc")
XCDS, RANKS = 8, 3


@pytest.fixture(scope="module")
def far1_from(tmp_path_factory):
    """XCDs that put partial sums of c_proj, of the header the kernels are built with"""
    d = tmp_path_factory.mktemp("order")
    (d / "o.cpp").write_text('#include "decode_resident_order.h"\nextern "C" int xcds() { return zg::resident::kXcds; }\n'
                             'extern "C" int far1_from() { return zg::resident::kFar1From; }\n')
    subprocess.check_call(["g++", "-std=c++17", "-fPIC", "-shared", f"-I{CSRC}", "-o", str(d / "o.so"), str(d / "o.cpp")])
    lib = C.CDLL(str(d / "o.so"))
    assert lib.xcds() == XCDS
    return lib.far1_from()


class Graph:
    def __init__(self):
        self.before = []          # node -> bits of the nodes in front of it, itself among them
        self.last = {}            # workgroup -> its last barrier
        self.open = {}            # workgroup -> puts read since
        self.place = {}           # place -> (put, [(workgroup, reads so far)])
        self.waiting = {}         # workgroup -> places read since its last barrier
        self.readers = {}         # put -> barriers behind its reads
        self.wrong = set()

    def node(self, preds):
        bits = 1 << len(self.before)
        for p in preds:
            bits |= self.before[p]
        self.before.append(bits)
        return len(self.before) - 1

    def barrier(self, wg):
        n = self.node(([self.last[wg]] if wg in self.last else []) + self.open.pop(wg, []))
        for put in self.waiting.pop(wg, []):
            self.readers.setdefault(put, []).append(n)
        self.last[wg] = n

    def read(self, wg, places):
        puts = [self.place[p] for p in places]
        self.open.setdefault(wg, []).extend(puts)
        self.waiting.setdefault(wg, []).extend(puts)
        return puts

    def put(self, wg, place, behind=()):
        n = self.node(([self.last[wg]] if wg in self.last else []) + list(behind))
        old = self.place.get(place)
        if old is not None:
            unread = [w for w, ps in self.waiting.items() if old in ps]
            if unread or any(not self.before[n] >> b & 1 for b in self.readers.get(old, [])):
                self.wrong.add(place[0])
        self.place[place] = n
        return n


def run(heads, batch, attending, layers, picks, far1_from):
    """picks: for every step, whether it ends in one.  attending(r): workgroup r of an XCD with heads attends."""
    g, wgs = Graph(), [(k, r) for k in range(XCDS) for r in range(RANKS)]
    has = lambda k: k < heads
    xcd = lambda name, k: [(name, k, r) for r in range(RANKS)]

    def each(what):
        for wg in wgs:
            what(*wg)

    def bar(k, r):
        g.barrier((k, r))

    def x(far, to, from_n):
        """far sums -> x, put by the threads that read them"""
        sums = {wg: g.read(wg, [(far, q, wg[1]) for q in range(from_n)]) for wg in wgs}
        if batch:
            each(bar)
        each(lambda k, r: g.put((k, r), (to, k, r), [] if batch else sums[k, r]))

    each(bar)
    for pick in picks:
        if batch:
            each(lambda k, r: g.put((k, r), ("x2", k, r)))
        for _ in range(layers):
            started = any(p[0] == "x2" for p in g.place)
            if started:
                each(lambda k, r: g.read((k, r), xcd("x2", k)) if has(k) or not batch else None)
            each(bar)
            each(lambda k, r: g.put((k, r), ("qkv", k, r)) if has(k) else g.put((k, r), ("far1", k, r)) if k < far1_from else None)
            for k, r in wgs:
                if has(k) and attending(r):
                    g.read((k, r), xcd("qkv", k))
                    bar(k, r)
                    bar(k, r)
            each(lambda k, r: g.put((k, r), ("att", k, r)) if has(k) and attending(r) else None)
            each(lambda k, r: g.read((k, r), [("att", k, i) for i in range(RANKS) if attending(i)]) if has(k) else None)
            for k, r in wgs:
                if has(k):
                    bar(k, r)
                    bar(k, r)
            each(lambda k, r: g.put((k, r), ("far1", k, r)) if has(k) else None)
            x("far1", "x1", far1_from)
            if batch:
                each(bar)
            each(lambda k, r: g.read((k, r), xcd("x1", k)))
            each(bar)
            each(lambda k, r: g.put((k, r), ("h", k, r)))
            if batch:
                each(bar)
            each(lambda k, r: g.read((k, r), xcd("h", k)))
            each(bar)
            each(bar)
            each(lambda k, r: g.put((k, r), ("far2", k, r)))
            x("far2", "x2", XCDS)
        if pick:
            each(lambda k, r: g.read((k, r), xcd("x2", k)))
            each(bar)
            each(bar)
            each(lambda k, r: g.put((k, r), ("best", k, r)))
            for k in range(XCDS):
                bests = g.read((k, 0), xcd("best", k))
                g.put((k, 0), ("pick", k), bests)
            each(lambda k, r: g.read((k, r), [("pick", q) for q in range(XCDS)]))
        elif not batch:
            each(lambda k, r: g.read((k, r), xcd("x2", k)))
        each(bar)
        each(bar)
    return g.wrong


ATTEND = {"one": lambda r: r == 0, "two": lambda r: r < 2, "all": lambda r: True}


@pytest.mark.parametrize("heads", [1, 6, 8, 12, 16])
@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("attend", sorted(ATTEND))
def test_every_read_lies_in_front_of_the_next_put(far1_from, heads, batch, attend):
    for layers in (2, 3):
        assert not run(heads, batch, ATTEND[attend], layers, (False, False, True, True), far1_from), layers


@pytest.mark.parametrize("batch", [False, True])
def test_sums_of_the_xcds_with_heads_alone_are_not_enough(batch):
    """What the graph says of the order without the words of XCDs that have no heads."""
    assert "far2" in run(6, batch, ATTEND["two"], 2, (True, True), 6)
    assert not run(8, batch, ATTEND["two"], 2, (True, True), 8)

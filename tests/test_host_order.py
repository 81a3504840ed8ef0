"""The order in which filters and batches enqueue their work, and what they do
when a call to the runtime fails, on the CPU: libesthera.so runs on a stand-in
for the HIP runtime (fake_hip.cpp) that launches nothing and logs every call.
Each scenario runs in a process of its own, where the stand-in is loaded first."""
import ctypes as C
import os
import re
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


class Fake:
    """The stand-in: its log, and failures asked for by a part of a log line."""

    def __init__(self, path):
        self.lib = C.CDLL(path, mode=C.RTLD_GLOBAL)
        self.lib.fake_log.restype = C.c_char_p
        self.lib.fake_fail.argtypes = [C.c_char_p]

    def log(self):
        return self.lib.fake_log().decode().splitlines()

    def take(self):
        lines = self.log()
        self.lib.fake_clear()
        return lines

    def fail(self, what):
        self.lib.fake_fail(what.encode())


def walk(ea, m=128, G=12, **k):
    """A random walk's filter and its step's arguments."""
    d = ea.filter_desc(ea.MODEL_RANDOMWALK3, m=m, G=G, weights=ea.WEIGHTS_LOG, resampler=ea.RESAMPLE_SYSTEMATIC, **k)
    p, c, z, _ = ea.randomwalk3_scenario(3, 1)
    return d, p, (c[0], z[0], 0.1)


def fails(ea, call, *args):
    try:
        call(*args)
    except ea.EsthError:
        return True
    return False


def failed_argmax(ea, fake):
    d, p, args = walk(ea)
    fake.take()
    f = ea.Filter(ea.Engine(0), d, p)
    # the estimate's pinned buffer: 4 + 2 * 16 doubles and the count of argmaxes that have published one
    at = [int(l.split()[1], 16) for l in fake.take() if l.startswith("hipHostMalloc") and l.endswith("bytes 296")]
    count = C.c_uint64.from_address(at[0] + 288)
    f.init_uniform([0.0, 0.0, 0.0])

    def waits():
        fake.take()
        f.estimate()
        return any(l.startswith("hipStreamSynchronize") for l in fake.take())

    f.step(*args)
    count.value = 1
    assert not waits()
    # a failed launch that did not run
    fake.fail("k_resample_argmax")
    assert fails(ea, f.step, *args)
    assert waits(), "after a failed launch the estimate waits for the stream"
    f.step(*args)
    count.value = 2
    assert not waits(), "the count is short for good"
    # one that ran although the call failed
    fake.fail("k_resample_argmax")
    assert fails(ea, f.step, *args)
    count.value = 3
    assert waits()
    f.step(*args)
    assert fails(ea, f.estimate), "an estimate that was not published is no estimate"
    f.step(*args)
    count.value = 4
    assert not waits()


def failed_batch_step(ea, fake):
    d, p, (c, z, dt) = walk(ea, rng=ea.RNG_MTGP_PER_FILTER)
    b = ea.Batch(ea.Engine(0), [d, d], [p, p])
    cs, zs, dts = (ea.RandomWalk3Control * 2)(c, c), (ea.RandomWalk3Measurement * 2)(z, z), [dt, dt]
    fake.take()
    b.step(cs, zs, dts)
    last = fake.take()[-1]   # an event after the step's kernels
    assert last.startswith("hipEventRecord")
    b.step(cs, zs, dts)
    b.estimate(0)
    fake.take()
    b.estimate(1)
    assert not fake.take(), "one wait for all estimates of a step"
    fake.fail(last)   # the third step, its kernels enqueued
    assert fails(ea, b.step, cs, zs, dts)
    assert any("GraphLaunch" in l for l in fake.take())
    b.estimate(0)
    assert any(l.startswith("hipStreamSynchronize") for l in fake.take()), "kernels may still write the estimates"


def creation_waits_for_no_stream(ea, fake):
    d, p, _ = walk(ea)
    e = ea.Engine(0)
    fake.take()
    f = ea.Filter(e, d, p)
    log = fake.take()
    assert f.h and sum(l.startswith("hipMemcpy") for l in log) >= 2   # statuses and streams go up
    assert not [l for l in log if "Synchronize" in l]


def steps_per_block(log):
    """(stream, steps) of each generator launch."""
    return [(l.split()[3], int(l.split()[5])) for l in log if "6k_mtgp" in l]


def carried_words(ea, fake):
    """Small filters' words ride in the step's own launches (those of test_gpu_carried_words among them): the
    generator is launched ahead of the first step only.  A block length asked for puts any filter's words on the
    second stream, in blocks of that length."""
    e = ea.Engine(0)
    for m, G, L, res in ((256, 64, 4, ea.RESAMPLE_SYSTEMATIC), (64, 100, 4, ea.RESAMPLE_ALIAS),
                         (512, 512, 20, ea.RESAMPLE_ALIAS)):
        p, c, z, _ = ea.unicycle_scenario(3, L, 20.0, 1)
        d = ea.filter_desc(ea.MODEL_UNICYCLE, m=m, G=G, t=1, resampler=res, weights=ea.WEIGHTS_LOG, seed=77)
        for block in (0, 1, 2, 3, 4):
            os.environ.pop("ESTH_RNG_BLOCK_STEPS", None)
            if block:
                os.environ["ESTH_RNG_BLOCK_STEPS"] = str(block)
            f = ea.Filter(e, d, p)
            f.init_uniform([0.0, 0.0, 0.0])
            fake.take()
            for _ in range(8):
                f.step(c[0], z[0], 0.1)
            got = steps_per_block(fake.take())
            if block == 0:
                assert len(got) == 1 and got[0][1] == 1, (m, G, got)
            else:
                assert f.rng_mode() == (False, block)
                assert len({s for s, _ in got}) == 2 and got[-1][1] == block, (m, G, block, got)


class Order:
    """Follows a log: which step's words lie where, and what is ordered before what (a clock per stream and for the
    host).  Words are read after they were written, overwritten after they were read, and every step's words are
    generated from the status that the step before left."""

    def __init__(self):
        self.now, self.events, self.host = {}, {}, {}   # stream -> clock (stream -> its count), event -> clock
        self.status, self.words = {}, {}                # address -> step; address -> [step, writer, readers]
        self.step = 0

    def restored(self, step):
        self.status, self.words, self.step = {}, {}, step

    def op(self, s):
        c = self.now.setdefault(s, {})
        for k, v in self.host.items():
            c[k] = max(c.get(k, 0), v)
        c[s] = c.get(s, 0) + 1
        return (s, c[s])

    def after(self, s, op):
        return self.now[s].get(op[0], 0) >= op[1]

    def line(self, l):
        t = l.split()
        if t[0] == "hipEventRecord":
            self.op(t[4])
            self.events[t[2]] = dict(self.now[t[4]])
        elif t[0] == "hipStreamWaitEvent":
            self.op(t[2])
            for k, v in self.events[t[4]].items():
                self.now[t[2]][k] = max(self.now[t[2]].get(k, 0), v)
        elif t[0] == "hipStreamSynchronize":
            for k, v in self.now.get(t[2], {}).items():
                self.host[k] = max(self.host.get(k, 0), v)
        elif t[0] == "launch" and "6k_mtgp" in t[1]:
            s, n, frm, to, ds, at, dw = t[3], *map(int, t[5:16:2])
            me = self.op(s)
            first, by = self.status.get(frm, (self.step, None))
            assert by is None or self.after(s, by), "the status is not there yet"
            for i in range(n):
                old = self.words.get(at + i * dw)
                assert old is None or all(self.after(s, r) for r in old[2]), f"words of step {old[0]} overwritten"
                self.words[at + i * dw] = [first + i, me, []]
                self.status[to + i * ds] = (first + i + 1, me)
        elif t[0] == "launch" and "k_sample" in t[1]:
            s = t[3]
            me = self.op(s)
            mine = [w for w in self.words.values() if w[0] == self.step]
            assert mine and all(self.after(s, w[1]) for w in mine), f"words of step {self.step} are not there yet"
            for w in mine:
                w[2].append(me)
            self.step += 1


def cold_start(ea, fake):
    """The first step after a creation or a restore waits for the words of two steps at most, whatever the block, and
    the others are there in time, from any step on and with prefetch switched off and on."""
    e = ea.Engine(0)
    d, p, args = walk(ea, G=3001)
    for block in (0, 3, 8):
        if block:
            os.environ["ESTH_RNG_BLOCK_STEPS"] = str(block)
        f = ea.Filter(e, d, p)
        B = f.rng_mode()[1]
        assert B == (block or 4)
        f.init_uniform([0.0, 0.0, 0.0])
        fake.take()
        o, taken = Order(), 0

        def step():
            f.step(*args)
            log = fake.take()
            for l in log:
                o.line(l)
            return log

        snaps = []
        for k in range(2 * B + 2):
            ahead = []
            for l in step():
                if "k_sample" in l:
                    break
                ahead.append(l)
            if k == 0:
                assert max(n for _, n in steps_per_block(ahead)[:1]) <= 2, ahead
            snaps.append(f.snapshot())
            for l in fake.take():
                o.line(l)
        for k, s in enumerate(snaps):
            for off, on in ((None, None), (1, 2), (1, 3), (2, 4), (3, 4)):
                f.restore(s)
                for l in fake.take():
                    o.line(l)
                o.restored(k + 1)
                for i in range(2 * B + 3):
                    if i in (off, on):
                        f.set_prefetch(i == on)
                    log = step()
                    if i == 0:
                        main = [l.split()[3] for l in log if "k_sample" in l][0]
                        assert sum(n for st, n in steps_per_block(log) if st == main) <= 2, log
        f.close()
        fake.take()


def words_by_size(ea, fake):
    """Where a filter's words are made, both sides of each line: the generator's own launches, and the work-groups
    that the step's launches carry (96 streams)."""
    def grids(log):
        names = {"k_sample": "sample", "k_resample": "resample", "k_alias": "resample"}
        return {v: int(l.split()[5]) for l in log for k, v in names.items() if k in l}

    e = ea.Engine(0)
    RW, U, S, A = ea.MODEL_RANDOMWALK3, ea.MODEL_UNICYCLE, ea.RESAMPLE_SYSTEMATIC, ea.RESAMPLE_ALIAS
    for model, m, G, L, res, inline, carriers in (
            (RW, 512, 256, 0, S, False, "resample"), (RW, 512, 1024, 0, S, False, "sample resample"),
            (RW, 512, 2048, 0, S, False, ""), (RW, 128, 1024, 0, S, False, "resample"), (RW, 128, 2048, 0, S, False, ""),
            (U, 512, 512, 20, A, False, "sample resample"), (U, 512, 512, 20, S, False, "sample resample"),
            (U, 512, 1024, 4, S, False, "sample resample"), (U, 512, 4096, 4, S, False, ""), (U, 512, 4096, 30, S, False, "sample resample"), (U, 512, 4096, 31, S, True, "sample"),
            (U, 512, 64, 40, S, True, "sample"), (U, 512, 64, 4, S, False, "resample"),
            (U, 64, 2500, 4, S, False, "sample resample")):
        p, c, z, _ = ea.randomwalk3_scenario(3, 1) if model == RW else ea.unicycle_scenario(3, L, 20.0, 1)
        f = ea.Filter(e, ea.filter_desc(model, m=m, G=G, t=1, resampler=res, weights=ea.WEIGHTS_LOG, seed=7), p)
        f.set_cross_step(False)
        f.init_uniform([0.0, 0.0, 0.0])
        for _ in range(3):
            fake.take()
            f.step(c[0], z[0], 0.1)
        carrying, mode = grids(fake.take()), f.rng_mode()[0]
        f.set_prefetch(False)
        fake.take()
        f.step(c[0], z[0], 0.1)
        alone = grids(fake.take())
        got = " ".join(n for n in alone if carrying[n] == alone[n] + 96)
        assert (mode, got) == (inline, carriers), (model, m, G, L, res, carrying, alone)


def room_for_the_words(ea, fake):
    """Where the second stream's words bound an arm's step, the fused launch leaves them LDS on every CU: the
    work-groups that fit into its 160 KB, allotted in steps of 1280 bytes, are so many and leave the generator's 3200."""
    e = ea.Engine(0)
    for model, m, G, L, room in (("ROBOTARM5", 512, 4096, 0, 3), ("ROBOTARM5", 512, 2048, 0, 5), ("ROBOTARM5", 256, 4096, 0, 9),
                                 ("ROBOTARM5", 256, 8192, 0, 6), ("ROBOTARM5", 1024, 2048, 0, 0), ("ROBOTARM5", 512, 1024, 0, 0),
                                 ("ROBOTARM5", 256, 2048, 0, 0), ("ROBOTARM5", 512, 64, 0, 0), ("ROBOTARM5", 128, 8192, 0, 0),
                                 ("DH6", 512, 2048, 0, 0), ("UNICYCLE", 512, 4096, 4, 0), ("RANDOMWALK3", 512, 4096, 0, 0)):
        if model == "ROBOTARM5":
            p, c, z = None, ea.RobotArm5Control(), ea.RobotArm5Measurement()
        elif model == "DH6":
            (p, zs, _), c = ea.dh6_scenario(3, 1), ea.DH6Control()
            z = zs[0]
        else:
            p, cs, zs, _ = ea.randomwalk3_scenario(3, 1) if model == "RANDOMWALK3" else ea.unicycle_scenario(3, L, 20.0, 1)
            c, z = cs[0], zs[0]
        S = ea.STATE_DIM[getattr(ea, "MODEL_" + model)]
        f = ea.Filter(e, ea.filter_desc(getattr(ea, "MODEL_" + model), m=m, G=G, t=1, resampler=ea.RESAMPLE_SYSTEMATIC,
                                        weights=ea.WEIGHTS_LOG), p)
        f.init_uniform([0.0] * S)
        fake.take()
        f.step(c, z, 0.1)
        lds = [int(l.split()[7]) for l in fake.take() if "k_sample_sort" in l]
        f.close()
        assert len(lds) == 1 and (lds[0] > 0) == (room > 0), (model, m, G, lds)
        if room:
            own = 4 * ((1 + S) * m + 2 * (m + 64)) + lds[0]
            each = -(-own // 1280) * 1280
            assert 163840 // each == room and own <= 65536 and 163840 - room * each >= 3200


SCENARIOS = [failed_argmax, failed_batch_step, creation_waits_for_no_stream, carried_words, cold_start, words_by_size,
             room_for_the_words]


@pytest.fixture(scope="session")
def stand_in(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("scenario", [s.__name__ for s in SCENARIOS])
def test_host_order(scenario, stand_in):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), scenario, stand_in], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    fake = Fake(sys.argv[2])
    sys.path.insert(0, os.path.dirname(HERE))
    import esthera_amd
    globals()[sys.argv[1]](esthera_amd, fake)

"""Workloads of the simulator's device paths, for timing and comparison.

A case is one pass a user's program makes through a public entry point:

  scan      the plain drop-in (jq_simulate_scan) over one pre-filled snapshot
            buffer: 2-state, X-propagating, or with X, arrivals and
            setup/hold checks
  lanes     the batched form (batched.BatchedRun): many stimulus lanes of one
            netlist, hashed or recorded stimulus, with or without a queue of
            more lanes than slots
  cosim     reactive co-simulation edges (cosim.Cosim) with the SPI flash
            model, or of a larger netlist
  changes   output change records of a finished run (vcd.output_changes_device)
  mlp       the partition cost model (costmodel.MLP): a train step, or the
            prediction of every partition of a design

A design is generated and compiled once per process, as a program compiles
its netlist once and then simulates it with many stimuli; everything that
depends on the stimulus is made anew from the seed by prepare().
"""
import ctypes
import functools
import random

import numpy as np
import torch

from jacquard_amd import _native as N
from jacquard_amd import batched, cosim, costmodel, sim, stimulus, vcd
from jacquard_amd.netlist import Netlist
from jacquard_amd.script import Compiled

MAX_BLOCKS = 256  # one workgroup per compute unit


# ---------------------------------------------------------------- designs

@functools.lru_cache(maxsize=None)
def _netlist(gates, depth, dffs, inputs, outputs, srams, local, delays):
    return Netlist.random(seed=2, gates=gates, depth=depth, dffs=dffs, inputs=inputs,
                          outputs=outputs, geometric_p=0.3 if local else 0.0,
                          invert_prob=0.5 if local else 0.2, srams=srams,
                          sram_addr_bits=10, delay=(20, 200) if delays else (0, 0))


@functools.lru_cache(maxsize=None)
def _multiplier(tiles, gates, depth, dffs, inputs, outputs):
    return Netlist.multiplier(seed=7, tiles=tiles, width=16, control_gates=gates,
                              control_depth=depth, dffs=dffs, inputs=inputs, outputs=outputs)


def _case_netlist(c):
    if c.get("tiles", 0):
        return _multiplier(c["tiles"], c["gates"], c["depth"], c["dffs"], c["inputs"],
                           c["outputs"])
    # the fan-ins of all but the smallest netlists favour nearby levels; a
    # netlist with SRAMs carries gate delays whether or not a run uses them
    return _netlist(c["gates"], c["depth"], c["dffs"], c["inputs"], c["outputs"],
                    c.get("srams", 0), c["gates"] > 5000, c.get("srams", 0) > 0)


@functools.lru_cache(maxsize=None)
def _compiled(nl, split, cap):
    return Compiled(nl, level_split=split, max_level_nodes=cap)


@functools.lru_cache(maxsize=None)
def _script(nl, split, cap, blocks, xprop, timing):
    comp = _compiled(nl, split, cap)
    s = comp.flatten(blocks or min(max(comp.parts_per_stage()), MAX_BLOCKS), xprop=xprop)
    cons = None
    if timing:
        s.inject_timing()
        s.enable_timing_arrivals()
        cons = s.build_timing_constraint_buffer(5000, 50, 20)
    return s, cons


def _design(c):
    return _script(_case_netlist(c), c["split"], c.get("cap", 0), c.get("blocks", 0),
                   bool(c.get("xprop")), bool(c.get("timing")))


# ---------------------------------------------------------------- the cases

_SMALL = dict(gates=2000, depth=24, dffs=256, inputs=32, outputs=16, split=6)
_MID = dict(gates=97531, depth=40, dffs=7001, inputs=123, outputs=77, srams=3)
_1M = dict(gates=1_000_000, depth=64, dffs=1 << 16, inputs=512, outputs=256)
_4M = dict(gates=4_000_000, depth=96, dffs=1 << 18, inputs=512, outputs=256, srams=8)


def listed():
    return [
        # a testbench that steps a small block a few cycles at a time: launch
        # and table latency
        dict(_SMALL, name="scan_2k_8cycles", kind="scan", cycles=8, toggle=0.5),
        # a unit test's run of the same block: the per-cycle chain of one workgroup
        dict(_SMALL, name="scan_2k_1000cycles", kind="scan", cycles=1000, toggle=0.5),
        # a subsystem with memories brought up from X, sizes nobody rounded
        dict(_MID, name="scan_100k_x_sram", kind="scan", split=6, cycles=151, toggle=0.1,
             xprop=True),
        # the plain run of the 1M-gate netlist at its tuned partition width
        dict(_1M, name="scan_1m", kind="scan", split=6, cap=800, cycles=200, toggle=0.1),
        # sign-off style: 4M gates, X, arrivals and setup/hold checks together
        dict(_4M, name="scan_4m_x_timing", kind="scan", split=6, cycles=32, toggle=0.1,
             xprop=True, timing=True),
        # a regression of recorded tests of differing length: more lanes than
        # slots, so finished lanes hand their slot on
        dict(_MID, name="lanes_100k_recorded", kind="lanes", split=4, groups=1, blocks=5,
             lanes=41, cycles_lo=20, cycles_hi=90, recorded=True),
        # many short seeds of the 1M-gate netlist: every slot of a full chip
        dict(_1M, name="lanes_1m_8x32", kind="lanes", split=4, groups=8, blocks=32, lanes=256,
             cycles_lo=64, cycles_hi=64, recorded=False),
        # the 4M-gate netlist in the shape its long lanes are run in
        dict(_4M, name="lanes_4m_4x64", kind="lanes", split=3, groups=4, blocks=64, lanes=128,
             cycles_lo=24, cycles_hi=40, recorded=False),
        # firmware boot through a flash: one dependent edge after another
        dict(name="cosim_spi", kind="cosim", gates=0, edges=512, batch=256),
        # the waveform of a finished run
        dict(name="changes_20k", kind="changes", gates=20011, depth=30, dffs=1999, inputs=99,
             outputs=256, split=6, cycles=8192, toggle=0.2),
        # the cost model: a minibatch step and the costs of a design's partitions
        dict(name="mlp_train_4096", kind="mlp_train", n=4096, features=24, h1=64, h2=64),
        dict(name="mlp_forward_5013", kind="mlp_forward", n=5013, features=24, h1=64, h2=64),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _draw_netlist(rng, lo, hi):
    gates = _log(rng, lo, hi)
    return dict(gates=gates, depth=rng.randint(12, 24 + min(72, gates // 10_000)),
                dffs=max(16, int(gates * rng.uniform(0.04, 0.13))),
                inputs=rng.randint(8, 512), outputs=rng.randint(1, 256))


def draw(rng: random.Random):
    kind = rng.choice(["scan", "scan", "scan", "lanes", "lanes", "lanes", "cosim", "changes",
                       "mlp_train", "mlp_forward"])
    if kind == "scan":
        c = dict(_draw_netlist(rng, 1000, 1_000_000), kind=kind, split=rng.randint(4, 8),
                 srams=rng.choice([0, 0, 1, 4]), cap=rng.choice([0, 0, 800, 1300]),
                 toggle=round(rng.uniform(0.02, 0.5), 3),
                 xprop=rng.random() < 0.4, timing=False)
        c["timing"] = c["srams"] > 0 and rng.random() < 0.4
        c["cycles"] = _log(rng, 1, 100 if c["gates"] > 100_000 else 500)
        return c
    if kind == "lanes":
        groups = rng.randint(1, 8)
        lanes = rng.randint(1, 32 * groups) if groups > 1 else rng.randint(1, 60)
        lo = _log(rng, 2, 30)
        c = dict(_draw_netlist(rng, 2000, 1_000_000), kind=kind, split=rng.randint(3, 6),
                 srams=rng.choice([0, 0, 2]), cap=rng.choice([0, 0, 1300]), groups=groups,
                 lanes=lanes, cycles_lo=lo, cycles_hi=lo + rng.randint(0, 30),
                 recorded=rng.random() < 0.3)
        if rng.random() < 0.25:  # structured: array multipliers and a control network
            c.update(tiles=rng.randint(2, 24), srams=0, gates=min(c["gates"], 300_000))
        size = c["gates"] + 20_000 * c.get("tiles", 0)
        c["blocks"] = min(MAX_BLOCKS // groups, _log(rng, 1 + size // 40_000, 1 + size // 15_000))
        return c
    if kind == "cosim":
        if rng.random() < 0.5:
            return dict(kind=kind, gates=0, edges=rng.randint(40, 512),
                        batch=_log(rng, 16, 1024))
        return dict(_draw_netlist(rng, 2000, 300_000), kind=kind, split=6,
                    edges=rng.randint(10, 200), batch=_log(rng, 16, 1024))
    if kind == "changes":
        return dict(_draw_netlist(rng, 2000, 50_000), kind=kind, split=6,
                    cycles=_log(rng, 20, 8000), toggle=round(rng.uniform(0.02, 0.5), 3),
                    xprop=rng.random() < 0.3)
    wide = rng.random() < 0.7
    return dict(kind=kind, n=_log(rng, 1, 4096 if kind == "mlp_train" else 50_000),
                features=24 if wide else rng.randint(1, 32),
                h1=64 if wide else rng.randint(1, 64), h2=64 if wide else rng.randint(1, 64))


# ---------------------------------------------------------------- prepare

def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _seed32(seed):
    return (int(seed) * 2654435761 + 12345) % 0x7FFFFFFF + 1


class _Scan:
    EVENTS = 1 << 14

    def __init__(self, c, seed):
        s, cons = _design(c)
        self.s, self.cycles = s, c["cycles"]
        xm = None
        if s.xprop_enabled:
            xm, _ = stimulus.dff_initial_xmask(s, 0.1, seed=_seed32(seed))
        self.ss = s.effective_state_size()
        self.states = sim.to_device(stimulus.build_states(
            s, self.cycles, seed=_seed32(seed), p=c["toggle"], initial_xmask=xm))
        self.bs = sim.to_device(np.ascontiguousarray(s.blocks_start, np.uint64))
        self.bd = sim.to_device(np.ascontiguousarray(s.blocks_data, np.uint32))
        self.sram = torch.zeros(max(s.sram_storage_size, 1), dtype=torch.int32, device="cuda")
        self.sram_x = torch.zeros(self.sram.numel() if s.xprop_enabled else 1,
                                  dtype=torch.int32, device="cuda")
        self.cons = sim.to_device(cons) if cons is not None else None
        self.events = None
        if cons is not None:
            self.events = torch.zeros(4 + 8 * self.EVENTS, dtype=torch.int32, device="cuda")

    def run(self):
        s = self.s
        if s.sram_storage_size:  # memories start at zero, all X under X propagation
            self.sram.zero_()
            if s.xprop_enabled:
                self.sram_x.fill_(-1)
        if self.events is not None:
            self.events.zero_()
        N.check(N.hip().jq_simulate_scan(
            s.num_blocks, s.num_major_stages, self.bs.data_ptr(), self.bd.data_ptr(),
            self.sram.data_ptr(), self.sram_x.data_ptr(), self.cycles, self.ss,
            self.states.data_ptr(), self.cons.data_ptr() if self.cons is not None else None,
            self.events.data_ptr() if self.events is not None else None,
            self.EVENTS if self.events is not None else 0, int(s.arrival_state_offset),
            _stream()))
        out = {"states": self.states, "sram": self.sram, "sram_x": self.sram_x}
        if self.events is not None:
            # records come in no defined order; a report takes them by
            # (cycle, word, kind)
            rec = self.events[4:].view(-1, 8)
            key = (rec[:, 2].long() << 40) | (rec[:, 1].long() << 8) | rec[:, 0].long()
            out["event_header"] = self.events[:4]
            out["events"] = rec[torch.argsort(key)]
        return out


class _Lanes:
    def __init__(self, c, seed):
        s, _ = _design(c)
        rng = np.random.default_rng(_seed32(seed))
        n = c["lanes"]
        lo, hi = c["cycles_lo"], c["cycles_hi"]
        # the lengths are the case's, which lane has which the seed's; where
        # lanes wait for slots no two of them are the same, so that the slot
        # a waiting lane gets is defined
        step = max(1, (hi - lo) // max(1, n - 1)) if n > 32 * c["groups"] else 0
        cycles = lo + (np.arange(n) * step if step else np.arange(n) * 7919 % (hi - lo + 1))
        cycles = rng.permutation(cycles)
        probs = rng.uniform(0.02, 0.5, n)
        seeds = rng.integers(1, 2**31, n).astype(np.uint32)
        if c["recorded"]:
            words = [stimulus.input_words(s, int(k), seed=int(q), p=float(p))
                     for k, q, p in zip(cycles, seeds, probs)]
            self.r = batched.BatchedRun(s, None, None, None, groups=c["groups"], stimulus=words)
        else:
            self.r = batched.BatchedRun(s, seeds, probs, cycles, groups=c["groups"])
        self.r.prepare()

    def run(self):
        r = self.r
        r.reset()
        r.launch()
        d = r.d
        return {"outputs": d["obs"], "states": d["states"], "sram": d["sram"],
                "lane_info": d["info"], "group_cycles": d["gcyc"]}


@functools.lru_cache(maxsize=None)
def _spi_script():
    return Compiled(Netlist.from_verilog(text=cosim.spi_master_verilog(0x000123))).flatten(1)


class _Cosim:
    def __init__(self, c, seed):
        rng = np.random.default_rng(_seed32(seed))
        self.c = c
        sched = cosim.MultiClockScheduler([cosim.ClockTiming(5000)])
        if c["gates"] == 0:
            s = _spi_script()
            ins, outs = s.netlist.ports()
            inbit = {n: s.input_map[p] for n, p, _ in ins}
            outbit = {n: s.output_map[lit] for n, lit in outs if lit > 1}
            nc = cosim.NC
            pins = cosim.FlashPins(clk_out=outbit["flash_clk"], csn_out=outbit["flash_csn"],
                                   d_out=(outbit["flash_d0"], nc, nc, nc),
                                   d_in=(nc, inbit["miso"], nc, nc))
            image = bytes(rng.integers(0, 256, 1 << 12, dtype=np.uint8))
            more = dict(reset_pos=inbit["rst"], reset_active=1, reset_edges=8, flash_pins=pins,
                        flash_image=image)
        else:
            s, _ = _design(c)
            data, _ = stimulus.input_roles(s)
            more = dict(constants=[(int(p), int(v)) for p, v in
                                   zip(data, rng.integers(0, 2, len(data)))])
        doms = [d for _, d in cosim.clock_domains_of(s)]
        self.r = cosim.Cosim(s, sched, doms, **more)

    def run(self):
        trace = self.r.run(self.c["edges"], batch=self.c["batch"], trace=True)
        return {"trace": trace, "states": self.r.states}


class _Changes:
    def __init__(self, c, seed):
        scan = _Scan(dict(c, kind="scan"), seed)
        scan.run()
        self.s, self.states = scan.s, scan.states
        rio = self.s.reg_io_state_size
        self.times = [(k * rio, 1000 * k) for k in range(c["cycles"] + 1)]
        # the program's own store of the run's records, as many as there can be
        self.records = np.zeros((c["cycles"] + 1) * len(vcd.output_mapping(self.s)), np.uint32)

    def run(self):
        counts, records = vcd.output_changes_device(self.s, self.states, self.times)
        self.records[:records.size] = records
        return {"counts": counts, "records": self.records}


def _mlp_inputs(c, seed):
    rng = np.random.default_rng(_seed32(seed))
    x = rng.standard_normal((c["n"], c["features"])).astype(np.float32)
    w = rng.standard_normal(c["features"]) / np.sqrt(c["features"])
    t = (np.tanh(x @ w) + 0.1 * rng.standard_normal(c["n"])).astype(np.float32)
    params = costmodel.he_init(c["features"], c["h1"], c["h2"], seed=_seed32(seed))
    return x, t, params


class _Mlp:
    LR = 0.05

    def __init__(self, c, seed):
        x, t, params = _mlp_inputs(c, seed)
        self.n, self.train = c["n"], c["kind"] == "mlp_train"
        self.m = costmodel.MLP(params=params, i=c["features"], h1=c["h1"], h2=c["h2"])
        self.x = torch.from_numpy(x).cuda()
        self.t = torch.from_numpy(t).cuda()
        self.y = torch.zeros(self.n, device="cuda")
        self.loss = torch.zeros(1, device="cuda")
        self.ws = torch.zeros(int(N.hip().jq_mlp_workspace_floats(
            c["features"], c["h1"], c["h2"], self.n)), device="cuda")

    def run(self):
        if self.train:
            self.m.train_step_raw(self.x, self.t, self.n, self.LR, self.ws, self.loss)
            return {"params": self.m.params, "grads": self.m.grads, "loss": self.loss}
        self.m.forward_raw(self.x, self.n, self.y)
        return {"y": self.y}


_KINDS = {"scan": _Scan, "lanes": _Lanes, "cosim": _Cosim, "changes": _Changes,
          "mlp_train": _Mlp, "mlp_forward": _Mlp}


def prepare(case, seed):
    return _KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------- work

def work(case):
    """Bytes: the program once, every snapshot or lane state the pass writes
    and the stimulus it reads.  Operations: one per gate, lane and cycle."""
    c, kind = case, case["kind"]
    if kind in ("mlp_train", "mlp_forward"):
        i, h1, h2, n = c["features"], c["h1"], c["h2"], c["n"]
        np_ = h1 * i + h1 + h2 * h1 + 2 * h2 + 1
        mac = i * h1 + h1 * h2 + h2
        if kind == "mlp_train":
            return {"bytes": 4 * (n * (i + 1) + 3 * np_), "flops": 2 * n * (3 * mac - i * h1)}
        return {"bytes": 4 * (n * (i + 1) + np_), "flops": 2 * n * mac}
    s = _spi_script() if kind == "cosim" and c["gates"] == 0 else _design(c)[0]
    gates = int(s.netlist.counts()["num_and"])
    ss, script = s.effective_state_size(), 4 * int(s.blocks_start[-1])
    if kind == "scan":
        return {"bytes": script + 4 * ss * (c["cycles"] + 1), "flops": gates * c["cycles"]}
    if kind == "cosim":
        return {"bytes": script + 8 * ss * c["edges"], "flops": gates * c["edges"]}
    if kind == "changes":
        bits = len(vcd.output_mapping(s))
        return {"bytes": (c["cycles"] + 1) * bits // 8 * (2 if c.get("xprop") else 1),
                "flops": (c["cycles"] + 1) * bits}
    cycles = c["lanes"] * (c["cycles_lo"] + c["cycles_hi"]) // 2
    state = 4 * 32 * s.reg_io_state_size * c["groups"]
    return {"bytes": script + 2 * state + 4 * cycles * len(s.input_layout) // 32,
            "flops": gates * cycles}


# ---------------------------------------------------------------- exact

def exact(case, seed):
    """The cost model in 64 bits; every other output is bits, not numbers."""
    c = case
    if c["kind"] not in ("mlp_train", "mlp_forward"):
        return None
    x, t, p = (a.astype(np.float64) for a in _mlp_inputs(c, seed))
    i, h1, h2, n = c["features"], c["h1"], c["h2"], c["n"]
    cut = np.cumsum([h1 * i, h1, h2 * h1, h2, h2])
    w1, b1, w2, b2, w3, b3 = np.split(p, cut)
    w1, w2 = w1.reshape(h1, i), w2.reshape(h2, h1)
    a1 = np.maximum(x @ w1.T + b1, 0)
    a2 = np.maximum(a1 @ w2.T + b2, 0)
    y = a2 @ w3 + b3[0]
    if c["kind"] == "mlp_forward":
        return {"y": y}
    dy = 2 * (y - t) / n
    d2 = np.where(a2 > 0, dy[:, None] * w3, 0)
    d1 = np.where(a1 > 0, d2 @ w2, 0)
    g = np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ a1).ravel(), d2.sum(0),
                        a2.T @ dy, [dy.sum()]])
    lr = float(np.float32(_Mlp.LR))
    return {"params": p - lr * g, "grads": g, "loss": np.array([np.mean((y - t) ** 2)])}

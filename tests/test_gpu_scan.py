"""Parity of the plain drop-in kernel (through the C ABI) with the CPU oracle.

Every snapshot of every cycle must be bit-identical to the oracle's
kernel-semantics run; the final values are also checked against the direct
AIG simulation, which does not look at the script at all."""
import numpy as np
import pytest

import oracle
from helpers import CONFIG1, design, direct_check
from jacquard_amd import sim, stimulus

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


class _sync_mode:
    """Sets the value-only scan launches' synchronisation (1: dataflow, the
    default; 0: grid barriers) for the duration of a with-block."""

    def __init__(self, mode):
        from jacquard_amd import _native as N
        self.L, self.mode = N.hip(), mode

    def __enter__(self):
        self.prev = self.L.jq_scan_sync_mode(self.mode)

    def __exit__(self, *exc):
        self.L.jq_scan_sync_mode(self.prev)


@pytest.mark.parametrize("num_blocks,split", [(1, 0), (8, 0), (16, 6), (64, 4)])
def test_config1_2state(num_blocks, split):
    nl, comp = design("c1", level_split=split, **CONFIG1)
    s = comp.flatten(num_blocks)
    cycles = 300
    _say("config1", num_blocks, split, "parts", s.num_parts)
    st = stimulus.build_states(s, cycles, seed=11, p=0.5)
    ref = st.copy()
    oracle.run(s, ref, cycles)
    got = sim.run_scan(s, st.copy(), cycles)["states"]
    assert np.array_equal(got, ref)
    direct_check(s, got, cycles, 11, 0.5)


@pytest.mark.parametrize("num_blocks", [128, 200])
@pytest.mark.parametrize("sync", [0, 1])
def test_many_blocks_hierarchical_barrier(num_blocks, sync):
    """At 128 workgroups or more the grid barrier counts arrivals through
    eight sub-counters; most blocks here are empty and still take part
    (sync 0).  With dataflow synchronisation (sync 1) the empty blocks
    publish progress that nobody waits for."""
    from jacquard_amd.netlist import Netlist
    from jacquard_amd.script import Compiled
    nl = Netlist.random(seed=5, gates=20000, depth=40, dffs=1024, inputs=64, outputs=32,
                        geometric_p=0.3, invert_prob=0.5)
    # small partitions: about ten per major stage, spread over the blocks
    s = Compiled(nl, level_split=4, max_part_nodes=500).flatten(num_blocks)
    cycles = 150
    _say("blocks", num_blocks, "major", s.num_major_stages, "parts", s.num_parts)
    st = stimulus.build_states(s, cycles, seed=21, p=0.3)
    ref = st.copy()
    oracle.run(s, ref, cycles)
    with _sync_mode(sync):
        got = sim.run_scan(s, st.copy(), cycles)["states"]
    assert np.array_equal(got, ref)


def test_reference_symbol_entry_point():
    nl, comp = design("c1", level_split=6, **CONFIG1)
    s = comp.flatten(16)
    cycles = 100
    st = stimulus.build_states(s, cycles, seed=12, p=0.3)
    ref = st.copy()
    oracle.run(s, ref, cycles)
    got = sim.run_scan(s, st.copy(), cycles, reference_symbols=True)["states"]
    assert np.array_equal(got, ref)


def test_srams_and_major_stages():
    nl, comp = design("sram", level_split=8, seed=4, gates=30000, depth=48,
                      dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=4)
    s = comp.flatten(32)
    cycles = 120
    _say("sram", s.num_parts, s.num_major_stages, s.sram_storage_size)
    st = stimulus.build_states(s, cycles, seed=13, p=0.2)
    ref = st.copy()
    sram_ref = np.zeros(s.sram_storage_size, np.uint32)
    oracle.run(s, ref, cycles, sram=sram_ref)
    out = sim.run_scan(s, st.copy(), cycles)
    assert np.array_equal(out["states"], ref)
    assert np.array_equal(out["sram"][:s.sram_storage_size], sram_ref)
    direct_check(s, out["states"], cycles, 13, 0.2)


@pytest.mark.parametrize("frac", [0.0, 0.1])
def test_xprop(frac):
    nl, comp = design("xp", level_split=8, seed=5, gates=20000, depth=40,
                      dffs=2000, inputs=64, outputs=32, geometric_p=0.3, srams=2)
    s = comp.flatten(16, xprop=True)
    cycles = 80
    m, pick = stimulus.dff_initial_xmask(s, frac, seed=7)
    st = stimulus.build_states(s, cycles, seed=14, p=0.4, initial_xmask=m)
    ref = st.copy()
    sram = np.zeros(s.sram_storage_size, np.uint32)
    sram_x = np.full(s.sram_storage_size, 0xFFFFFFFF, np.uint32)
    oracle.run(s, ref, cycles, sram=sram, sram_x=sram_x)
    out = sim.run_scan(s, st.copy(), cycles)
    assert np.array_equal(out["states"], ref)
    assert np.array_equal(out["sram_x"][:s.sram_storage_size], sram_x)


@pytest.mark.parametrize("xprop", [False, True])
def test_dataflow_and_barrier_sync_agree(xprop):
    """Value-only launches wait only for the blocks whose words the next
    major stage reads (each up to the stage that wrote them) instead of
    taking a grid barrier.  Both schedules must give the oracle's bits:
    every snapshot, the SRAM contents and their X shadow."""
    from jacquard_amd import _native as N
    assert N.hip().jq_scan_sync_mode(-1) == 1, "dataflow is the default"
    nl, comp = design("sync", level_split=4, seed=9, gates=40000, depth=48,
                      dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=3)
    s = comp.flatten(48, xprop=xprop)
    cycles = 100
    _say("sync modes", xprop, s.num_blocks, s.num_major_stages, s.num_parts)
    m = None
    if xprop:
        m, _pick = stimulus.dff_initial_xmask(s, 0.1, seed=8)
    st = stimulus.build_states(s, cycles, seed=15, p=0.3, initial_xmask=m)
    ref = st.copy()
    sram = np.zeros(s.sram_storage_size, np.uint32)
    sram_x = np.full(s.sram_storage_size, 0xFFFFFFFF, np.uint32)
    oracle.run(s, ref, cycles, sram=sram, sram_x=sram_x if xprop else None)
    for mode in (1, 0):
        with _sync_mode(mode):
            out = sim.run_scan(s, st.copy(), cycles)
        assert np.array_equal(out["states"], ref), mode
        assert np.array_equal(out["sram"][:s.sram_storage_size], sram), mode
        if xprop:
            assert np.array_equal(out["sram_x"][:s.sram_storage_size], sram_x), mode


@pytest.mark.parametrize("cycles", [1, 7, 8, 9])
def test_launch_lengths_around_the_dataflow_threshold(cycles):
    """Launches shorter than 8 cycles keep grid barriers; from 8 cycles on
    the producer table is built.  Both sides of the threshold, on a
    multi-block script with SRAMs, give the oracle's snapshots and SRAMs."""
    nl, comp = design("sync", level_split=4, seed=9, gates=40000, depth=48,
                      dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=3)
    s = comp.flatten(48)
    st = stimulus.build_states(s, cycles, seed=16, p=0.3)
    ref = st.copy()
    sram = np.zeros(s.sram_storage_size, np.uint32)
    oracle.run(s, ref, cycles, sram=sram)
    out = sim.run_scan(s, st.copy(), cycles)
    assert np.array_equal(out["states"], ref)
    assert np.array_equal(out["sram"][:s.sram_storage_size], sram)


def test_more_major_stages_than_the_dataflow_table_holds():
    """One logic level per major stage on a depth-140 netlist gives more
    than 120 major stages: the launch keeps grid barriers and stays exact."""
    nl, comp = design("deep", level_split=1, seed=12, gates=6000, depth=140,
                      dffs=256, inputs=32, outputs=16, geometric_p=0.3)
    s = comp.flatten(8)
    assert s.num_major_stages > 120
    cycles = 20
    _say("deep", s.num_major_stages, s.num_parts)
    st = stimulus.build_states(s, cycles, seed=17, p=0.3)
    ref = st.copy()
    oracle.run(s, ref, cycles)
    got = sim.run_scan(s, st.copy(), cycles)["states"]
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("sync", [0, 1])
def test_wait_time_out_aborts_the_launch_and_the_next_launch_is_exact(sync):
    """The time-out path, forced from the host: with a one-poll bound nearly
    every wait gives up, the first one marks the launch aborted, every
    workgroup leaves at its next wait, and the launch ends promptly with the
    device flag raised (run_scan raises and clears it).  With the bound
    restored the next launch of the same script matches the oracle."""
    import time
    from jacquard_amd import _native as N
    L = N.hip()
    nl, comp = design("sync", level_split=4, seed=9, gates=40000, depth=48,
                      dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=3)
    s = comp.flatten(48)
    cycles = 200
    st = stimulus.build_states(s, cycles, seed=18, p=0.3)
    ref = st.copy()
    oracle.run(s, ref, cycles)
    with _sync_mode(sync):
        prev = L.jq_wait_limit(1)
        try:
            t = time.time()
            with pytest.raises(RuntimeError, match="timed out"):
                sim.run_scan(s, st.copy(), cycles)
            _say("aborted launch ended in", time.time() - t, "s")
            assert time.time() - t < 30
        finally:
            assert L.jq_wait_limit(prev) == 1
        got = sim.run_scan(s, st.copy(), cycles)["states"]
    assert np.array_equal(got, ref)


def test_captured_launch_replays_match_the_oracle():
    """A value-only launch through jq_simulate_scan captured into a hipGraph
    on a side stream: under capture it is an ordinary kernel node with grid
    barriers (no dataflow table is built into the graph).  Before each of
    three replays the snapshot buffer gets its input back, with a junk
    pattern in every word the launch writes (a replay that skipped a word
    would show it), the SRAMs are cleared, and an eager launch of another
    script runs; every replay reproduces the oracle's snapshots and SRAM
    contents, and no wait times out."""
    import ctypes
    import torch
    from jacquard_amd import _native as N
    L = N.hip()
    nl, comp = design("cap", level_split=4, seed=9, gates=40000, depth=48,
                      dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=3)
    s = comp.flatten(48)
    cycles = 60
    ss = s.effective_state_size()
    st = stimulus.build_states(s, cycles, seed=19, p=0.3)
    ref = st.copy()
    sram_ref = np.zeros(s.sram_storage_size, np.uint32)
    oracle.run(s, ref, cycles, sram=sram_ref)
    # the launch's input: snapshot 0 and the pre-filled primary inputs, and
    # a junk pattern in every writeout word of snapshots 1.. (the words
    # past the inputs' n // 32 + 1), which each cycle rewrites in full
    ws = len(s.input_layout) // 32 + 1
    inp = st.copy().reshape(cycles + 1, ss)
    inp[1:, ws:] = 0xA5C3F00D
    inp = inp.reshape(-1)
    d_bs = sim.to_device(np.ascontiguousarray(s.blocks_start, np.uint64))
    d_bd = sim.to_device(np.ascontiguousarray(s.blocks_data, np.uint32))
    d_in = sim.to_device(inp)
    d_st = d_in.clone()
    d_sram = torch.zeros(s.sram_storage_size, dtype=torch.int32, device="cuda")
    d_sx = torch.zeros(1, dtype=torch.int32, device="cuda")
    _, small = design("c1", level_split=0, **CONFIG1)
    s2 = small.flatten(8)
    st2 = stimulus.build_states(s2, 50, seed=3, p=0.5)
    ref2 = st2.copy()
    oracle.run(s2, ref2, 50)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            rc = L.jq_simulate_scan(
                s.num_blocks, s.num_major_stages, d_bs.data_ptr(), d_bd.data_ptr(),
                d_sram.data_ptr(), d_sx.data_ptr(), cycles, ss, d_st.data_ptr(),
                None, None, 0, 0, ctypes.c_void_p(side.cuda_stream))
    torch.cuda.current_stream().wait_stream(side)
    N.check(rc)
    for k in range(3):
        d_st.copy_(d_in)
        d_sram.zero_()
        assert np.array_equal(sim.run_scan(s2, st2.copy(), 50)["states"], ref2)
        _say("replay", k)
        g.replay()
        torch.cuda.synchronize()
        assert not sim.device_error(), f"replay {k}: a wait timed out"
        assert np.array_equal(sim.from_device(d_st, np.uint32), ref), f"replay {k}"
        assert np.array_equal(sim.from_device(d_sram, np.uint32), sram_ref), f"replay {k}"


def test_timing_events():
    nl, comp = design("tm", level_split=6, seed=6, gates=8000, depth=30,
                      dffs=800, inputs=32, outputs=16, geometric_p=0.3)
    d = np.zeros(nl.counts()["num_pins"] + 1, np.uint16)
    rng = np.random.default_rng(1)
    A = nl.arrays()
    ands = A["drv"] == 1
    d[ands] = rng.integers(20, 201, ands.sum())
    nl.set_delays(d)
    s = comp.flatten(16)
    s.inject_timing()
    s.enable_timing_arrivals()
    cons = s.build_timing_constraint_buffer(190, 50, 20)
    cycles = 60
    st = stimulus.build_states(s, cycles, seed=15, p=0.5)
    ref = st.copy()
    ev_ref, n_ref = oracle.run(s, ref, cycles, constraints=cons,
                               arrival_state_offset=s.arrival_state_offset,
                               event_capacity=1 << 20)
    out = sim.run_scan(s, st.copy(), cycles, constraints=cons,
                       event_capacity=1 << 20)
    assert np.array_equal(out["states"], ref)
    assert out["event_count"] == n_ref and n_ref > 0
    a = sim.canonical_events(out["events"])
    b = sim.canonical_events(ev_ref)
    assert np.array_equal(a, b)


def test_timed_reference_symbol_keeps_1024_events():
    """simulate_v1_noninteractive_timed_hip keeps the reference buffer's
    1024 records (csrc/event_buffer.h:99-111): the header counts every
    violation, sets the overflow flag, and the kept records are violations
    of the full list."""
    nl, comp = design("tm", level_split=6, seed=6, gates=8000, depth=30,
                      dffs=800, inputs=32, outputs=16, geometric_p=0.3)
    d = np.zeros(nl.counts()["num_pins"] + 1, np.uint16)
    rng = np.random.default_rng(1)
    A = nl.arrays()
    ands = A["drv"] == 1
    d[ands] = rng.integers(20, 201, ands.sum())
    nl.set_delays(d)
    s = comp.flatten(16)
    s.inject_timing()
    s.enable_timing_arrivals()
    cons = s.build_timing_constraint_buffer(190, 50, 20)
    cycles = 60
    st = stimulus.build_states(s, cycles, seed=15, p=0.5)
    ref = st.copy()
    ev_ref, n_ref = oracle.run(s, ref, cycles, constraints=cons,
                               arrival_state_offset=s.arrival_state_offset,
                               event_capacity=1 << 20)
    assert n_ref > 1024
    out = sim.run_scan(s, st.copy(), cycles, constraints=cons, reference_symbols=True)
    assert np.array_equal(out["states"], ref)
    assert out["event_count"] == n_ref and out["overflow"] == 1
    kept = sim.canonical_events(out["events"])
    assert len(kept) == 1024
    full = {bytes(e) for e in sim.canonical_events(ev_ref)}
    assert all(bytes(e) in full for e in kept)


def test_xprop_timing_srams_together():
    """X lane, arrivals, setup/hold and SRAMs in one run (the 4M-gate
    workload's feature mix at test size)."""
    nl, comp = design("xts", level_split=6, seed=9, gates=40000, depth=48,
                      dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=2,
                      delay=(20, 200))
    s = comp.flatten(24, xprop=True)
    s.inject_timing()
    s.enable_timing_arrivals()
    cons = s.build_timing_constraint_buffer(1500, 50, 20)
    cycles = 60
    m, _ = stimulus.dff_initial_xmask(s, 0.1, seed=8)
    st = stimulus.build_states(s, cycles, seed=16, p=0.3, initial_xmask=m)
    ref = st.copy()
    sram = np.zeros(s.sram_storage_size, np.uint32)
    sram_x = np.full(s.sram_storage_size, 0xFFFFFFFF, np.uint32)
    ev_ref, n_ref = oracle.run(s, ref, cycles, sram=sram, sram_x=sram_x, constraints=cons,
                               arrival_state_offset=s.arrival_state_offset,
                               event_capacity=1 << 20)
    out = sim.run_scan(s, st.copy(), cycles, constraints=cons, event_capacity=1 << 20)
    _say("xts", s.num_parts, s.num_major_stages, "events", n_ref)
    assert np.array_equal(out["states"], ref)
    assert np.array_equal(out["sram"][:s.sram_storage_size], sram)
    assert np.array_equal(out["sram_x"][:s.sram_storage_size], sram_x)
    assert out["event_count"] == n_ref and n_ref > 0
    assert np.array_equal(sim.canonical_events(out["events"]), sim.canonical_events(ev_ref))


@pytest.mark.parametrize("xprop", [False, True])
def test_device_output_changes_match_host_writer(xprop):
    """VCD text from device change records equals the host writer's text
    from the full snapshots (values and X), on a random design with many
    outputs and skipped timestamps."""
    from jacquard_amd import vcd
    nl, comp = design("xp", level_split=8, seed=5, gates=20000, depth=40,
                      dffs=2000, inputs=64, outputs=32, geometric_p=0.3, srams=2)
    s = comp.flatten(16, xprop=xprop)
    cycles = 70
    m = stimulus.dff_initial_xmask(s, 0.2, seed=3)[0] if xprop else None
    st = stimulus.build_states(s, cycles, seed=17, p=0.4, initial_xmask=m)
    out = sim.run_scan(s, st.copy(), cycles, return_device=True)
    rio, ess = s.reg_io_state_size, s.effective_state_size()
    offs = [((k + 1) * rio, vcd.U64_MAX if k % 7 == 3 else 10 * k) for k in range(cycles)]
    S = out["states"].reshape(-1, ess)
    values = np.ascontiguousarray(S[:, :rio]).reshape(-1)
    xm = np.ascontiguousarray(S[:, rio:2 * rio]).reshape(-1) if xprop else None
    host = vcd.write_output_vcd(s, offs, values, xmask_states=xm)
    cnt, rec = vcd.output_changes_device(s, out["device"]["states"], offs)
    dev = vcd.write_output_vcd_changes(s, offs, cnt, rec)
    assert dev == host
    assert len(rec) < S[1:].size  # compacted: far fewer words than snapshots


def test_tune_plain_chooses_a_fitting_width_that_stays_exact():
    """The measured partition-width choice only changes how the netlist is
    cut: whatever cap it keeps, the script fits the co-resident workgroups
    and simulates bit-exactly."""
    from jacquard_amd.netlist import Netlist
    nl = Netlist.random(seed=5, gates=20000, depth=40, dffs=1024, inputs=64, outputs=32,
                        geometric_p=0.3, invert_prob=0.5)
    comp, s, table = sim.tune_plain(nl, 4, caps=(2600, 400, 200), trial_cycles=20)
    _say("tune table", table)
    assert any(r["fits"] for r in table)
    assert s.num_blocks == max(comp.parts_per_stage())
    cycles = 60
    st = stimulus.build_states(s, cycles, seed=31, p=0.3)
    ref = st.copy()
    oracle.run(s, ref, cycles)
    got = sim.run_scan(s, st.copy(), cycles)["states"]
    assert np.array_equal(got, ref)


def test_scan_profiled_samples_every_partition_and_keeps_values():
    """jq_simulate_scan_profiled writes a positive tick count for every
    partition execution of the sampled cycles and simulates exactly like the
    unprofiled kernel."""
    from jacquard_amd import costmodel as CM
    nl, comp = design("c1", level_split=6, **CONFIG1)
    s = comp.flatten(8)
    cycles, sampled = 40, 10
    st = stimulus.build_states(s, cycles, seed=41, p=0.4)
    ref = st.copy()
    oracle.run(s, ref, cycles)
    d = sim.to_device(st.copy())
    ticks = CM.profile_partitions(s, d, cycles, sampled)
    assert np.array_equal(d.cpu().numpy().view(np.uint32), ref)
    assert ticks.shape == (sampled, s.num_parts)
    assert (ticks > 0).all()


@pytest.mark.parametrize("xprop", [False, True])
def test_global_read_wider_than_prefetched_rounds(xprop):
    """Scripts whose global read needs more rounds than the kernel prefetches
    (up to 32 single-bit rounds per thread here): the extra rounds are read
    after the prefetched ones, with the X lane when X-capable."""
    from helpers import OneBitRounds
    from jacquard_amd.netlist import Netlist
    from jacquard_amd.script import Compiled
    nl = Netlist.random(seed=5, gates=20000, depth=40, dffs=1024, inputs=64, outputs=32,
                        geometric_p=0.3, invert_prob=0.5)
    s = Compiled(nl, level_split=4, max_part_nodes=500).flatten(8, xprop=xprop)
    w = OneBitRounds(s)
    _say("xprop", xprop, "max rounds", w.max_rounds)
    assert w.max_rounds > 16
    cycles = 60
    st = stimulus.build_states(s, cycles, seed=33, p=0.3)
    ref = st.copy()
    oracle.run(s, ref, cycles)  # the original script: same values
    got = sim.run_scan(w, st.copy(), cycles)["states"]
    assert np.array_equal(got, ref)


class _WideState:
    """The script over a snapshot of `extra` more words, with every global
    read of input word 0 sent to the word after the last writeout instead:
    a word past the first writeout that no partition writes."""

    def __init__(self, script, extra):
        self._s, self.extra = script, extra
        bd = np.array(script.blocks_data, np.uint32)
        self.moved = 0
        for off in script.parts[:, 3].tolist():
            a, R = int(off) + 256, int(bd[int(off) + 6])
            gr = bd[a:a + 512 * R].reshape(-1, 2)
            hit = ((gr[:, 0] & 0x7FFFFFFF) == 0) & (gr[:, 1] != 0)
            gr[hit, 0] = (gr[hit, 0] & 0x80000000) | script.reg_io_state_size
            self.moved += int(hit.sum())
        self.blocks_data = bd

    def effective_state_size(self):
        return self._s.effective_state_size() + self.extra

    def __getattr__(self, name):
        return getattr(self._s, name)


def test_a_script_that_reads_past_the_writeouts_keeps_grid_barriers():
    """A read past the first writeout word of a word that no partition
    writes would wait for ever in the exchange ring: the builders see it and
    the launch keeps grid barriers, with the oracle's snapshots."""
    nl, comp = design("sync", level_split=4, seed=9, gates=40000, depth=48,
                      dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=3)
    w = _WideState(comp.flatten(48), 2)
    assert w.moved > 0
    cycles = 60
    rio = w.reg_io_state_size
    st = np.zeros((cycles + 1, rio + 2), np.uint32)
    st[:, :rio] = stimulus.build_states(w._s, cycles, seed=20, p=0.3).reshape(cycles + 1, rio)
    st[:, rio] = st[:, 0]
    st = st.reshape(-1)
    ref = st.copy()
    oracle.run(w, ref, cycles)
    got = sim.run_scan(w, st.copy(), cycles, validate=False)["states"]
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("blocks", [1, 48])
def test_x_masks_at_offset_0_keep_grid_barriers(blocks):
    """X-capable partitions whose masks lie on the words themselves: the
    launch without the X lane must not take them for partitions without X."""
    nl, comp = design("sync", level_split=4, seed=9, gates=8000, depth=24,
                      dffs=800, inputs=64, outputs=32, geometric_p=0.3)
    s = comp.flatten(blocks, xprop=True)
    bd = np.array(s.blocks_data, np.uint32)
    capable = 0
    for off in s.parts[:, 3].tolist():
        if bd[int(off) + 8]:
            bd[int(off) + 9] = 0
            capable += 1
    assert capable > 0

    class Script:
        blocks_data = bd

        def __getattr__(self, name):
            return getattr(s, name)

    cycles = 40
    st = stimulus.build_states(s, cycles, seed=21, p=0.3)
    got = []
    for mode in (0, 1):
        with _sync_mode(mode):
            got.append(sim.run_scan(Script(), st.copy(), cycles, validate=False)["states"])
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("blocks,xprop", [(3, True), (1, False), (61, True)])
def test_dataflow_over_many_laps_of_the_ring(blocks, xprop):
    """300 cycles, 37 laps of the exchange ring, with one block, with fewer
    blocks than partitions and with more: every snapshot is the oracle's."""
    from jacquard_amd.script import Compiled
    nl, _ = design("laps", level_split=3, seed=23, gates=9000, depth=30, dffs=700,
                   inputs=40, outputs=24, geometric_p=0.3, srams=2)
    s = Compiled(nl, level_split=3, max_level_nodes=200).flatten(blocks, xprop=xprop)
    cycles = 300
    st = stimulus.build_states(s, cycles, seed=4, p=0.2)
    ref = st.copy()
    sram = np.zeros(s.sram_storage_size, np.uint32)
    sram_x = np.full(s.sram_storage_size, 0xFFFFFFFF, np.uint32)
    oracle.run(s, ref, cycles, sram=sram, sram_x=sram_x if xprop else None)
    out = sim.run_scan(s, st.copy(), cycles)
    assert np.array_equal(out["states"], ref)
    assert np.array_equal(out["sram"][:s.sram_storage_size], sram)


class _SplitRounds:
    """The script with every global-read mask split into masks of at most
    `bits` bits, in the order the pext takes them, as more rounds of the same
    words: what a partition computes stays the same."""

    def __init__(self, script, bits):
        self._s = script
        bd = np.asarray(script.blocks_data, np.uint32)
        starts = np.asarray(script.blocks_start, np.uint64)
        pieces, new_starts, self.rounds = [], [0], set()
        for k in range(len(starts) - 1):
            pos, end = int(starts[k]), int(starts[k + 1])
            while pos < end:
                ns, last, R = int(bd[pos]), int(bd[pos + 1]), int(bd[pos + 6])
                if ns == 0:
                    pieces.append(bd[pos:end])
                    break
                gr = bd[pos + 256:pos + 256 + 512 * R].reshape(R, 256, 2)
                split = [[] for _ in range(256)]
                for r in range(R):
                    for t in range(256):
                        w, m = int(gr[r, t, 0]), int(gr[r, t, 1])
                        while m:
                            part = 0
                            for _ in range(bits):
                                part |= m & -m
                                m &= m - 1
                            split[t].append((w, part))
                n = max(len(q) for q in split)
                self.rounds.add(n)
                new = np.zeros((n, 256, 2), np.uint32)
                for t, q in enumerate(split):
                    new[:len(q), t] = np.array(q, np.uint32).reshape(-1, 2)
                head = bd[pos:pos + 256].copy()
                head[6] = n
                tail = pos + 256 + 512 * R
                pos = tail + 5120 * (ns + 2)
                pieces += [head, new.reshape(-1), bd[tail:pos]]
                if last:
                    pieces.append(bd[pos:end])
                    break
            new_starts.append(sum(len(p) for p in pieces))
        pieces.append(bd[int(starts[-1]):])
        self.blocks_data = np.concatenate(pieces)
        self.blocks_start = np.array(new_starts, np.uint64)

    def __getattr__(self, name):
        return getattr(self._s, name)


@pytest.mark.parametrize("blocks,xprop,bits,rounds", [
    (24, False, 32, (1, 7)), (24, True, 2, (8, 16)), (24, False, 1, (17, 31)),
    (1, False, 2, (8, 16)), (1, True, 1, (17, 31))])
def test_composed_permutations(blocks, xprop, bits, rounds):
    """Launches long enough to compose the first stage's permutations, over
    partitions of few rounds, of more than 16-bit indexes reach and of more
    than are prefetched (test_global_read_wider_than_prefetched_rounds has
    some that are not composed), with a few partitions to a block and with
    more in the one block than the table has slots; and a launch too short
    for a table."""
    nl, _ = design("laps", level_split=3, seed=23, gates=9000, depth=30, dffs=700,
                   inputs=40, outputs=24, geometric_p=0.3, srams=2)
    from jacquard_amd.script import Compiled
    s = Compiled(nl, level_split=3, max_part_nodes=150).flatten(blocks, xprop=xprop)
    w = _SplitRounds(s, bits)
    _say("rounds", sorted(w.rounds), "partitions", s.num_parts, "stages", s.num_major_stages)
    assert rounds[0] <= max(w.rounds) <= rounds[1]
    if blocks == 1:
        assert s.num_parts > 8 * s.num_major_stages
    for cycles in (7, 20):
        st = stimulus.build_states(s, cycles, seed=4, p=0.2)
        ref = st.copy()
        sram = np.zeros(s.sram_storage_size, np.uint32)
        sram_x = np.full(s.sram_storage_size, 0xFFFFFFFF, np.uint32)
        oracle.run(s, ref, cycles, sram=sram, sram_x=sram_x if xprop else None)
        out = sim.run_scan(w, st.copy(), cycles, validate=False)
        assert np.array_equal(out["states"], ref)
        assert np.array_equal(out["sram"][:s.sram_storage_size], sram)


@pytest.mark.parametrize("xprop", [False, True])
@pytest.mark.parametrize("cycles", [7, 60])
def test_timing_launches_in_both_sync_modes(xprop, cycles):
    """Setup/hold launches exchange their words through the ring (short ones
    and mode 0: grid barriers), masks beside the words under X: snapshots with
    arrivals, SRAMs and the set of events are the oracle's."""
    nl, comp = design("xts", level_split=6, seed=9, gates=40000, depth=48,
                      dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=2,
                      delay=(20, 200))
    s = comp.flatten(24, xprop=xprop)
    s.inject_timing()
    s.enable_timing_arrivals()
    cons = s.build_timing_constraint_buffer(1500, 50, 20)
    m = stimulus.dff_initial_xmask(s, 0.1, seed=8)[0] if xprop else None
    st = stimulus.build_states(s, cycles, seed=16, p=0.3, initial_xmask=m)
    ref = st.copy()
    sram = np.zeros(s.sram_storage_size, np.uint32)
    sram_x = np.full(s.sram_storage_size, 0xFFFFFFFF, np.uint32)
    ev_ref, n_ref = oracle.run(s, ref, cycles, sram=sram, sram_x=sram_x if xprop else None,
                               constraints=cons, arrival_state_offset=s.arrival_state_offset,
                               event_capacity=1 << 20)
    for mode in (1, 0):
        with _sync_mode(mode):
            out = sim.run_scan(s, st.copy(), cycles, constraints=cons, event_capacity=1 << 20)
        assert np.array_equal(out["states"], ref), mode
        assert np.array_equal(out["sram"][:s.sram_storage_size], sram), mode
        assert out["event_count"] == n_ref and n_ref > 0
        assert np.array_equal(sim.canonical_events(out["events"]), sim.canonical_events(ev_ref))


@pytest.mark.parametrize("kw,cycles", [
    (dict(seed=3, gates=300, depth=9, dffs=40, inputs=5, outputs=7), 9),
    (dict(seed=4, gates=6000, depth=20, dffs=900, inputs=40, outputs=24, srams=3), 61),
    # more than 512 words of primary inputs; no flip-flops
    (dict(seed=5, gates=30000, depth=12, dffs=300, inputs=17000, outputs=32), 12),
    (dict(seed=6, gates=2000, depth=14, dffs=0, inputs=70, outputs=50), 8),
    # more state words than stay in LDS
    (dict(seed=7, gates=200000, depth=12, dffs=140000, inputs=40, outputs=24), 8)])
def test_one_block_keeps_its_state_in_lds(kw, cycles):
    """Launches of one block with a small state, beside one whose state is too
    large and one with X masks (both in the ring): every snapshot and SRAM word
    is the oracle's, in both sync modes."""
    from jacquard_amd.netlist import Netlist
    from jacquard_amd.script import Compiled
    nl = Netlist.random(geometric_p=0.3, invert_prob=0.4, **kw)
    comp = Compiled(nl, level_split=3)
    for xprop in (False, True):
        s = comp.flatten(1, xprop=xprop)
        _say("words", s.effective_state_size(), "partitions", s.num_parts)
        assert (s.effective_state_size() > 4095) == (kw["dffs"] > 100000) or xprop
        st = stimulus.build_states(s, cycles, seed=4, p=0.3)
        ref = st.copy()
        sram = np.zeros(s.sram_storage_size, np.uint32)
        sram_x = np.full(s.sram_storage_size, 0xFFFFFFFF, np.uint32)
        oracle.run(s, ref, cycles, sram=sram, sram_x=sram_x if xprop else None)
        for mode in (1, 0):
            with _sync_mode(mode):
                out = sim.run_scan(s, st.copy(), cycles)
            assert np.array_equal(out["states"], ref), (xprop, mode)
            assert np.array_equal(out["sram"][:s.sram_storage_size], sram), (xprop, mode)


def _stage_of_word(script):
    """{state word: major stage that writes it}."""
    bd = np.asarray(script.blocks_data, np.uint32)
    return {w: int(m) for m, _b, _i, off, _l in script.parts.tolist()
            for w in range(int(bd[int(off) + 3]), int(bd[int(off) + 3]) + int(bd[int(off) + 2]))}


@pytest.mark.parametrize("xprop", [False, True])
@pytest.mark.parametrize("blocks,capacity", [(1, 100), (24, 7), (24, 1024), (68, 1 << 20)])
def test_violations_come_in_the_order_of_the_stages(xprop, blocks, capacity):
    """In both sync modes the records lie in the buffer cycle by cycle and
    stage by stage, as a barrier after every stage brings them, and one that
    overflows has kept the earliest: every violation of a (cycle, stage)
    before that of its last record is there."""
    from jacquard_amd.script import Compiled
    nl, _ = design("xts", level_split=6, seed=9, gates=40000, depth=48,
                   dffs=3000, inputs=64, outputs=32, geometric_p=0.3, srams=2,
                   delay=(20, 200))
    s = Compiled(nl, level_split=6, max_part_nodes=400).flatten(blocks, xprop=xprop)
    s.inject_timing()
    s.enable_timing_arrivals()
    cons = s.build_timing_constraint_buffer(1000, 50, 20)
    cycles = 60
    stage = _stage_of_word(s)

    def when(events):
        return [(int(e["cycle"]), stage[int(e["data"][0])]) for e in events]

    st = stimulus.build_states(s, cycles, seed=16, p=0.3)
    ev_ref, n_ref = oracle.run(s, st.copy(), cycles, sram=np.zeros(s.sram_storage_size, np.uint32),
                               sram_x=np.full(s.sram_storage_size, 0xFFFFFFFF, np.uint32)
                               if xprop else None,
                               constraints=cons, arrival_state_offset=s.arrival_state_offset,
                               event_capacity=1 << 20)
    ref = when(ev_ref)
    full = {bytes(e) for e in sim.canonical_events(ev_ref)}
    assert n_ref == len(ref) > 1024 and len(set(ref)) > 100
    for mode in (1, 0):
        with _sync_mode(mode):
            out = sim.run_scan(s, st.copy(), cycles, constraints=cons, event_capacity=capacity)
        assert out["event_count"] == n_ref and out["overflow"] == (n_ref > capacity), mode
        kept = when(out["events"])
        assert len(kept) == min(n_ref, capacity)
        assert kept == sorted(kept), mode
        assert sum(k < kept[-1] for k in kept) == sum(k < kept[-1] for k in ref), mode
        assert all(bytes(e) in full for e in sim.canonical_events(out["events"])), mode


class _UnevenBlocks:
    """Block 0 runs ten partitions of 16 words a cycle, block 1 a single one;
    all of them read primary inputs only, so nothing but the launch's own
    rules holds block 1 back, and every word violates its hold limit in every
    cycle."""

    num_blocks, num_major_stages, sram_storage_size, xprop_enabled = 2, 1, 0, False
    inputs, per, slow = 256, 16, 10
    reg_io_state_size = arrival_state_offset = inputs + per * (slow + 1)

    def __init__(self):
        from handscripts import HDR, M, tree_probe_script
        rng = np.random.default_rng(3)
        zeros = np.zeros(256, np.uint32)
        parts = []
        for k in range(self.slow + 1):
            p = tree_probe_script(zeros, zeros, np.full(256, M, np.uint32),
                                  rng.integers(0, 300, 256), num_ios=self.per)[:-HDR]
            p[1] = k >= self.slow - 1  # the last of its block
            p[3] = self.inputs + self.per * k
            p[-1023::4] = M  # clock enables forced
            parts.append(p)
        n = parts[0].size
        self.blocks_start = np.array([0, n * self.slow, n * (self.slow + 1)], np.uint64)
        self.blocks_data = np.concatenate(parts + [np.zeros(2048, np.uint32)])

    def effective_state_size(self):
        return 2 * self.reg_io_state_size


@pytest.mark.parametrize("mode", [1, 0])
@pytest.mark.parametrize("symbol", [False, True])
def test_a_block_that_runs_ahead_records_no_violation_early(mode, symbol):
    """An event buffer of a few cycles' violations keeps those of the first
    cycles, of every block, as grid barriers do."""
    s = _UnevenBlocks()
    cycles, ss = 40, s.effective_state_size()
    rio, each = s.reg_io_state_size, s.per * (s.slow + 1)
    cons = np.zeros(1 + rio, np.uint32)
    cons[0] = 60000
    cons[1 + s.inputs:] = 0xFFFF
    st = np.zeros((cycles + 1, ss), np.uint32)
    st[:, :s.inputs] = np.random.default_rng(4).integers(0, 1 << 32, (cycles + 1, s.inputs))
    st = st.reshape(-1)
    ref = st.copy()
    _, n_ref = oracle.run(s, ref, cycles, constraints=cons, event_capacity=1 << 14,
                          arrival_state_offset=rio)
    assert n_ref == each * cycles
    capacity = 1024 if symbol else 5 * each
    with _sync_mode(mode):
        out = sim.run_scan(s, st.copy(), cycles, constraints=cons, event_capacity=capacity,
                           reference_symbols=symbol, validate=False)
    assert np.array_equal(out["states"], ref)
    assert out["event_count"] == n_ref and out["overflow"] == 1
    kept = [int(e["cycle"]) for e in out["events"]]
    assert kept == [k // each for k in range(capacity)]


@pytest.mark.parametrize("kind", ["torch", "handle"])
def test_device_output_changes_on_a_stream_of_the_caller(kind):
    """The records of a run whose snapshots reach the device on a side stream,
    extracted on that stream while the current one keeps allocating and
    overwriting: those of the default call, from a torch stream and from an
    object that holds a stream's handle."""
    from types import SimpleNamespace

    import torch
    from jacquard_amd import vcd
    nl, comp = design("xp", level_split=8, seed=5, gates=20000, depth=40,
                      dffs=2000, inputs=64, outputs=32, geometric_p=0.3, srams=2)
    s = comp.flatten(16)
    cycles, rio = 300, s.reg_io_state_size
    st = stimulus.build_states(s, cycles, seed=17, p=0.4)
    offs = [((k + 1) * rio, vcd.U64_MAX if k % 7 == 3 else 10 * k) for k in range(cycles)]
    d = sim.run_scan(s, st, cycles, return_device=True)["device"]["states"]
    cnt, rec = vcd.output_changes_device(s, d, offs)
    assert rec.size > 0
    side = torch.cuda.Stream()
    stream = side if kind == "torch" else SimpleNamespace(cuda_stream=side.cuda_stream)
    for k in range(3):
        late = torch.zeros_like(d)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            late.copy_(d)
        junk = [torch.full((1 << 12,), -1, dtype=torch.int32, device="cuda") for _ in range(8)]
        got_cnt, got_rec = vcd.output_changes_device(s, late, offs, stream=stream)
        junk += [torch.full((1 << 12,), -1, dtype=torch.int32, device="cuda") for _ in range(8)]
        assert np.array_equal(got_cnt, cnt) and np.array_equal(got_rec, rec), k
        assert torch.cuda.current_stream() != side

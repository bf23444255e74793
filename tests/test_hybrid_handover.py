"""What the hybrid decode kernel's hand-over rests on, worked out from its schedules without a GPU.

An instruction waits only for the units that it reads (an attention's parts: for all arrivals of their stage), and buffers are used by one layer
after the other.  So whoever writes a place must come behind everyone that reads what was there, by what it has waited for itself; and its store must be
known to come last, by somebody that has seen the old value there (or by an arrival, which is counted behind the stores).  Here every instruction has
its reads and writes as the kernel makes them (csrc/qmk_hybrid_ops.h) and a clock: per queue, how many instructions it is behind."""
import dataclasses

import numpy as np
import pytest

from qimeng_megakernel_amd import registry, synthetic
from qimeng_megakernel_amd.decode_schedule_hybrid.instructions import instruction_defs as D
from qimeng_megakernel_amd.decode_schedule_hybrid.instructions import scheduler as S
from test_hybrid_schedule import odd_shape
from test_looped_schedule import odd_shape as odd_plain_shape

BRANCHES = 2      # QMK_HYBRID_MAX_BRANCHES


class Accesses:
    """Reads and writes of one instruction, (buffer, first, end) each; ``parts``: of the counted buffers."""

    def __init__(self, shape, position, capacity, empty_parts_wait=True):
        self.shape, self.position, self.capacity, self.empty_parts_wait = shape, position, capacity, empty_parts_wait
        self.place = {}
        proj = mix = 0
        for i, e in enumerate(shape.entries):
            l = e.shape
            if e.branch == 0:
                proj = mix = 0
            ff_at = sum(b.shape.mix_width for b in shape.entries[i : i + e.branches]) if shape.plain and e.ff else 0
            self.place[i] = (proj, mix, ff_at)
            if shape.plain and l.type not in ("join", "final"):
                proj, mix = proj + l.in_rows + (l.mix_width if l.type == "delta" else 0), mix + l.mix_width

    def residual(self, i):
        width, e = self.shape.width_s, self.shape.entries[i]
        e = self.shape.entries[i - e.branch]
        if e.prev < 0:
            return [("x%d" % e.x_from, 0, width)] if e.x_from >= 0 else []
        run = self.shape.entries[e.prev]
        slots = [1, 2][: run.branches] + [1 + BRANCHES if run.ff else 0]
        return [("x%d" % run.x_to, s * width, (s + 1) * width) for s in slots]

    def attention(self, ins):
        """(first head, heads, key head, keys there, holds the position, columns, parts' row) of one part."""
        l, latent = self.shape.entries[ins.layer].shape, self.shape.entries[ins.layer].type == "latent_attention"
        group = l.heads if latent else l.heads // l.kv_heads
        blocks = -(-group // 16)
        kv, block = divmod(ins.sub, blocks)
        window = min(l.window, self.capacity) if latent else self.capacity
        first = max(self.position + 1 - window, 0)
        per = -(-(-(-(self.position + 1 - first) // ins.count)) // 32) * 32
        lo = first + ins.start * per
        hi = min(lo + per, self.position + 1)
        columns = l.rank_s if latent else l.v_s
        return kv * group + block * 16, min(16, group - block * 16), kv, lo < hi, lo <= self.position < hi, columns

    def of(self, ins):
        shape, i = self.shape, ins.layer
        e, width = shape.entries[i], shape.width_s
        l, (proj, mix, ff_at), op, a, n = e.shape, self.place[i], type(ins), ins.start, ins.count
        lead = shape.entries[i - e.branch]
        reads, writes, counted = [], [], []
        if op in (D.RMS_InProject, D.RMS_UpGate_Gelu, D.RMS_LMHead, D.JoinProject):
            reads = self.residual(i) if shape.plain else [("u", 0, width)] if i or op is not D.RMS_InProject else []
            if op is D.RMS_InProject:
                writes = [("proj", proj + a, proj + a + n)] + ([("x%d" % lead.x_to, 0, width)] if shape.plain and ins.extra else [])
            elif op is D.RMS_UpGate_Gelu:
                writes = [("mix", ff_at + a, ff_at + a + n)]
            elif op is D.JoinProject:
                writes = [("x%d" % e.x_to, a, a + n)]
        elif op is D.GatedRecurrence:
            at = ins.sub * l.block_s
            reads = [("proj", l.mix_width + at, l.mix_width + at + l.block_s), ("proj", at + a, at + a + n)]
            writes = [("mix", at + a, at + a + n)]
        elif op is D.LatentAbsorb:
            reads = [("proj", ins.sub * l.q_stride, (ins.sub + 1) * l.q_stride)]
            writes = [("absorbed", ins.sub * l.rank_s + a, ins.sub * l.rank_s + a + n)]
        elif op is D.AttendSplitKV:
            head0, heads, kv, keys, appends, columns = self.attention(ins)
            latent = l.type == "latent_attention"
            rows = range(head0, head0 + (16 if latent else heads))
            heads16 = S._ceil_div(l.heads, 16) * 16
            if not keys:
                at = ("absorbed", head0 * l.rank_s) if latent else ("proj", proj + head0 * l.q_stride)
                reads = [(at[0], at[1], at[1] + 1)] if self.empty_parts_wait else []
            elif latent:
                reads = [("absorbed", head0 * l.rank_s, (head0 + heads) * l.rank_s)] + [("proj", h * l.q_stride + l.dim_s, h * l.q_stride + l.dim_s + l.rot_s) for h in range(head0, head0 + heads)]
                row = l.heads * (l.q_stride + l.v_s)
                reads += [("proj", row, row + l.rank_s + l.rot_s)] if appends else []
            else:
                reads = [("proj", proj + head0 * l.q_stride, proj + (head0 + heads) * l.q_stride)]
                k, v = proj + l.heads * l.q_stride + kv * l.dim_s, proj + l.heads * l.q_stride + l.kv_heads * l.dim_s + kv * l.v_s
                reads += [("proj", k, k + l.dim_s), ("proj", v, v + l.v_s)] if appends else []
            if ins.extra == 0:
                counted += [("ml", a * heads16 + h, a * heads16 + h + 1) for h in rows]
            c0, c1 = ins.extra * 128, min(columns, ins.extra * 128 + 128)
            counted += [("part", (a * heads16 + h) * columns + c0, (a * heads16 + h) * columns + c1) for h in rows]
        elif op in (D.LatentValue, D.AttendMerge):
            latent, heads16 = op is D.LatentValue, S._ceil_div(l.heads, 16) * 16
            parts, columns = (ins.extra, l.rank_s) if latent else (n, l.v_s)
            counted = [(b, (p * heads16 + ins.sub) * w, (p * heads16 + ins.sub + 1) * w) for p in range(parts) for b, w in (("ml", 1), ("part", columns))]
            first, count = (a, n) if latent else (0, l.v_s)
            gate = (l.heads * l.q_stride if latent else proj + l.heads * l.q_stride + l.kv_heads * (l.dim_s + l.v_s)) + ins.sub * l.v_s + first
            reads = [("proj", gate, gate + count)]
            writes = [("mix", mix + ins.sub * l.v_s + first, mix + ins.sub * l.v_s + first + count)]
        elif op is D.WkvStep:
            m, d = l.mix_width, l.dim_s
            reads = [("proj", 4 * m, 4 * m + l.rank_s)] + [("proj", k * m + ins.sub * d, k * m + (ins.sub + 1) * d) for k in range(4)]
            writes = [("mix", ins.sub * d, (ins.sub + 1) * d)]
        elif op is D.GatedStateStep:
            delta, keys, d = l.type == "delta", l.kv_heads * l.dim_s, l.dim_s
            kv, v = ins.sub // (l.heads // l.kv_heads), proj + 2 * keys + ins.sub * l.v_s
            rank = proj + 2 * keys + l.heads * l.v_s * (1 if delta else 2)
            reads = [("proj", proj + kv * d, proj + (kv + 1) * d), ("proj", proj + keys + kv * d, proj + keys + (kv + 1) * d), ("proj", v + a, v + a + n), ("proj", rank, rank + l.rank_s)]
            steps = rank + l.rank_s + l.gate_rank_s
            reads += [("proj", steps, steps + l.heads_s)] if delta else []
            writes = [("mix", mix + ins.sub * l.v_s + a, mix + ins.sub * l.v_s + a + n)]
        elif op is D.OutputGate:
            at = proj + l.conv_channels + l.rank_s
            reads, writes = [("proj", at, at + l.gate_rank_s)], [("proj", proj + l.in_rows + a, proj + l.in_rows + a + n)]
        elif op is D.OutProject_Streams:
            down = ins.sub == 1
            reads = [("mix", ff_at, ff_at + shape.layers[e.layer].ff_s)] if down else [("mix", mix, mix + l.mix_width)]
            if not shape.plain:
                writes = [("u", a, a + n)]
            else:
                if not down and l.type != "attention":
                    gate = proj + (l.in_rows if l.type == "delta" else 2 * l.heads * l.dim_s + l.mix_width)
                    reads += [("proj", gate, gate + l.mix_width)]
                if down:
                    reads += [("x%d" % lead.x_to, a, a + n)]
                slot = (1 + (BRANCHES if down else e.branch)) * width
                writes = [("x%d" % lead.x_to, slot + a, slot + a + n)]
        return reads, writes, counted


class Buffer:
    def __init__(self, size, queues):
        self.writer = np.full(size, -1)                            # instruction that wrote the place last
        self.seen = np.full((size, queues), -1, dtype=np.int32)    # ... and per queue the last that read it since

    def grow(self, end):
        if end > len(self.writer):
            more = Buffer(2 * end - len(self.writer), self.seen.shape[1])
            self.writer, self.seen = np.concatenate((self.writer, more.writer)), np.concatenate((self.seen, more.seen))


def faults(shape, queues, position, capacity, empty_parts_wait=True):
    """What is wrong with one step, as texts."""
    found, accesses = [], Accesses(shape, position, capacity, empty_parts_wait)
    sched = S.HybridScheduler(shape, queues, capacity)
    buffers: dict[str, Buffer] = {}
    behind = np.zeros((queues, queues), dtype=np.int32)      # clock of every queue's last instruction
    clocks, at = [], []                                      # per instruction: its clock when it writes; (queue, number)
    done = np.zeros(queues, dtype=np.int32)

    def place(name, first, end):
        b = buffers.setdefault(name, Buffer(0, queues))
        b.grow(end)
        return b, slice(first, end)

    for k, stage in enumerate(sched.stages()):
        arrivals, looked = None, {}
        before = len(clocks) - (len(sched.stages()[k - 1]) if k else 0)
        for j, ins in enumerate(stage):
            q = j % queues
            reads, writes, counted = accesses.of(ins)
            merge = isinstance(ins, (D.LatentValue, D.AttendMerge))
            clock = behind[q].copy()
            for interval in reads:
                if interval not in looked:
                    b, part = place(*interval)
                    writers = np.unique(b.writer[part])
                    if writers[0] < 0:
                        found.append(f"{ins} reads what nobody has written: {interval}")
                        writers = writers[1:]
                    # (a writer's reads are done when its value is there)
                    own = np.zeros(queues, dtype=np.int32)
                    for w in writers:
                        own[at[w][0]] = max(own[at[w][0]], at[w][1] + 1)
                    looked[interval] = np.maximum(own, np.max([clocks[w] for w in writers], axis=0)) if len(writers) else own
                clock = np.maximum(clock, looked[interval])
            if merge:
                if arrivals is None:
                    own = np.zeros(queues, dtype=np.int32)
                    for w in range(before, before + len(sched.stages()[k - 1])):
                        own[at[w][0]] = max(own[at[w][0]], at[w][1] + 1)
                    arrivals = np.maximum(own, np.max(clocks[before : before + len(sched.stages()[k - 1])], axis=0))
                clock = np.maximum(clock, arrivals)
            number, ident = int(done[q]), len(clocks)
            for name, first, end in writes + ([] if merge else counted):
                b, part = place(name, first, end)
                late = b.seen[part] >= np.maximum(clock, number * (np.arange(queues) == q))[None]
                if late.any():
                    found.append(f"{ins} overwrites {name}[{first}:{end}] while it may be read")
                old = b.writer[part]
                unread = (old >= 0) & (b.seen[part].max(axis=1) < 0)
                if name not in ("ml", "part") and unread.any():
                    found.append(f"{ins} overwrites {name}[{first}:{end}], which nobody has seen")
                if name in ("ml", "part"):      # an arrival counts stores that are done
                    for w in np.unique(old[old >= 0]):
                        if at[w][0] != q and clock[at[w][0]] <= at[w][1]:
                            found.append(f"{ins} overwrites {name}[{first}:{end}] while it may be written")
                b.writer[part], b.seen[part] = ident, -1
            for name, first, end in reads + (counted if merge else []):
                b, part = place(name, first, end)
                b.seen[part, q] = number
            clocks.append(clock)
            at.append((q, number))
            behind[q] = clock
            behind[q, q] = done[q] = number + 1
    return found


def uneven(width, layers, **kw):
    """Latent attentions of different sizes, one after the other."""
    base = dict(width=width, vocab=96, streams=2, heads=3, dim=32, rot_dim=16, v_dim=32, rank=64, window=100)
    return dataclasses.replace(synthetic.hybrid_shape("a", **base), layers=tuple(synthetic.hybrid_shape("a", **{**base, **l}).layers[0] for l in layers))


def uneven_plain(width, layers):
    base = dict(width=width, vocab=96, ff={"p": 48}, heads=4, kv_heads=2, dim=32, v_dim=32, delta_heads=2, delta_kv_heads=2, delta_dim=16, delta_v_dim=16, delta_rank=16, gate_rank=16)
    return dataclasses.replace(synthetic.looped_shape("p", **base), layers=tuple(synthetic.looped_shape("p", **{**base, **l}).layers[0] for l in layers))


SHAPES = {
    "odd": odd_shape(),
    "odd, every order": odd_shape(pattern="aawwraawr"),
    "odd plain": odd_plain_shape(),
    "odd plain, no feed-forward": odd_plain_shape("pgpp", ff={"g": 20}, loop=None),
    "windows": uneven(208, [dict(window=300), dict(window=100), dict(window=300)]),
    "ranks and heads": uneven(64, [dict(rank=144, heads=1), dict(rank=400, heads=18), dict(rank=64, heads=2)]),
    "plain heads": uneven_plain(64, [dict(heads=2), dict(heads=40, v_dim=80), dict(heads=4, kv_heads=4, v_dim=200)]),
    "delta heads": synthetic.looped_shape("pp", width=64, vocab=96, heads=2, kv_heads=1, dim=32, v_dim=32, delta_heads=17, delta_kv_heads=17, delta_dim=16, delta_v_dim=80,
                                          delta_rank=16, gate_rank=48),
}


@pytest.mark.parametrize("queues", [256, 40, 7])
@pytest.mark.parametrize("name", SHAPES)
def test_nothing_is_overwritten_while_it_may_be_read(name, queues):
    for position in (0, 33, 130, 511):
        assert faults(SHAPES[name], queues, position, 512) == []


def test_registered_shapes():
    for name in ("lusupel-1b", "givopel-1b"):
        shape = registry.shape_of(name)
        few = dataclasses.replace(shape, layers=shape.layers[:4], vocab=2048, loop=None)
        assert faults(few, 256, 1000, 4096) == []


SMALL = dict(heads=1, dim=16, rot_dim=16, v_dim=16, rank=144)
#: the second attention has parts without a key where the first has some, and queues 52 to 63 hold nothing but a part of each
BARE = uneven(64, [dict(window=3072, **SMALL), dict(window=2100, **SMALL)])


def test_a_part_without_keys_has_to_wait():
    assert faults(BARE, 256, 3100, 8192) == []
    assert any("while it may be read" in f for f in faults(BARE, 256, 3100, 8192, empty_parts_wait=False))

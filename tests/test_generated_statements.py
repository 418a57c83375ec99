"""The generated statements of the four-wave kernels that load straight into the LDS (gen_w4_loop.py, classes Wide and Ring), executed: scalar
registers, branches, the queue of memory operations that s_waitcnt vmcnt counts.  A work-group's tiles one behind the other, as the kernels give them."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MASK = 0xFFFFFFFF
P_BYTES, Q_BYTES = 0x1000, 0x2000                # of a slice or k-tile of either operand
CHUNK = 1024


@pytest.fixture(scope="module")
def macros(tmp_path_factory):
    out = tmp_path_factory.mktemp("loop") / "loop.inc"
    env = {k: v for k, v in os.environ.items() if k != "W4_OPTS"}
    subprocess.run([sys.executable, os.path.join(ROOT, "ml_dataflow_amd", "csrc", "matmul", "gen_w4_loop.py"), str(out)], check=True, env=env, cwd=ROOT)
    return dict(re.findall(r"#define (\w+)(.*?)(?=\n#define|\Z)", out.read_text(), re.S))


def lines_of(macros, *names):
    return [line for name in names for line in re.findall(r'"([^"]*?)\\n\\t"', macros[name])]


class Machine:
    """what one wave of the work-group does with a statement"""

    def __init__(self, lines):
        self.lines = lines
        self.s = {"m0": 0}
        self.queue = []                          # memory operations in flight, oldest first
        self.loads = []                          # every load into the LDS: (operand, address, place in the LDS)
        self.mfmas = self.from_zero = self.stores = self.barriers = 0
        self.at_barrier = self.at_load = self.at_epilogue = lambda: None

    def value(self, name):
        return self.s[name] if re.fullmatch(r"s\d+|m0", name) else int(name, 0) & MASK

    def target(self, at, label):
        number, direction = label[:-1], label[-1]
        places = range(at + 1, len(self.lines)) if direction == "f" else range(at - 1, -1, -1)
        return next(i for i in places if self.lines[i] == number + ":")

    def run(self):
        at, scc, last_mfma = 0, 0, False
        while at < len(self.lines):
            op, _, rest = self.lines[at].partition(" ")
            a = [x.strip() for x in rest.split(",")]
            at += 1
            if op == "s_mov_b32":
                self.s[a[0]] = self.value(a[1])
            elif op in ("s_add_u32", "s_addc_u32"):
                total = self.value(a[1]) + self.value(a[2]) + (scc if op == "s_addc_u32" else 0)
                self.s[a[0]], scc = total & MASK, int(total > MASK)
            elif op in ("s_sub_u32", "s_subb_u32"):
                total = self.value(a[1]) - self.value(a[2]) - (scc if op == "s_subb_u32" else 0)
                self.s[a[0]], scc = total & MASK, int(total < 0)
            elif op.startswith("s_cmp_"):
                x, y = self.value(a[0]), self.value(a[1])
                scc = int({"lg": x != y, "eq": x == y, "lt": x < y, "ge": x >= y}[op.split("_")[2]])
            elif op == "s_cselect_b32":
                self.s[a[0]] = self.value(a[1]) if scc else self.value(a[2])
            elif op == "s_bitcmp1_b32":
                scc = self.value(a[0]) >> int(a[1]) & 1
            elif op in ("s_cbranch_scc0", "s_cbranch_scc1"):
                if scc == int(op[-1]):
                    at = self.target(at - 1, a[0])
            elif op == "s_branch":
                at = self.target(at - 1, a[0])
            elif op == "s_barrier":
                self.at_barrier()
                self.barriers += 1
            elif op == "s_waitcnt":
                left = re.search(r"vmcnt\((\d+)\)", rest)
                if left:
                    assert int(left.group(1)) <= 63          # the field's width
                    self.queue = self.queue[len(self.queue) - int(left.group(1)):] if len(self.queue) > int(left.group(1)) else self.queue
            elif op == "buffer_load_dwordx4" and rest.endswith(" lds"):
                operand, base = ("P", 64) if "s[64:67]" in rest else ("Q", 68)
                self.loads.append((operand, self.s["s%d" % base] | self.s["s%d" % (base + 1)] << 32, self.s["m0"]))
                self.queue.append(len(self.loads) - 1)
                self.at_load()
            elif op == "buffer_load_dwordx4":
                assert "s[84:87]" in rest
                self.queue.append("C")
            elif op == "buffer_load_dword":
                assert "s[80:83]" in rest or "s[88:91]" in rest
                self.maps_asked = getattr(self, "maps_asked", 0) + 1
                self.queue.append(("map", self.maps_asked))
            elif op == "buffer_store_dwordx4":
                assert "s[92:95]" in rest
                self.stores += 1
                self.queue.append("D")
            elif op.startswith("v_mfma"):
                self.mfmas += 1
                self.from_zero += a[-1] == "0"
                last_mfma = True
            elif op.startswith("v_accvgpr_read") and last_mfma:
                self.at_epilogue()
                last_mfma = False
            else:
                assert op[0] == "v" or op.startswith(("ds_read", "ds_bpermute")) or op == "s_nop" or op[:-1].isdigit(), op


def cursor(tile, at):
    """both operands of tile `tile` at slice or k-tile `at`, none of a tile that does not exist"""
    if tile is None:
        return [0] * 8
    p, q = (tile + 1 << 32) + at * P_BYTES, (tile + 1 << 36) + at * Q_BYTES
    return [p & MASK, p >> 32, 0, 1, q & MASK, q >> 32, 0, 1]


def give(machine, first_register, values):
    for n, v in enumerate(values):
        machine.s["s%d" % (first_register + n)] = v


@pytest.mark.parametrize("scaled", [0, 4])
@pytest.mark.parametrize("name,least", [("W4K_C", 8), ("W4K_NOC", 5)])
def test_sliced_kernel_waits_for_what_it_reads(macros, name, least, scaled):
    slot_bytes, slots, per_slice = 32768, 5, 8
    tiles = [least, least + 1, least + 2, least, 11, 12, 40, least, 9, 23]
    start = [sum(tiles[:t]) for t in range(len(tiles))]                    # the stream's slice that the tile begins with
    m = Machine(lines_of(macros, name + "_ASM"))

    def slices_there():
        """slices whose loads have all arrived, this wave's"""
        waiting = [x for x in m.queue if isinstance(x, int)]
        return (waiting[0] if waiting else len(m.loads)) // per_slice

    def at_barrier():
        if m.barriers == 0:
            assert slices_there() == slots                                 # the first tile's first loads
        else:
            assert slices_there() > m.barriers, (name, m.barriers)         # barrier b lets all waves at slice b of the stream

    def at_load():
        operand, address, place = m.loads[-1]
        g, u = divmod(len(m.loads) - 1, per_slice)
        assert g < slots or m.barriers > g - slots + 1                     # every wave is done with the slice whose slot it takes
        assert place == 4096 * 2 + g % slots * slot_bytes + u % 4 * CHUNK + (16384 if u >= 4 else 0)
        tile = max(t for t in range(len(tiles)) if start[t] <= g)
        if g - start[tile] < tiles[tile]:
            assert (operand, address) == (("P", (tile + 1 << 32) + (g - start[tile]) * P_BYTES), ("Q", (tile + 1 << 36) + (g - start[tile]) * Q_BYTES))[u // 4]

    def at_epilogue():
        assert "C" not in m.queue

    m.at_barrier, m.at_load, m.at_epilogue = at_barrier, at_load, at_epilogue
    for t, slices in enumerate(tiles):
        before = m.mfmas, m.from_zero, m.stores, m.barriers, len(m.loads)
        give(m, 32, [7, 0, 1 << 20, 512, 9, 0, 0x3f800000, 0x3f800000])
        give(m, 40, cursor(t, 0) if t == 0 else cursor(t if slices > slots else None, slots))
        give(m, 48, cursor(t + 1 if t + 1 < len(tiles) else None, 0))
        give(m, 56, [slices, (t == 0) | scaled, P_BYTES, Q_BYTES, start[t] % slots * slot_bytes, 0, 16384, 4096 * 2])
        m.run()
        assert m.mfmas - before[0] == 64 * slices and m.from_zero - before[1] == 64
        assert m.stores - before[2] == 32
        assert m.barriers - before[3] == slices + (t == 0)
        assert len(m.loads) - before[4] == per_slice * (slices + (slots if t == 0 else 0))


@pytest.mark.parametrize("scaled", [0, 4])
@pytest.mark.parametrize("name", ["W4D_PKC_PACKED", "W4D_PKC_GATHER", "W4D_PKM_PACKED", "W4D_PKM_GATHER"])
def test_wide_kernel_waits_for_what_it_reads(macros, name, scaled):
    stage_p, stage_q, place_p, place_q, of_p, of_q = 32768, 49152, 8 * CHUNK, 65536 + 12 * CHUNK, 8, 12
    tiles = [2, 4, 2, 2, 6, 16, 2, 10]
    start = [sum(tiles[:t]) for t in range(len(tiles))]
    m = Machine(lines_of(macros, name + "_HEAD", name + "_ASM", name + "_END"))

    def k_tiles(operand, of):
        mine = [n for n, load in enumerate(m.loads) if load[0] == operand]
        waiting = {x for x in m.queue if isinstance(x, int)}
        return next((n for n, load in enumerate(mine) if load in waiting), len(mine)) // of

    def at_barrier():
        there = min(k_tiles("P", of_p), k_tiles("Q", of_q))
        assert there >= 1 if m.barriers == 0 else there > m.barriers, (name, m.barriers)

    def at_load():
        operand, address, place = m.loads[-1]
        g, u = divmod(sum(load[0] == operand for load in m.loads) - 1, of_p if operand == "P" else of_q)
        assert place == (place_p + g % 2 * stage_p if operand == "P" else place_q + g % 2 * stage_q) + u * CHUNK
        if operand == "P":
            assert g < 2 or m.barriers > g - 1                             # P is shared: every wave is done with the k-tile whose stage it takes
        tile = max(t for t in range(len(tiles)) if start[t] <= g)
        if g - start[tile] < tiles[tile]:
            assert address == ((tile + 1 << 32) + (g - start[tile]) * P_BYTES if operand == "P" else (tile + 1 << 36) + (g - start[tile]) * Q_BYTES)

    m.at_barrier, m.at_load = at_barrier, at_load
    for t, count in enumerate(tiles):
        before = m.mfmas, m.from_zero, m.stores, m.barriers, len(m.loads)
        give(m, 32, [7, 0, 1 << 20, 512, 0, 0, 0x3f800000, 0])
        give(m, 40, cursor(t, 0))
        give(m, 48, cursor(t + 1 if t + 1 < len(tiles) else None, 0))
        give(m, 56, [count, (t == 0) | scaled, P_BYTES, Q_BYTES, 0, place_p, place_q, 65536])
        m.run()
        assert m.mfmas - before[0] == 192 * count and m.from_zero - before[1] == 96
        assert m.stores - before[2] == 48
        assert m.barriers - before[3] == count + (t == 0)
        assert len(m.loads) - before[4] == (of_p + of_q) * (count + (2 if t == 0 else 0))


class Operands(Machine):
    """... and the fragments of P and Q that its multiplies take: what each register holds, or has on the way from the LDS"""

    class Lines(list):
        """the statement, each line looked at as it is executed"""

        def __getitem__(self, at):
            line = list.__getitem__(self, at)
            self.look(line)
            return line

    def __init__(self, lines):
        super().__init__(self.Lines(lines))
        self.lines.look = self.look
        self.plain = lines
        self.held, self.on_the_way, self.multiplied = {}, [], []

    def target(self, at, label):
        places = range(at + 1, len(self.plain)) if label[-1] == "f" else range(at - 1, -1, -1)
        return next(i for i in places if self.plain[i] == label[:-1] + ":")

    def look(self, line):
        if line.startswith("ds_read"):
            numbers = [int(x) for x in re.findall(r"\d+", line.split(" ", 1)[1])]
            offset = numbers[-1] if "offset" in line else 0
            self.on_the_way.append((list(range(numbers[0], numbers[1] + 1)), (numbers[2], offset)))
            for r in self.on_the_way[-1][0]:
                self.held[r] = None
        elif "lgkmcnt" in line:
            left = int(re.search(r"lgkmcnt\((\d+)\)", line).group(1))
            while len(self.on_the_way) > left:
                registers, what = self.on_the_way.pop(0)
                for r in registers:
                    self.held[r] = what
        elif line.startswith("v_mfma"):
            regs = re.findall(r"([av])\[(\d+):(\d+)\]", line)
            first = lambda n: [self.held[r] for r in range(int(regs[n][1]), int(regs[n][2]) + 1)]
            self.multiplied.append((regs[0][0] + regs[0][1], first(1), first(2)))


@pytest.mark.parametrize("blocks", [6, 5, 4, 3, 2])
@pytest.mark.parametrize("name", ["W4D_PKC_PACKED", "W4D_PKC_GATHER", "W4D_PKM_PACKED", "W4D_PKM_GATHER"])
def test_wide_kernel_multiplies_short_tiles(macros, name, blocks):
    """Tiles of `blocks` column blocks a wave among full ones: every multiply's operands, where the loads go and when."""
    stage_p, stage_q, place_p, place_q, of_p, of_q = 32768, 49152, 8 * CHUNK, 65536 + 12 * CHUNK, 8, 12
    tiles = [(2, 6), (4, blocks), (2, blocks), (6, 6), (2, blocks), (16, blocks), (8, 6), (4, blocks)]
    start = [sum(n for n, _ in tiles[:t]) for t in range(len(tiles))]
    m = Operands(lines_of(macros, name + "_HEAD", name + "_ASM", name + "_END"))
    kmajor, M_ARD, M_BRD = "PKM" in name, 192, 200

    def there(operand, of):
        mine = [n for n, load in enumerate(m.loads) if load[0] == operand]
        waiting = {x for x in m.queue if isinstance(x, int)}
        return next((n for n, load in enumerate(mine) if load in waiting), len(mine)) // of

    def at_barrier():
        k = min(there("P", of_p), there("Q", of_q))
        assert k >= 1 if m.barriers == 0 else k > m.barriers, (name, m.barriers)

    def at_load():
        operand, address, place = m.loads[-1]
        g, u = divmod(sum(load[0] == operand for load in m.loads) - 1, of_p if operand == "P" else of_q)
        assert place == (place_p + g % 2 * stage_p if operand == "P" else place_q + g % 2 * stage_q) + u * CHUNK
        if operand == "P":
            assert g < 2 or m.barriers > g - 1
        else:
            # the wave's own rows: every fragment of the k-tile whose stage this takes is in its registers
            assert g < 2 or not [what for _, what in m.on_the_way if what[0] in (M_BRD + g % 2, M_BRD + 2 + g % 2) and m.barriers <= g - 1]
        tile = max(t for t in range(len(tiles)) if start[t] <= g)
        k = g - start[tile]
        if k < tiles[tile][0]:
            assert address == ((tile + 1 << 32) + k * P_BYTES if operand == "P" else (tile + 1 << 36) + k * Q_BYTES)

    m.at_barrier, m.at_load = at_barrier, at_load
    for t, (count, nb) in enumerate(tiles):
        before = m.mfmas, m.from_zero, m.stores, m.barriers, len(m.loads)
        m.multiplied = []
        give(m, 32, [7, 0, 1 << 20, 512, 0, 0, 0x3f800000, 0])
        give(m, 40, cursor(t, 0))
        give(m, 48, cursor(t + 1 if t + 1 < len(tiles) else None, 0))
        give(m, 56, [count, (t == 0) | (0 if nb == 6 else 1 << 14 - nb), P_BYTES, Q_BYTES, 0, place_p, place_q, 65536])
        m.run()
        assert m.mfmas - before[0] == 32 * nb * count and m.from_zero - before[1] == 16 * nb
        assert m.stores - before[2] == 48
        assert m.barriers - before[3] == count + (t == 0)
        assert len(m.loads) - before[4] == (of_p + of_q) * (count + (2 if t == 0 else 0))
        want = set()
        for k in range(count):
            stage = k & 1
            for s in range(2):
                for i in range(16):
                    for j in range(nb):
                        group, low = (i // 4) * 6 + j, (i % 4) * 4
                        acc = "a%d" % (16 * group + low) if group < 16 else "v%d" % (16 * (group - 16) + low)
                        if kmajor:
                            at = stage * 32768 + s * 32 * 512 + (i // 8) * 256
                            a = [(M_ARD + i % 8, at)] * 2 + [(M_ARD + i % 8, at + 4 * 512)] * 2
                        else:
                            a = [(M_ARD + s, stage * 32768 + i * 2048)] * 4
                        want.add((k, acc, tuple(a), tuple([(M_BRD + 2 * s + stage, j * 2048)] * 4)))
        got = {(n // (32 * nb), acc, tuple(a), tuple(b)) for n, (acc, a, b) in enumerate(m.multiplied)}
        assert got == want and len(m.multiplied) == len(want)


class Gathering(Machine):
    """... and, lane by lane, the registers with which a wave finds the rows of its loads of P"""

    MAP0 = 224                                   # first of them in the statement

    class Lines(list):
        def __getitem__(self, at):
            line = list.__getitem__(self, at)
            self.look(line)
            return line

    def __init__(self, lines, maps):
        super().__init__(self.Lines(lines))
        self.lines.look = self.look
        self.plain, self.maps = lines, maps
        self.v, self.pending, self.vcc, self.taken = {}, {}, None, []

    def target(self, at, label):
        places = range(at + 1, len(self.plain)) if label[-1] == "f" else range(at - 1, -1, -1)
        return next(i for i in places if self.plain[i] == label[:-1] + ":")

    def lanes(self, name):
        if name[0] == "v" and name[1:].isdigit():
            n = int(name[1:])
            if n in self.pending:                # of a load of the map: there once it is no longer in the queue
                assert not [x for x in self.queue if isinstance(x, tuple) and x[1] == self.pending[n][0]], name
                self.v[n] = self.pending.pop(n)[1]
            assert n not in [x for x, _ in self.taken], name
            return list(self.v[n])
        return [self.value(name)] * 64

    def look(self, line):
        op, _, rest = line.partition(" ")
        a = [x.strip() for x in rest.replace(" offset:", ", ").replace(" offen", "").split(",")]
        if op == "s_waitcnt" and "lgkmcnt(0)" in rest:
            for n, value in self.taken:
                self.v[n] = value
            self.taken = []
        if op.startswith("buffer_load_dwordx4") or not a[0].startswith("v") or not (a[0] == "vcc" or a[0][1:].isdigit() and (self.MAP0 <= int(a[0][1:]) < 240 or 208 <= int(a[0][1:]) < 212)):
            return
        n = None if a[0] == "vcc" else int(a[0][1:])
        if op == "buffer_load_dword":
            buffer = int(re.search(r"s\[(\d+):", rest).group(1))
            entries, bytes_ = self.maps.get(self.s["s%d" % buffer], []), self.s["s%d" % (buffer + 2)]
            assert n not in self.pending or not [x for x in self.queue if isinstance(x, tuple) and x[1] == self.pending[n][0]]
            self.pending[n] = (getattr(self, "maps_asked", 0) + 1, [entries[x // 4] if x < bytes_ else 0 for x in self.lanes(a[1])])
            return
        if n in self.pending:                    # written behind the load, which is over
            self.lanes(a[0])
        if op == "v_cmp_gt_u32":
            self.vcc = [x > y for x, y in zip(self.lanes(a[1]), self.lanes(a[2]))]
        elif op == "v_cndmask_b32":
            self.v[n] = [y if c else x for x, y, c in zip(self.lanes(a[1]), self.lanes(a[2]), self.vcc)]
        elif op == "ds_bpermute_b32":
            where, what = self.lanes(a[1]), self.lanes(a[2])
            self.taken.append((n, [what[(x + int(a[3]) >> 2) & 63] for x in where]))
        elif op == "v_mov_b32":
            self.v[n] = self.lanes(a[1])
        else:
            do = {"v_add_u32": lambda x, y: x + y & MASK, "v_min_u32": min, "v_mul_lo_u32": lambda x, y: x * y & MASK}[op]
            self.v[n] = [do(x, y) for x, y in zip(self.lanes(a[1]), self.lanes(a[2]))]


@pytest.mark.parametrize("wave", [0, 3])
@pytest.mark.parametrize("name,with_c", [("W4K_C_GATHER", 4), ("W4K_NOC_GATHER", 0)])
def test_sliced_kernel_finds_the_rows_of_gathered_loads(macros, name, with_c, wave):
    """the offsets of every load of P against the map, tiles of 8 to 40 slices whose last one is not full, rows outside the source"""
    import random
    rng = random.Random(wave)
    slot_bytes, slots, per_slice, pitch, source_rows = 32768, 5, 8, 512, 1000
    rows = [250, 256, 257, 300, 512, 513, 1280, 100, 255, 700, 256, 513]
    tiles = [max(8, -(-r // 32)) for r in rows]
    start = [sum(tiles[:t]) for t in range(len(tiles))]
    maps = {(t + 1) << 20: [rng.choice([rng.randrange(source_rows)] * 9 + [MASK]) for _ in range(r)] for t, r in enumerate(rows)}
    m = Gathering(lines_of(macros, name + "_ASM"), maps)

    def swizzle(k):
        return (k & 3) << 2 ^ (k >> 3 & 1) << 1

    m.v[230] = [4 * (32 * (l >> 3) + 8 * wave + (l & 7)) for l in range(64)]
    m.v[229] = [4 * (l >> 5) for l in range(64)]
    for odd in range(2):
        m.v[231 + odd] = [((l & 31) ^ swizzle(8 * wave + 2 * odd + (l >> 5))) * 16 for l in range(64)]

    def slices_there():
        waiting = [x for x in m.queue if isinstance(x, int)]
        return (waiting[0] if waiting else len(m.loads)) // per_slice

    def at_barrier():
        assert slices_there() == slots if m.barriers == 0 else slices_there() > m.barriers, (name, m.barriers)

    def at_load():
        operand, address, place = m.loads[-1]
        g, u = divmod(len(m.loads) - 1, per_slice)
        assert g < slots or m.barriers > g - slots + 1
        assert place == 4096 * 2 + g % slots * slot_bytes + u % 4 * CHUNK + (16384 if u >= 4 else 0)
        t = max(t for t in range(len(tiles)) if start[t] <= g)
        k = g - start[t]
        if k >= tiles[t]:
            return
        if u >= 4:
            assert (operand, address) == ("Q", (t + 1 << 36) + k * Q_BYTES)
            return
        assert (operand, address) == ("P", t + 1 << 32)
        for l in range(64):
            row = 32 * k + 8 * wave + 2 * u + (l >> 5)
            column = ((l & 31) ^ swizzle(row)) * 16
            got = m.lanes("v%d" % (208 + u))[l]
            if row < rows[t] and maps[(t + 1) << 20][row] < source_rows:
                assert got == maps[(t + 1) << 20][row] * pitch + column
            else:
                assert got >= source_rows * pitch                          # outside the source: zeros

    m.at_barrier, m.at_load = at_barrier, at_load
    for t, slices in enumerate(tiles):
        before = m.mfmas, m.from_zero, m.stores, m.barriers, len(m.loads)
        following = t + 1 if t + 1 < len(tiles) else None
        source = lambda n: [0, n + 1, source_rows * pitch, source_rows] if n is not None else [0, 0, 0, source_rows]
        give(m, 32, [7, 0, 1 << 20, 512, 9, 0, 0x3f800000, 0x3f800000])
        give(m, 40, source(t) + cursor(t, 0 if t == 0 else slots)[4:])
        give(m, 48, source(following) + cursor(following, 0)[4:])
        give(m, 56, [slices, t == 0, pitch, Q_BYTES, start[t] % slots * slot_bytes, 0, 16384, 4096 * 2])
        give(m, 80, [(t + 1) << 20, 0, 4 * rows[t], 0x20000])
        give(m, 88, [(t + 2) << 20, 0, 4 * rows[t + 1], 0x20000] if following is not None else [0, 0, 0, 0x20000])
        m.run()
        assert m.mfmas - before[0] == 64 * slices and m.from_zero - before[1] == 64
        assert m.stores - before[2] == 32
        assert m.barriers - before[3] == slices + (t == 0)
        assert len(m.loads) - before[4] == per_slice * (slices + (slots if t == 0 else 0))

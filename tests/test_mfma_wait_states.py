"""The kernels that issue matrix instructions from inline assembly (to pin their accumulators to
VGPRs) hide them from the compiler's hazard recognizer, which would otherwise put two wait states
between a vector-ALU write of a register and the MFMA that reads it as an operand.  The sources
place `s_nop 1` where such a write comes last; this test compiles them to assembly and checks the
rule on what the compiler scheduled: no vector-ALU instruction that writes an MFMA's A or B operand
may be one of the two instructions in front of it, and no instruction may read an MFMA's result
within nineteen wait states of it (thirteen for the eight-pass scaled FP8 instruction) unless it is an MFMA accumulating into it.  (Violations give wrong numbers only now and
then, depending on timing, which is why the rule is checked on the code and not on results.)  The same
goes for the other distances the compiler keeps for its own instructions only: scalar registers that a
vector-ALU instruction writes and a copy from assembly takes its address from, and registers that a load from assembly fills."""
import functools
import os
import re
import subprocess
import tempfile

import pytest

from cwick_amd import build as B

ASM_MFMA_SOURCES = ["gqa_prefill.hip", "indexer_band.hip", "mla_prefill64.hip", "mla_roles.hip"]


def _regs(tok):
    m = re.match(r"v\[(\d+):(\d+)\]", tok)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.match(r"v(\d+)$", tok)
    return {int(m.group(1))} if m else set()


def _operands(text):
    """Registers of every operand, "v7", "a12", "s3" ("vcc" is its two halves), an operand's in one set."""
    out = []
    for o in re.split(r",(?![^\[]*\])", text):
        o = re.sub(r"^-?\|?|\|$", "", o.strip().split(" ")[0])
        m = re.match(r"([vas])(?:(\d+)|\[(\d+):(\d+)\])$", o)
        if m:
            lo, hi = (m.group(2), m.group(2)) if m.group(2) else (m.group(3), m.group(4))
            out.append({m.group(1) + str(i) for i in range(int(lo), int(hi) + 1)})
        else:
            out.append({"vcc_lo", "vcc_hi"} if o == "vcc" else {o} if o in ("vcc_lo", "vcc_hi") else set())
    return out


class _Code:
    """A function's instructions, and which may be the one executed before each."""

    def __init__(self, name):
        self.name, self.text, self.op, self.regs, self.asm, self.label = name, [], [], [], [], {}

    def link(self):
        self.before = [[] for _ in self.text]
        for k, op in enumerate(self.op):
            if op.startswith(("s_branch", "s_cbranch")):
                self.before[self.label[self.text[k].split()[-1]]].append(k)
            if not op.startswith(("s_branch", "s_endpgm")) and k + 1 < len(self.text):
                self.before[k + 1].append(k)
        self.behind = [[] for _ in self.text]
        for k, b in enumerate(self.before):
            for j in b:
                self.behind[j].append(k)

    def valu(self, k):
        return self.op[k].startswith("v_") and not self.op[k].startswith("v_mfma")

    def written(self, k):
        """by a vector-ALU instruction (carries and exchanges have a second result)"""
        return set().union(*self.regs[k][:2 if re.search(r"swap|_co_|div_scale|mad_[iu]64", self.op[k]) else 1])

    def in_front(self, k, states):
        """(instruction, wait states in between) of all that may run less than so many in front, whatever the branches"""
        least, todo = {}, [(j, 0) for j in self.before[k]]
        while todo:
            j, w = todo.pop()
            if w < states and w < least.get(j, states):
                least[j] = w
                w += int(self.text[j].split()[1], 0) + 1 if self.op[j] == "s_nop" else 1
                todo += [(i, w) for i in self.before[j]]
        return least.items()

    def where(self, j, k, w):
        return "%s: %s | %s (%d in between)" % (self.name[:60], self.text[j][:80], self.text[k][:80], w)


@functools.lru_cache(maxsize=None)
def _functions(src):
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "k.s")
        cmd = [B._hipcc()] + B.COMMON + B.PER_FILE.get(src, []) + ["-w", "-S", "--cuda-device-only", os.path.join(B.CSRC, src), "-o", out]
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        lines = open(out).read().splitlines()
    found, cur, in_asm = [], None, False
    for line in lines:
        t = line.strip()
        if t.startswith(";;#ASM"):
            in_asm = t.startswith(";;#ASMSTART")
        elif re.match(r"\w+:", line):
            cur = _Code(line.split(":")[0])
            found.append(cur)
        elif t.startswith((".section", ".set")):
            cur = None
        elif cur and re.match(r"\.LBB\w+:", t):
            cur.label[t.split(":")[0]] = len(cur.text)
        elif cur and t and t[0] not in ";.":
            t = t.split(";")[0].strip()
            op, _, rest = t.partition(" ")
            cur.text.append(t), cur.op.append(op), cur.regs.append(_operands(rest)), cur.asm.append(in_asm)
    found = [f for f in found if f.text]
    for f in found:
        f.link()
    assert found
    return found


@pytest.mark.parametrize("src", ASM_MFMA_SOURCES)
def test_no_operand_of_an_mfma_is_written_right_before_it(src):
    """The first rule for everything that an MFMA from assembly reads: the two factors, the sum and the two registers of
    scales, whichever half of the register file they are in, and along every branch that leads to it."""
    n_mfma, bad = 0, []
    for f in _functions(src):
        for k, op in enumerate(f.op):
            if op.startswith("v_mfma") and f.asm[k]:
                n_mfma += 1
                read = set().union(*f.regs[k][1:6])
                bad += [f.where(j, k, w) for j, w in f.in_front(k, 2) if f.valu(j) and f.written(j) & read]
    assert n_mfma > 0
    assert not bad, "%d written within two wait states of the MFMA that reads it: %s" % (len(bad), bad[:3])


@pytest.mark.parametrize("src", ASM_MFMA_SOURCES)
def test_no_result_of_an_mfma_is_touched_too_early(src):
    """The other direction along every branch that leads away from an MFMA from assembly: what it leaves, in vector or in
    accumulation registers, may be neither read nor written over before it is there, except by an MFMA that goes on from it
    (the figures of test_no_valu_write_right_before_an_mfma_reads_it)."""
    n_mfma, bad = 0, []
    for f in _functions(src):
        for k in range(len(f.text)):
            onward = f.op[k].startswith("v_mfma")
            touched = set().union(*(f.regs[k][1:3] + f.regs[k][4:6] if onward else f.regs[k]))
            n_mfma += onward and f.asm[k]
            for j, w in f.in_front(k, 19):
                if f.op[j].startswith("v_mfma") and f.asm[j] and w < (13 if "16x16x128" in f.op[j] else 19) and f.regs[j][0] & touched:
                    bad.append(f.where(j, k, w))
    assert n_mfma > 0
    assert not bad, "%d touch an MFMA's result before the matrix pipe has written it: %s" % (len(bad), bad[:3])


@pytest.mark.parametrize("src", ["mla_roles.hip", "mla_prefill64.hip", "gqa_prefill.hip"])
def test_scalar_addresses_of_copies_come_from_the_scalar_unit(src):
    """A copy from assembly may take its base address out of scalar registers that a vector-ALU instruction wrote
    (v_readfirstlane, v_readlane) only five wait states later: the compiler, which keeps that distance for its own loads, does
    not for what a statement holds."""
    n_copies, bad = 0, []
    for f in _functions(src):
        for k, op in enumerate(f.op):
            if f.asm[k] and op.startswith(("global_", "buffer_", "flat_", "scratch_")):
                read = {r for r in set().union(*f.regs[k]) if r[0] == "s" or r.startswith("vcc")}
                n_copies += bool(read)
                bad += [f.where(j, k, w) for j, w in f.in_front(k, 5) if f.valu(j) and f.written(j) & read]
    assert n_copies > 0
    assert not bad, "%d scalar addresses are used before they are there: %s" % (len(bad), bad[:3])


@pytest.mark.parametrize("src", ASM_MFMA_SOURCES)
def test_no_valu_write_right_before_an_mfma_reads_it(src):
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "k.s")
        cmd = [B._hipcc()] + B.COMMON + B.PER_FILE.get(src, []) + [
            "-w", "-S", "--cuda-device-only", os.path.join(B.CSRC, src), "-o", out]
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        ins, from_asm, in_asm = [], [], False
        for line in open(out):
            t = line.strip()
            if t.startswith(";;#ASMSTART"):
                in_asm = True
            elif t.startswith(";;#ASMEND"):
                in_asm = False
            if not t or t.startswith((";", ".")) or t.endswith(":"):
                continue
            ins.append(t)
            from_asm.append(in_asm)
    n_mfma, bad, early = 0, [], []
    for i, t in enumerate(ins):
        if not t.startswith("v_mfma"):
            continue
        n_mfma += from_asm[i]
        ops = [o.strip() for o in t.split(None, 1)[1].split(",")]
        src_regs = _regs(ops[1]) | _regs(ops[2])
        for back in (1, 2):
            p = ins[i - back]
            # (an MFMA that the compiler issued itself is its own business: it knows what it wrote)
            if from_asm[i] and p.startswith("v_") and not p.startswith("v_mfma"):
                dst = _regs(p.split(None, 1)[1].split(",")[0].strip())
                if dst & src_regs:
                    bad.append((p, t))
        # The other direction: a result must not be read by anything but an MFMA that accumulates
        # into it before the matrix pipe has written it.  The compiler's own figure for the
        # longest MFMA is 19 wait states (an s_nop N counts N + 1, any other instruction 1);
        # the scan follows straight-line code and stops at a branch or after 24.
        dst_regs = _regs(ops[0])
        waited = 0
        for q in ins[i + 1:i + 64]:
            if q.startswith(("s_cbranch", "s_branch", "s_endpgm")) or waited >= 24:
                break
            qops = [o.strip() for o in q.split(None, 1)[1].split(",")] if " " in q else []
            reads = set()
            for o in (qops[1:] if q.startswith("v_") and not q.startswith("v_mfma") else qops):
                reads |= _regs(o.split()[0]) if o else set()
            if q.startswith("v_mfma"):
                reads = _regs(qops[1]) | _regs(qops[2])          # accumulating into the result is allowed
            # (the scaled FP8 16x16x128 instruction takes eight passes: the compiler's figure for an
            # eight-pass result is eleven wait states, twelve on this chip; thirteen are asked here)
            need = 13 if t.startswith("v_mfma_scale_f32_16x16x128") else 19
            if reads & dst_regs and waited < need:
                early.append((t[:60], q[:60], waited))
                break
            m = re.match(r"s_nop (\d+)", q)
            waited += int(m.group(1)) + 1 if m else 1
    assert n_mfma > 0
    assert not bad, "VALU write within two instructions of the MFMA that reads it: %r" % bad[:3]
    assert not early, "MFMA result read before the matrix pipe has written it: %r" % early[:3]


@functools.lru_cache(maxsize=None)
def _ir(src, kernel):
    """The lines of each instantiation of a kernel in the compiler's input to the scheduler, and what uses each value."""
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "k.ll")
        cmd = [B._hipcc()] + B.COMMON + B.PER_FILE.get(src, []) + [
            "-w", "-S", "-emit-llvm", "--cuda-device-only", os.path.join(B.CSRC, src), "-o", out]
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        functions = [f.splitlines() for f in open(out).read().split("\ndefine ")[1:]]
    found = []
    for lines in functions:
        if kernel not in lines[0]:
            continue
        users = {}
        for t in lines[1:]:
            for name in set(re.findall(r"%[\w.]+", t.split(" = ", 1)[-1])):
                users.setdefault(name, []).append(t.strip())
        found.append((lines, users))
    return found


@pytest.mark.parametrize("src,kernel,wait", [("gqa_prefill.hip", "gqa_prefill_team_kernel", "s_nop 15"),
                                             ("indexer_band.hip", "indexer_approx_kernel", "s_nop 15"),
                                             ("mla_roles.hip", "mla_roles_kernel", "s_nop 6")])
def test_the_wait_behind_the_matrix_instructions_carries_their_results(src, kernel, wait):
    """The rule above holds for what the compiler happened to schedule.  That it may not schedule otherwise takes the results
    through the wait: in the compiler's input to the scheduler, nothing but a further MFMA or the statement that waits
    may use what an MFMA from assembly leaves in VGPRs."""
    n_mfma, loose = 0, []
    for lines, users in _ir(src, kernel):
        for t in lines:
            m = re.match(r'\s+(%\w+) = .*\basm .*"(?:s_nop 1\\0A\\09)?v_mfma.*", "=&?v', t)
            if m:
                n_mfma += 1
                loose += [u for u in users.get(m.group(1), ()) if not re.search(r'\basm .*"(v_mfma|%s)' % wait, u)]
    assert n_mfma > 0
    assert not loose, "an MFMA's result is used by what no wait is in front of: %r" % loose[:3]


def test_what_a_load_from_assembly_brings_is_used_behind_its_wait():
    """The first loads of the latent decode (the query's rope block, the list's entries) are statements whose wait is a later
    one, so that the copies behind them stay in flight; to the compiler their values are there at once.  In its input to the
    scheduler nothing may use them but the empty statement behind the wait, wherever branches meet on the way to it."""
    n_loads, loose = 0, []
    for lines, users in _ir("mla_roles.hip", "mla_roles_kernel"):
        for t in lines:
            m = re.match(r'\s+(%\w+) = .*\basm .*"global_load_dword', t)
            if not m:
                continue
            n_loads += 1
            todo, seen = [m.group(1)], set()
            while todo:
                name = todo.pop()
                seen.add(name)
                for u in users.get(name, ()):
                    if re.search(r" = (extractvalue|phi) ", u):
                        todo += {u.split(" = ")[0]} - seen
                    elif not re.search(r'\basm sideeffect "",', u):
                        loose.append(u)
    assert n_loads == 2 + 1, "a rope block in both instantiations, the list's entries in one: %d" % n_loads
    assert not loose, "a load's result is used by what its wait is not in front of: %r" % loose[:3]


def test_decode_kernels_keep_their_tiles_in_registers():
    """The decode requests a tile while it works on the one before.  Where the two tiles and what belongs to them do
    not fit the registers, the compiler parks the requested one in scratch memory and waits for it there, and
    with that the request ahead is gone.  No variant of the kernel may have scratch memory."""
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "k.s")
        cmd = [B._hipcc()] + B.COMMON + ["-w", "-S", "--cuda-device-only", os.path.join(B.CSRC, "gqa_decode.hip"), "-o", out]
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        text = open(out).read()
    seen = re.findall(r"\.name:\s+(\S*gqa_decode_split_kernel\S*)\n\s+\.private_segment_fixed_size:\s+(\d+)", text)
    assert len(seen) == 20, "ten shapes, with a list and without: %d" % len(seen)
    assert not [k for k in seen if int(k[1])], [k for k in seen if int(k[1])]


LDS_DMA_SOURCES = ["mla_roles.hip", "mla_prefill64.hip", "gqa_prefill.hip"]


@pytest.mark.parametrize("src", LDS_DMA_SOURCES)
def test_m0_belongs_to_the_lds_copies_only(src):
    """The global -> LDS copies are issued from inline assembly that sets M0 (the LDS address)
    itself.  M0 is reserved to the compiler and cannot be declared clobbered, so the sources rely
    on the compiler having no use of M0 of its own in these kernels: on the compiled code, every
    instruction that names m0 must be the `s_mov_b32 m0, <scalar register>` of a copy statement,
    followed by its `s_nop 0` and its `global_load_lds_*`, and every such load must follow one.  (The
    register is the statement's "s" operand: the compiler may also hand out the two halves of vcc
    where no comparison needs them.  An immediate, exec or m0 itself is none of its choices.)"""
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "k.s")
        cmd = [B._hipcc()] + B.COMMON + B.PER_FILE.get(src, []) + [
            "-w", "-S", "--cuda-device-only", os.path.join(B.CSRC, src), "-o", out]
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        ins = []
        for line in open(out):
            t = line.split(";")[0].strip()
            if not t or t.startswith(".") or t.endswith(":"):
                continue
            ins.append(t)
    n_copies = 0
    for i, t in enumerate(ins):
        if re.search(r"\bm0\b", t):
            assert re.match(r"s_mov_b32 m0, (s\d+|vcc_lo|vcc_hi)$", t), "compiler-generated use of m0: " + t
            assert ins[i + 1] == "s_nop 0" and ins[i + 2].startswith("global_load_lds_"), ins[i:i + 3]
        if t.startswith("global_load_lds_"):
            n_copies += 1
            assert ins[i - 2].startswith("s_mov_b32 m0,") and ins[i - 1] == "s_nop 0", ins[i - 2:i + 1]
    assert n_copies > 0

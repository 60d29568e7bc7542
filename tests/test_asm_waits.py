"""Wait states around inline assembly, read from the compiler's own listing (no GPU).

The compiler inserts the wait states that gfx950 asks for between its own
instructions; what stands inside an asm statement it neither counts nor looks
into. For every path through every kernel that mixes the two, this checks:

- a matrix product's result that asm reads has passed through
  mfma_results_ready (an asm s_nop that names the registers): whatever order
  the scheduler chooses, the read cannot come too close;
- a cross-lane instruction (v_permlane*_swap, DPP) comes at least 2 slots after
  the asm instruction that wrote its operand;
- an asm direct load comes at least 5 slots after the vector instruction that
  wrote one of its scalar operands;
- an asm vector instruction comes at least 1 slot after the transcendental
  instruction that wrote its operand.
"""

import concurrent.futures
import re
import subprocess

import pytest

from gaudirt_amd import build

MFMA_WAIT = 8  # slots until a 16x16 product can be read, as the compiler counts them
SOURCES = ["decode_stream.hip", "decode_unit.hip", "paged_decode.hip", "paged_prefill.hip"]
TRANS = re.compile(r"v_(exp|log|rcp|rsq|sqrt|sin|cos)_")
REGISTER = re.compile(r"\b([vas])(?:(\d+)\b|\[(\d+):(\d+)\])")


def registers(text):
    """The registers of an operand list, one set an operand."""
    out = []
    for operand in text.split(","):
        regs = set()
        for kind, one, lo, hi in REGISTER.findall(operand):
            regs.update((kind, n) for n in range(int(one or lo), int(one or hi) + 1))
        out.append(regs)
    return out


class Instruction:
    def __init__(self, text, in_asm):
        code, _, comment = text.partition(";")
        self.op, _, rest = code.strip().partition(" ")
        self.in_asm = in_asm
        operands = registers(rest)
        self.swap = self.op.startswith("v_permlane") and "swap" in self.op
        stores = self.op.startswith(("buffer_store", "global_store", "flat_store", "ds_write", "s_cmp", "s_waitcnt"))
        stores = stores or (self.op.startswith("buffer_load") and rest.endswith("lds"))
        written = 0 if stores else 2 if self.swap else 1
        self.writes = set().union(*operands[:written])
        self.reads = set().union(*(operands if self.swap else operands[written:]))
        if self.op.startswith(("v_fmac", "v_mac", "v_writelane")):
            self.reads |= self.writes
        self.crosses_lanes = self.swap or bool(re.search(r"\b(row_\w+|quad_perm|wave_\w+):?", rest))
        # What the comment of an asm statement names.
        self.named = set().union(*registers(comment)) if in_asm else set()
        self.vector = self.op.startswith("v_")
        self.slots = int(rest) + 1 if self.op == "s_nop" else 1
        self.target = rest.strip() if self.op.startswith(("s_branch", "s_cbranch")) else None
        self.falls_through = self.op not in ("s_branch", "s_endpgm", "s_setpc_b64")


def kernels(listing):
    """{name: (instructions, predecessors of each)} of a device listing."""
    found, body, in_asm, labels = {}, None, False, {}
    for line in listing.splitlines():
        label = re.match(r"([\w.$]+):", line)
        text = line.strip()
        if label:
            name = label.group(1)
            if not name.startswith("."):
                body, labels = [], {}
                found[name] = (body, labels)
            elif body is not None:
                labels[name] = len(body)
        elif text.startswith(";;#ASMSTART"):
            in_asm = True
        elif text.startswith(";;#ASMEND"):
            in_asm = False
        elif body is not None and text and text[0] not in ".;":
            body.append(Instruction(text, in_asm))
        elif text.startswith(".section") or text.startswith(".end_amdgpu"):
            body = None
    out = {}
    for name, (body, labels) in found.items():
        before = [[i - 1] if i and body[i - 1].falls_through else [] for i in range(len(body))]
        for i, ins in enumerate(body):
            if ins.target in labels and labels[ins.target] < len(body):
                before[labels[ins.target]].append(i)
        out[name] = (body, before)
    return out


def definitions(body, before, at, reg, advance=lambda state, ins: state):
    """Writers of `reg` that reach instruction `at`, over every path back: (instruction, slots between, state, index).
    `advance` folds the instructions of a path, last one first, into its state (0 at first)."""
    work, done = [(p, 0, 0) for p in before[at]], set()
    while work:
        i, slots, state = work.pop()
        if (i, min(slots, 25), state) in done or (i, 25, state) in done:
            continue
        done.add((i, min(slots, 25), state))
        ins = body[i]
        if reg in ins.writes:
            yield ins, slots, state, i
            continue
        state = advance(state, ins)
        work += [(p, slots + ins.slots, state) for p in before[i]]


def unguarded_products(body, before, at, reg):
    """Products whose result asm instruction `at` reads in `reg` as soon as the scheduler likes."""
    def guarded(state, ins):
        return state or (ins.in_asm and ins.op == "s_nop" and ins.slots >= MFMA_WAIT and reg in ins.named)

    for d, _, state, i in definitions(body, before, at, reg, guarded):
        sources = [d]
        if "v_accvgpr_read" in d.op:  # the allocator's choice: a copy out of an accumulation register
            sources = [m for r in d.reads for m, *_ in definitions(body, before, i, r)]
        if not state:
            yield from {m for m in sources if "mfma" in m.op}


def faults(body, before):
    for at, ins in enumerate(body):
        if ins.in_asm and ins.vector:
            for reg in ins.reads:
                if reg[0] != "v":
                    continue
                for product in unguarded_products(body, before, at, reg):
                    yield f"{ins.op} reads {reg} of {product.op} as soon as the scheduler likes"
                for d, slots, *_ in definitions(body, before, at, reg):
                    if TRANS.match(d.op) and not d.in_asm and slots < 1:
                        yield f"{ins.op} reads {reg} of {d.op} at once"
        if not ins.in_asm and ins.crosses_lanes:
            for reg in ins.reads:
                for d, slots, *_ in definitions(body, before, at, reg):
                    if d.in_asm and d.vector and slots < 2:
                        yield f"{ins.op} reads {reg} {slots} slots after the asm {d.op}"
        if ins.in_asm and ins.op.startswith("buffer_load"):
            for reg in ins.reads:
                if reg[0] != "s":
                    continue
                for d, slots, *_ in definitions(body, before, at, reg):
                    if d.vector and slots < 5:
                        yield f"{ins.op} reads {reg} {slots} slots after {d.op}"


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    folder = tmp_path_factory.mktemp("listings")

    def listing(source):
        out = folder / (source + ".s")
        subprocess.run([build.HIPCC, *build.COMMON, *build.DEVICE_FLAGS, "--offload-device-only", "-S",
                        str(build.CSRC / source), "-o", str(out)], check=True, capture_output=True)
        return out.read_text()

    with concurrent.futures.ThreadPoolExecutor(len(SOURCES)) as pool:
        return dict(zip(SOURCES, pool.map(listing, SOURCES)))


@pytest.mark.parametrize("source", SOURCES)
def test_waits_around_asm(listings, source):
    checked, bad = 0, []
    for name, (body, before) in kernels(listings[source]).items():
        checked += sum(ins.in_asm and ins.vector for ins in body)
        bad += [f"{name}: {fault}" for fault in sorted(set(faults(body, before)))]
    assert checked, "no asm vector instruction found: the listing is not read as it is written"
    assert not bad, f"{len(bad)} faults, the first:\n" + "\n".join(bad[:10])


PRODUCT = "\tv_mfma_f32_16x16x32_bf16 v[0:3], v[8:11], v[12:15], v[0:3]\n"
MAXIMUM = "\t;;#ASMSTART\n\tv_max3_f32 v4, v0, v1, v2\n\t;;#ASMEND\n"
READY = "\t;;#ASMSTART\n\ts_nop 7 ; v[0:3]\n\t;;#ASMEND\n"
COPIED = PRODUCT.replace("v[0:3]", "a[0:3]") + "\tv_accvgpr_read_b32 v1, a1\n"


@pytest.mark.parametrize("text,count", [
    (PRODUCT + MAXIMUM, 3), (PRODUCT + READY + MAXIMUM, 0), (READY + PRODUCT + MAXIMUM, 3),
    (PRODUCT + READY.replace("s_nop 7", "s_nop 6") + MAXIMUM, 3),
    (PRODUCT + "\ts_nop 15\n" + MAXIMUM, 3),           # far enough, but only as this compiler ordered it
    (PRODUCT + "\ts_cbranch_scc1 .L1\n" + READY + ".L1:\n" + MAXIMUM, 3),
    (COPIED + MAXIMUM, 1), (COPIED + READY + MAXIMUM, 0),
    (MAXIMUM + "\tv_permlane32_swap_b32_e32 v4, v5\n", 1),
    (MAXIMUM + "\tv_mov_b32_dpp v5, v4 row_mirror row_mask:0xf bank_mask:0xf\n", 1),
    (MAXIMUM + "\tv_mov_b32_e32 v5, v4\n\ts_nop 0\n\tv_permlane32_swap_b32_e32 v4, v5\n", 0),
    ("\tv_exp_f32_e32 v1, v9\n" + MAXIMUM, 1), ("\tv_exp_f32_e32 v1, v9\n\ts_nop 0\n" + MAXIMUM, 0),
    ("\tv_readfirstlane_b32 s4, v9\n\t;;#ASMSTART\n\tbuffer_load_dwordx4 v1, s[4:7], 0 offen lds\n\t;;#ASMEND\n", 1),
])
def test_the_reader_sees_planted_faults(text, count):
    body, before = kernels("kernel:\n" + text + "\ts_endpgm\n")["kernel"]
    assert len(list(faults(body, before))) == count

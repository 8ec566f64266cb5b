"""What the compiler cannot check around the inline assembly of the HIP kernels, checked on the device assembly of every build.

The compiler inserts the wait states gfx9-family hardware needs between certain instruction pairs, but it does not
look inside inline assembly.  Three of those pairs involve the hand-written vector-memory instructions of the tuned
kernels (direct-to-LDS copies, non-temporal stores):
  * a vector instruction writes a scalar register (v_readlane / v_readfirstlane, e.g. the reload of a spilled scalar)
    and a vector-memory instruction reads that register fewer than five wait states later: it sees the old value --
    for a buffer descriptor that means a wild address;
  * a 12- or 16-byte store is followed within two wait states by a vector instruction that overwrites its data
    registers: the store writes the new value;
  * a scalar instruction writes m0 and the very next instruction is a copy to LDS (a buffer load with the lds
    modifier), which takes its LDS address from m0: one wait state must lie between them.
The first two were met while developing these kernels (a GPU memory fault, and wrong dwords in the output); the
third is the rule the compiler applies to its own copies of this kind.  Besides, the four-wave kernels name registers in the text of their
statements that the compiler does not know to be in use: nothing else keeps it from using them.

The build fails where one of these finds something (build.py), so that no library exists that was not looked over.
"""
import re


def _regs(tok: str, kind: str):
    m = re.match(kind + r"\[(\d+):(\d+)\]$", tok)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.match(kind + r"(\d+)$", tok)
    return {int(m.group(1))} if m else set()


def _wait_states(line: str) -> int:
    m = re.match(r"s_nop (\d+)", line)
    return int(m.group(1)) + 1 if m else 1


def scan(text: str):
    """Returns a list of (first instruction, second instruction, wait states between them) for every hazard found."""
    code = []
    for raw in text.splitlines():
        line = raw.split(";")[0].strip()
        if line and not line.startswith(".") and not line.endswith(":"):
            code.append(line)
    bad = []
    for i, line in enumerate(code):
        op = line.split()[0]
        toks = [t.strip(",") for t in line.split()[1:]]
        if not op.startswith(("buffer_", "global_", "flat_", "scratch_")):
            continue
        if op.startswith("buffer_load") and toks[-1] == "lds" and i > 0:
            prev = code[i - 1].split()
            if prev[0].startswith("s_") and len(prev) > 1 and prev[1].strip(",") == "m0":
                bad.append((code[i - 1], line, 0))
        need = set().union(*[_regs(t, "s") for t in toks]) if toks else set()
        ws = 0
        for d in range(1, 8):
            if not need or i - d < 0 or ws >= 5:
                break
            prev = code[i - d]
            ptoks = prev.split()
            if ptoks[0].startswith("v_") and len(ptoks) > 1 and _regs(ptoks[1].strip(","), "s") & need:
                bad.append((prev, line, ws))
                break
            ws += _wait_states(prev)
        if re.match(r"(buffer|global|flat|scratch)_store_dwordx[34]", op):
            data = _regs(toks[0], "v") if op.startswith("buffer") else _regs(toks[1], "v")
            ws = 0
            for d in range(1, 4):
                if i + d >= len(code) or ws >= 2:
                    break
                nxt = code[i + d]
                ntoks = nxt.split()
                if ntoks[0].startswith("v_") and len(ntoks) > 1 and _regs(ntoks[1].strip(","), "v") & data:
                    bad.append((line, nxt, ws))
                    break
                ws += _wait_states(nxt)
    return bad


# The four-wave kernel keeps operand chunks that are in flight across loop iterations in v[192:255], named in the
# text of its own load and LDS-write statements; the compiler must never have allocated one of them for itself (it
# would move or overwrite a value it knows nothing about).
_RESERVED = set(range(192, 256))


def stray_uses_of_reserved_registers(text: str):
    """Lines of the four-wave kernels that touch v192..v255 other than the staging loads and LDS writes."""
    stray, inside = [], False
    for raw in text.splitlines():
        line = raw.split(";")[0].strip()
        if line.endswith(":") and not line.startswith("."):
            inside = "gemm_w4_kernel" in line
            continue
        if not inside or not line or line.startswith("."):
            continue
        toks = [t.strip(",") for t in line.split()]
        used = set().union(*[_regs(t, "v") for t in toks[1:]]) & _RESERVED
        if not used:
            continue
        staged_load = toks[0] == "buffer_load_dwordx4" and _regs(toks[1], "v") == used and toks[-1] != "lds"
        staged_write = toks[0] == "ds_write_b128" and _regs(toks[2], "v") == used
        if not (staged_load or staged_write):
            stray.append(line)
    return stray


# The four-wave kernel's multiplies are inline assembly, so the compiler does not know when their results land: it
# places the epilogue's v_accvgpr_read wherever the source order allows.  The source order is written so that a block
# is read no sooner than three multiplies (48 cycles of issue) after the multiply that wrote it, or behind a
# statement of idle cycles; this scanner checks the kept assembly for it, in text order (what crosses a loop's back
# edge is further apart than what it sees).
_MIN_MULTIPLIES_BETWEEN = 3
_MIN_IDLE_WAIT_STATES = 12


def accumulator_reads_too_early(text: str):
    """(multiply, read, multiplies in between, idle wait states in between) for every v_accvgpr_read in a four-wave
    kernel that follows the multiply that wrote its register too closely."""
    bad, inside = [], False
    last_write = {}  # accumulator register -> (index of the multiply that wrote it, its text, idle wait states issued so far)
    n_mul, idle = 0, 0
    for raw in text.splitlines():
        line = raw.split(";")[0].strip()
        if line.endswith(":") and not line.startswith("."):
            inside = "gemm_w4_kernel" in line
            last_write, n_mul, idle = {}, 0, 0
            continue
        if not inside or not line or line.startswith("."):
            continue
        toks = [t.strip(",") for t in line.split()]
        if toks[0].startswith("v_mfma"):
            for r in _regs(toks[1], "a"):
                last_write[r] = (n_mul, line, idle)
            n_mul += 1
        elif toks[0] == "s_nop":
            idle += _wait_states(line)
        elif toks[0] == "v_accvgpr_read_b32":
            for r in _regs(toks[2], "a"):
                if r in last_write:
                    at, mul, idle_then = last_write[r]
                    between, waited = n_mul - at - 1, idle - idle_then
                    if between < _MIN_MULTIPLIES_BETWEEN and waited < _MIN_IDLE_WAIT_STATES:
                        bad.append((mul, line, between, waited))
    return bad


# The K-grouped four-wave kernels hold a work-queue draw that is in flight across K steps in v255 (KgDraw, w4_common.hpp).
K_GROUPED = {"gemm_wgrad": "gemm_wgrad_kernel", "fp8_w4": "fp8_w4_kernel"}  # source file, kernel


def _kernel_lines(text: str, kernel: str):
    inside = False
    for raw in text.splitlines():
        line = raw.split(";")[0].strip()
        if line.endswith(":") and not line.startswith("."):
            inside = kernel in line
        elif inside and line and not line.startswith("."):
            yield line, [t.strip(",") for t in line.split()]


def stray_uses_of_v255(text: str, kernel: str):
    stray = []
    for line, toks in _kernel_lines(text, kernel):
        if not any(255 in _regs(t, "v") for t in toks[1:]):
            continue
        drawn = toks[0] == "global_atomic_add" and toks[1] == "v255" and toks[-1] == "sc0" and "v255" not in toks[2:]
        taken = toks[0] == "v_readfirstlane_b32" and toks[2] == "v255"
        if not (drawn or taken):
            stray.append(line)
    return stray


# Their fragment reads are inline assembly as well, and those of fp8_w4.hip are in flight across groups of multiplies and across the
# slab loop: nothing may touch a register that a read is still to fill.  LDS operations complete in order, so a wait
# for lgkmcnt(n) leaves the n youngest in flight.
def uses_of_reads_in_flight(text: str, kernel: str):
    bad, flight = [], []
    for line, toks in _kernel_lines(text, kernel):
        if toks[0] == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", line)
            if m:
                flight = flight[max(0, len(flight) - int(m.group(1))):]
            continue
        used = set().union(*[_regs(t, "v") for t in toks[1:]]) if len(toks) > 1 else set()
        if used & set().union(set(), *flight):
            bad.append(line)
        if toks[0].startswith("ds_"):
            flight.append(_regs(toks[1], "v") if toks[0].startswith("ds_read") else set())
    return bad


# The four-wave kernel names its fragments (v[64:191]), staged chunks (v[192:255]) and accumulators (all AGPRs) in the text of its own statements;
# the compiler, which knows nothing of what they hold, must not use any of them itself.
def compiler_uses_of_named_registers(text: str):
    stray, inside, ours = [], False, False
    for raw in text.splitlines():
        if "#ASMSTART" in raw or "#ASMEND" in raw:
            ours = "#ASMSTART" in raw
            continue
        line = raw.split(";")[0].strip()
        if line.endswith(":") and not line.startswith("."):
            inside = "gemm_w4_kernel" in line
            continue
        if not inside or ours or not line or line.startswith("."):
            continue
        toks = [t.strip(",") for t in line.split()[1:]]
        if any(_regs(t, "a") or any(r >= 64 for r in _regs(t, "v")) for t in toks):
            stray.append(line)
    return stray


def findings(stem: str, text: str):
    """What is wrong with the device assembly of csrc/<stem>.hip, one line each."""
    checks = [("wait states missing", scan(text))]
    if stem == "gemm_w4":
        checks += [("compiler-generated uses of v[192:255]", stray_uses_of_reserved_registers(text)),
                   ("compiler-generated uses of named registers", compiler_uses_of_named_registers(text)),
                   ("accumulator reads too close behind the multiply", accumulator_reads_too_early(text))]
    if stem in K_GROUPED:
        kernel = K_GROUPED[stem]
        checks += [("uses of v255", stray_uses_of_v255(text, kernel)),
                   ("uses of a register that an LDS read is to fill", uses_of_reads_in_flight(text, kernel)),
                   ("accumulator reads too close behind the multiply", accumulator_reads_too_early(text.replace(kernel, "gemm_w4_kernel"))),
                   # a spilled value would be reloaded behind the copies
                   ("uses of scratch memory", [line for line, _ in _kernel_lines(text, kernel) if "scratch_" in line])]
    expected = {"gemm_w4": "gemm_w4_kernel", **K_GROUPED}.get(stem)
    if expected and expected not in text:
        checks.append(("no kernel of this name", [expected]))
    return [f"{stem}: {len(found)} {what}, first: {found[0]}" for what, found in checks if found]

"""Kernels that ask for loads the compiler does not track (written as instructions) wait for them by count: `vmcnt(n)` lets
the n youngest operations stay on their way, and n counts other loads of the kernel among them, the compiler's own too. A
load that the compiler takes out or joins with another makes such a wait too short, silently. So this build step reads the
compiler's assembly and follows the counter along every path of every such kernel (a state is the queue of operations on
their way; a branch goes both ways, except over an empty execution mask, which none of these kernels has in its loops).

decode.hip, the matrix product over laid-out inputs: inputs go to LDS three chunks ahead, a barrier a chunk. At a barrier
only those asked for since the barrier before may be on their way (at the first, and at the end, none).

exl3.hip, the packed products: words and activations are loaded into registers by instructions, from LDS and from memory.
From such a load to the wait that covers it, past the loop too, no instruction may name a register that it writes: the
compiler takes them for written, copies them, and gives those that nothing reads to other values. The weights go by a ring
of four stages in LDS: a stage's words may be asked for when its loads have landed, and its place filled again when they
have come.

Needs hipcc, no GPU. Run by the library's build (__graft_entry__.build) and by tests/test_counted_waits.py;
`python check_counted_waits.py` runs it alone."""
import concurrent.futures
import functools
import os
import re
import shutil
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
MOST_STATES = 400000
MEMORY = re.compile(r"(global|buffer|flat|scratch)_(load|store|atomic)")
BRANCH = re.compile(r"s_(cbranch_\w+|branch)\s+(\S+)")


@functools.lru_cache(maxsize=None)
def assembly_of(source):
    """The compiler's gfx950 assembly of a source of this folder, with the library's flags."""
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "kernels.s")
        subprocess.run(
            [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-I" + os.path.join(ROOT, "include"), "-I" + HERE,
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", out,
             os.path.join(HERE, source)],
            check=True, capture_output=True, timeout=1200)
        with open(out) as f:
            return f.read()


def kernels_of(assembly, pattern):
    for m in re.finditer(r"^(_ZN\S*(?:%s)\S*):" % pattern, assembly, re.M):
        yield m.group(1), assembly[m.end():assembly.index(".Lfunc_end", m.end())]


def blocks_of(body):
    """The kernel's basic blocks in order, (label, [(instruction, written by hand)])."""
    blocks, own = [("entry", [])], False
    for line in body.split("\n"):
        text = line.strip()
        if "#ASMSTART" in text or "#ASMEND" in text:
            own = "#ASMSTART" in text
            continue
        label = re.match(r"(\.LBB\d+_\d+):", text)
        if label:
            blocks.append((label.group(1), []))
            continue
        code = text.split(";")[0].strip()
        if code and not code.startswith(".") and not code.endswith(":"):
            blocks[-1][1].append((code, own))
    return blocks


def follow(body, state, step):
    """Every reachable state along every path: step(instruction, written by hand, state) gives the state after it."""
    blocks = blocks_of(body)
    at = {label: i for i, (label, _) in enumerate(blocks)}
    seen, todo = set(), [(0, state)]
    while todo:
        here = todo.pop()
        if here in seen:
            continue
        seen.add(here)
        assert len(seen) <= MOST_STATES, "more states than this check follows"
        block, state = here
        for code, own in blocks[block][1]:
            branch = BRANCH.match(code)
            if branch:
                if branch.group(1) == "cbranch_execz":
                    continue
                todo.append((at[branch.group(2)], state))
                if branch.group(1) == "branch":
                    break
                continue
            state = step(code, own, state)
            if code.startswith("s_endpgm"):
                break
        else:
            if block + 1 < len(blocks):
                todo.append((block + 1, state))


def after_wait(queue, left):
    return queue[len(queue) - left:] if 0 < left < len(queue) else queue if left > 0 else ()


def check_panel(name, body):
    """Raises AssertionError where a chunk's inputs may not be in LDS yet at the barrier that says they are."""
    assert "scratch_" not in body, f"{name}: spills"

    def step(code, own, state):
        first, queue = state  # oldest first: the barriers passed since an input was asked for, None for any other operation
        if code.startswith("global_load_lds"):
            queue += (0,)
        elif MEMORY.match(code):
            queue += (None,)
        elif code.startswith("s_waitcnt"):
            left = re.search(r"vmcnt\((\d+)\)", code)
            if left:
                queue = after_wait(queue, int(left.group(1)))
        elif code.startswith("s_barrier"):
            late = sum(1 for age in queue if age is not None and (first or age > 0))
            assert late == 0, f"{name}: {late} loads to LDS may still be on their way at the barrier that needs them"
            first, queue = False, tuple(None if age is None else age + 1 for age in queue)
        elif code.startswith("s_endpgm"):
            assert all(age is None for age in queue), f"{name}: loads to LDS on their way at the end"
        while queue and queue[0] is None:
            queue = queue[1:]
        return first, queue

    follow(body, (True, ()), step)


def registers(code):
    """The vector registers an instruction names."""
    named = set()
    for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", code):
        named.update(range(int(a), int(b) + 1))
    named.update(int(v) for v in re.findall(r"\bv(\d+)\b", code))
    return frozenset(named)


def check_registers(name, body):
    """Raises AssertionError where an instruction names a register that a load written by hand has yet to write."""
    assert "scratch_" not in body, f"{name}: spills"
    nothing = frozenset()

    def step(code, own, state):
        memory, lds = state  # oldest first: the registers that each operation on its way writes (of loads written by hand)
        touched = registers(code) & nothing.union(*memory, *lds) if memory or lds else nothing
        assert not touched, f"{name}: `{code}` names v{sorted(touched)} while a load to it is on its way"
        if code.startswith("ds_"):
            lds += (registers(code.split(",")[0]) if own and code.startswith("ds_read") else nothing,)
        elif code.startswith("s_load"):
            lds += (nothing,)
        elif MEMORY.match(code):
            to_register = own and re.match(r"global_load_dword(x[234])?\s", code)
            memory += (registers(code.split(",")[0]) if to_register else nothing,)
        elif code.startswith("s_waitcnt"):
            left = re.search(r"vmcnt\((\d+)\)", code)
            if left:
                memory = after_wait(memory, int(left.group(1)))
            left = re.search(r"lgkmcnt\((\d+)\)", code)
            if left:
                lds = after_wait(lds, int(left.group(1)))
        elif code.startswith("s_endpgm"):
            assert not any(memory) and not any(lds), f"{name}: a load to a register on its way at the end"
        while memory and not memory[0]:
            memory = memory[1:]
        while lds and not lds[0]:
            lds = lds[1:]
        return memory, lds

    follow(body, ((), ()), step)


RING_STAGES = 4  # exl3.hip's kRingDepth
ASK_LEAST = 16   # words of a stage that a lane asks for at a time, at least


def check_ring(name, body, loads):
    """Raises AssertionError where a stage of the ring (`loads` loads to LDS, in order) may not have landed when its words are
    asked for, or is asked for again while the words of the stage in its place may still be on their way. An ask is a run
    of reads of LDS written by hand with no wait among them (shorter runs read the activations, which lie apart). Of two parts
    that lanes go through by a condition, a load in the second is one in the first for the other lanes, as far as those go."""

    def step(code, own, state):
        # Loads to LDS issued since the first load of the oldest stage whose words have not come; of the stages since, those
        # asked for; the reads of LDS since the last wait; the memory operations on their way, oldest first, True: to LDS.
        # And the loads to LDS of a part under a condition (-1: in none), and of the first part's those the second has yet to repeat.
        held, asked, reads, queue, part, again = state
        if code.startswith("global_load_lds"):
            held, again, part = held + (again == 0), max(again - 1, 0), part + (part >= 0)
            queue += (True,)
            assert held <= RING_STAGES * loads, f"{name}: a stage is filled again before its words have come"
        elif MEMORY.match(code):
            queue += (False,)
        elif own and code.startswith("ds_read"):
            reads += 1
            if reads == ASK_LEAST:
                asked += 1
                late = sum(queue) - (held - asked * loads)
                assert late <= 0, f"{name}: {late} loads of a stage may be on their way when its words are asked for"
        elif code.startswith("s_waitcnt"):
            left = re.search(r"vmcnt\((\d+)\)", code)
            if left:
                queue = after_wait(queue, int(left.group(1)))
            if "lgkmcnt(0)" in code:
                held -= asked * loads
                asked, reads = 0, 0
        elif "_saveexec_b64" in code:
            part, again = 0, max(part, 0) if code.startswith("s_andn2") else 0
        elif code.startswith("s_or_b64 exec"):
            part, again = -1, 0
        while queue and not queue[0]:
            queue = queue[1:]
        return held, asked, reads, queue, part, again

    follow(body, (0, 0, 0, (), -1, 0), step)


def ring_loads(name):
    """Of a packed product: its loads to LDS a stage, 256 bytes a bit of a weight, a KB a load."""
    bits = int(re.search(r"ProductKernelILi\d+ELi(\d+)E", name).group(1))
    return (bits * 256 + 1023) // 1024


def check():
    """The number of kernels followed; raises AssertionError (or the compiler's error) where a count does not hold."""
    with concurrent.futures.ThreadPoolExecutor() as pool:
        decode, exl3 = pool.map(assembly_of, ("decode.hip", "exl3.hip"))
    kernels = 0
    for name, body in kernels_of(decode, "DecodeMatrixPanelKernel"):
        check_panel(name, body)
        kernels += 1
    assert kernels >= 5, f"only {kernels} kernels of the matrix product over laid-out inputs were found"
    products = 0
    for name, body in kernels_of(exl3, "WideProductKernel|13ProductKernel"):
        check_registers(name, body)
        check_ring(name, body, ring_loads(name))
        products += 1
    assert products >= 48, f"only {products} packed products were found"
    return kernels + products


if __name__ == "__main__":
    print(f"{check()} kernels wait for their loads by counts that hold in this build")

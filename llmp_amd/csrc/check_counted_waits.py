"""Kernels that ask for loads the compiler does not track (written as instructions) wait for them by count: `vmcnt(n)` lets
the n youngest operations stay on their way, and n counts other loads of the kernel among them, the compiler's own too. A
load that the compiler takes out or joins with another makes such a wait too short, silently. So this build step reads the
compiler's assembly and follows the counter along every path of every such kernel (a state is the queue of operations on
their way; a branch goes both ways, except over an empty execution mask, which none of these kernels has in its loops).

decode.hip, the matrix product over laid-out inputs: inputs go to LDS three chunks ahead, a barrier a chunk. At a barrier
only those asked for since the barrier before may be on their way (at the first, and at the end, none).

Needs hipcc, no GPU. Run by the library's build (__graft_entry__.build) and by tests/test_counted_waits.py;
`python check_counted_waits.py` runs it alone."""
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


def check():
    """The number of kernels followed; raises AssertionError (or the compiler's error) where a count does not hold."""
    kernels = 0
    for name, body in kernels_of(assembly_of("decode.hip"), "DecodeMatrixPanelKernel"):
        check_panel(name, body)
        kernels += 1
    assert kernels >= 5, f"only {kernels} kernels of the matrix product over laid-out inputs were found"
    return kernels


if __name__ == "__main__":
    print(f"{check()} kernels wait for their loads by counts that hold in this build")

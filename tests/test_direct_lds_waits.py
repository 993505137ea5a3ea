"""The few-row prefill GEMMs' direct-to-LDS loads have landed where a barrier
publishes them, on every path of the built kernels.

Those kernels (prefill.hip, SmallWave) count outstanding loads by hand
(s_waitcnt vmcnt(n)). Such a count holds only for the loads that are really in
the code: a weight load whose result no later step uses is removed by the
compiler, and a wait that counted it then waits for less. This test follows
the gfx950 code of the built libfmx.so: a step reads what the step before the
last one requested, so at a barrier no direct-to-LDS load issued before the
previous barrier may be outstanding."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "freemoe_amd" / "libfmx.so"
LLVM = Path("/opt/rocm/llvm/bin")

VM = re.compile(r"(global|buffer|flat|scratch)_(load|store|atomic)")


def code_objects():
    """The gfx950 code objects in libfmx.so's offload bundles."""
    data, at = LIB.read_bytes(), 0
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    while (at := data.find(magic, at)) >= 0:
        entry = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(magic))[0]):
            off, size, name_len = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + name_len] and size:
                yield data[at + off:at + off + size]
            entry += 24 + name_len
        at += len(magic)


def kernels(code, tmp_path):
    """{symbol: [(address, mnemonic, operands, branch target or None)]} of the
    few-row GEMM kernels in one code object."""
    if b"small_down_kernel" not in code:
        return {}
    obj = tmp_path / "code.elf"
    obj.write_bytes(code)
    text = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", obj], check=True, text=True,
                          capture_output=True).stdout
    found, base = {}, {}
    body = None
    for line in text.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.+)>:$", line)
        if head:
            base[head[2]] = int(head[1], 16)
            body = found.setdefault(head[2], []) if "small_" in head[2] else None
            continue
        ins = body is not None and re.match(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)$", line)
        if ins:
            to = re.search(r"<([^>+]+)(?:\+0x([0-9a-f]+))?>", ins[4])
            target = base[to[1]] + int(to[2] or "0", 16) if to and "branch" in ins[1] else None
            body.append((int(ins[3], 16), ins[1], ins[2], target))
    return found


def unwaited_barriers(code):
    """Addresses of the barriers that some path reaches with a direct-to-LDS
    load of before its previous barrier outstanding."""
    index = {ins[0]: i for i, ins in enumerate(code)}
    bad, seen, todo = set(), set(), [(0, "")]
    while todo:
        i, queue = todo.pop()  # queue, oldest first: o / n a load into LDS before / since the last barrier, w another
        while i < len(code):
            if (i, queue) in seen:
                break
            seen.add((i, queue))
            address, op, operands, target = code[i]
            if "load_lds" in op:
                queue += "n"
            elif VM.match(op):
                queue += "w"
            elif op == "s_waitcnt" and (n := re.search(r"vmcnt\((\d+)\)", operands)):
                queue = queue[max(0, len(queue) - int(n[1])):]
            elif op == "s_barrier":
                if "o" in queue:
                    bad.add(address)
                queue = queue.replace("n", "o")
            elif op == "s_endpgm":
                break
            queue = queue[-64:]  # vmcnt counts no further
            if target is not None:
                if op == "s_branch":
                    i = index[target]
                    continue
                todo.append((index[target], queue))
            i += 1
    return bad


@pytest.fixture(scope="module")
def small_kernels(tmp_path_factory):
    if not LIB.exists():
        from freemoe_amd import build
        build.build()
    tmp = tmp_path_factory.mktemp("code")
    return {name: code for obj in code_objects() for name, code in kernels(obj, tmp).items() if code}


def test_few_row_gemms_wait_for_their_direct_lds_loads(small_kernels):
    kinds = [n for n in small_kernels if "small_gate_up_kernel" in n or "small_down_kernel" in n]
    assert len(kinds) == 6  # gate/up and down of Q8_0, Q4_0 and Q4_K
    for name in kinds:
        code = small_kernels[name]
        assert sum("load_lds" in ins[1] for ins in code) > 0 and sum(ins[1] == "s_barrier" for ins in code) > 8
        assert unwaited_barriers(code) == set(), name


def test_the_walk_follows_waits_barriers_and_branches():
    """The walk itself on hand-written streams: a load left outstanding over
    its barrier, the same waited for, and one left only round a loop."""
    load, other, barrier, end = ("global_load_lds_dwordx4", ""), ("global_load_dwordx4", ""), ("s_barrier", ""), ("s_endpgm", "")

    def stream(*ops):
        return [(4 * i, o[0], o[1], o[2] if len(o) > 2 else None) for i, o in enumerate(ops)]

    wait = lambda n: ("s_waitcnt", f"vmcnt({n}) lgkmcnt(0)")
    assert unwaited_barriers(stream(load, barrier, load, wait(1), barrier, end)) == set()
    assert unwaited_barriers(stream(load, barrier, load, wait(2), barrier, end)) == {16}
    assert unwaited_barriers(stream(load, barrier, load, other, wait(2), barrier, end)) == set()
    # the loop's second round reaches the barrier with the first round's load
    assert unwaited_barriers(stream(load, other, wait(2), barrier, ("s_cbranch_scc1", "", 0), end)) == set()
    assert unwaited_barriers(stream(load, wait(2), barrier, ("s_cbranch_scc1", "", 0), end)) == {8}

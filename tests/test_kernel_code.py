"""The search kernel's machine code, as it is built: what no run shows reliably."""
import os
import re
import struct
import subprocess

import pytest

from splishsplash_for_cuda_amd import build

LIB = os.path.join(build.HERE, "libdfsph_hip.so")
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "llvm", "bin", "llvm-objdump")


def _code_objects():
    """the gfx950 code objects in the library's offload bundles"""
    data = open(LIB, "rb").read()
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, length = struct.unpack_from("<QQQ", data, entry)
            if size and b"gfx950" in data[entry + 24:entry + 24 + length]:
                yield data[at + off:at + off + size]
            entry += 24 + length
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> [(address, instruction, branch target or None)]"""
    out = {}
    path = str(tmp_path_factory.mktemp("code") / "code.co")
    for obj in _code_objects():
        with open(path, "wb") as f:
            f.write(obj)
        text = subprocess.run([OBJDUMP, "-d", path], check=True, capture_output=True, text=True).stdout
        body, start = None, 0
        for line in text.splitlines():
            head = re.match(r"([0-9a-f]{16}) <(\w+)>:", line)
            if head:
                start, body = int(head[1], 16), out.setdefault(head[2], [])
                continue
            code = re.match(r"\t(.*?)\s*// ([0-9A-F]{12}):[^<]*(?:<\w+(?:\+0x([0-9a-f]+))?>)?", line)
            if code and body is not None:
                branch = re.match(r"s_c?branch", code[1])
                body.append((int(code[2], 16), code[1], start + int(code[3] or "0", 16) if branch else None))
    assert out
    return out


def _barriers_after(body, at):
    """addresses of the barriers (None: the kernel's end) that a wavefront comes to next, after instruction `at`"""
    index = {a: k for k, (a, _, _) in enumerate(body)}
    found, seen, todo = set(), set(), [at + 1]
    while todo:
        k = todo.pop()
        if k in seen:
            continue
        seen.add(k)
        addr, text, target = body[k]
        if text.startswith("s_barrier"):
            found.add(addr)
            continue
        if text.startswith("s_endpgm"):
            found.add(None)
            continue
        if target is not None:
            todo.append(index[target])
        if not text.startswith("s_branch"):
            todo.append(k + 1)
    return found


def test_search_barrier_between_boxes_and_statistics(kernels):
    """The wavefronts' boxes and the block's statistics share words of LDS: after the barrier that
    completes the boxes, a wavefront that has read them meets another one on every way to the
    last, in front of which it stores its statistics."""
    names = [n for n in kernels if "k_neighborsILb0E" in n]
    assert len(names) == 1
    body = kernels[names[0]]
    barriers = [k for k, (_, text, _) in enumerate(body) if text.startswith("s_barrier")]
    assert len(barriers) > 4
    last = {body[k][0] for k in barriers if None in _barriers_after(body, k)}
    assert last and body[barriers[0]][0] not in last
    assert not _barriers_after(body, barriers[0]) & last


def _scalars(operand):
    """the scalar registers that an operand names"""
    if re.search(r"\bvcc\b", operand):
        return {"vcc"}
    m = re.match(r"-?\|?s\[(\d+):(\d+)\]", operand)
    if m:
        return {"s%d" % k for k in range(int(m[1]), int(m[2]) + 1)}
    m = re.match(r"-?\|?(s\d+)\b", operand)
    return {m[1]} if m else set()


def test_wait_states_behind_scalar_results(kernels):
    """A vector instruction that reads a scalar register or VCC which another vector instruction has
    written comes at least three instructions behind it (two wait states, the rule on
    gfx940 and later): the compiler sees to it, except inside inline assembly."""
    early, pairs = [], 0
    for name, body in kernels.items():
        written = {}                                    # register -> wait states passed since
        for addr, text, _ in body:
            op, _, rest = text.partition(" ")
            operands = [o.strip() for o in rest.split(",")]
            if op.startswith("v_"):
                second = re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale|v_mad_[ui]64", op)
                results = operands[:2] if second else operands[:1]
                reads = set().union(*map(_scalars, operands[len(results):])) | ({"vcc"} if "div_fmas" in op else set())
                for r in reads & written.keys():
                    pairs += 1
                    if written[r] < 2:
                        early.append("%s %x: %s" % (name, addr, text))
            waits = 1 + int(operands[0]) if op == "s_nop" else 1
            written = {r: w + waits for r, w in written.items() if w < 8}
            if op.startswith("v_"):
                written.update((r, 0) for r in set().union(*map(_scalars, results)))
            else:                                       # a scalar result takes its place
                for r in _scalars(operands[0]):
                    written.pop(r, None)
            if op == "s_branch":
                written = {}
    assert pairs > 100 and not early, early[:8]

"""What the compiler made of kernels whose correctness or speed hangs on it: the built library's own gfx950 code, read back (no GPU).

A wait of the form `s_waitcnt vmcnt(N)` lets a wave's N newest memory requests go on. Written in the source with a count, it is right
only if the compiler kept every request that the count has in mind."""
import functools
import re
import shutil
import struct
import subprocess
import tempfile

import pytest

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:/opt/rocm/bin")
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The gfx950 ELF images of every offload bundle in a host library: magic, u64 count, then (u64 offset, u64 size, u64 length, triple)."""
    at = blob.find(BUNDLE)
    while at >= 0:
        pos = at + len(BUNDLE)
        count, = struct.unpack_from("<Q", blob, pos)
        pos += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in triple and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(BUNDLE, at + len(BUNDLE))


@functools.lru_cache(maxsize=None)
def kernels(part):
    """{symbol: [(address, instruction, branch target or None)]} of the kernels whose symbols contain `part`."""
    import fieldfare_moe as ff
    ff.ensure_built()
    found = {}
    for image in _code_objects(ff.LIB_PATH.read_bytes()):
        if part.encode() not in image:
            continue
        with tempfile.NamedTemporaryFile(suffix=".co") as f:
            f.write(image)
            f.flush()
            names = subprocess.run([OBJDUMP, "--syms", f.name], capture_output=True, text=True, check=True).stdout
            mine = [s for s in re.findall(r" F \.text\t\S+ (?:\.protected )?(\S+)", names) if part in s]
            if not mine:
                continue
            text = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + ",".join(mine), f.name], capture_output=True, text=True, check=True).stdout
        start, body = 0, None
        for line in text.splitlines():
            head = re.match(r"^([0-9a-f]+) <(\S+)>:$", line)
            if head:
                start, body = int(head[1], 16), found.setdefault(head[2], [])
                continue
            code = re.match(r"^\t(.*?)\s*// ([0-9A-F]+): .*?(?:<\S+?(?:\+0x([0-9a-f]+))?>)?$", line)
            if code and body is not None:
                op = code[1].split("//")[0].strip()
                target = start + int(code[3] or "0", 16) if "branch" in op.split()[0] else None
                body.append((int(code[2], 16), op, target))
    assert found, part
    return found


def _graph(code):
    """Predecessors of each instruction by index."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    before = [[] for _ in code]
    for i, (_, op, target) in enumerate(code):
        if target is not None:
            before[at[target]].append(i)
        if i + 1 < len(code) and not op.startswith(("s_branch", "s_endpgm", "s_setpc")):
            before[i + 1].append(i)
    return before


REQUEST = re.compile(r"(global|buffer|flat|scratch)_(load|store|atomic)")


def _newest(code, before, i, n):
    """For every way to instruction i: of the n newest memory requests in front of it, newest first, which are row loads into LDS."""
    out, todo, seen = set(), [(p, 0, ()) for p in before[i]], set()
    while todo:
        k, taken, rows = todo.pop()
        if (k, taken, rows) in seen:
            continue
        seen.add((k, taken, rows))
        if REQUEST.match(code[k][1]):
            taken += 1
            rows += (code[k][1].startswith("global_load_lds"),)
        if taken >= n or not before[k]:
            out.add(rows)
            continue
        todo += [(p, taken, rows) for p in before[k]]
    return out


@pytest.mark.skipif(OBJDUMP is None, reason="needs llvm-objdump")
def test_the_streaming_products_barriers_cover_the_rows_that_are_read_next():
    # prefill_stream_kernel's ring of row buffers: tiles of up to NM 16-pair blocks ask for NM pieces of rows per wave and chunk, kAhead = buffers - 1
    # chunks ahead. A chunk's barrier has to leave none of the next chunk's in flight, nor (NM > 1, where the block then makes the sums of the chunk behind it)
    # of that one's. So the requests it lets go on may hold the rows of kAhead - 1 chunks (- 2), wherever in the tile it stands.
    checked = 0
    for name, code in kernels("prefill_stream_kernel").items():
        max_nm = int(re.search(r"ILb[01]ELi(\d)", name)[1])
        ahead = 3 if max_nm <= 2 else 2
        before = _graph(code)
        for i, (_, op, _) in enumerate(code):
            wait = re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)", op)
            if not wait or not code[i + 1][1].startswith("s_barrier"):
                continue
            n = int(wait[1])
            for requests in _newest(code, before, i, n):
                rows = "".join("r" if r else "." for r in requests)
                nm = max(map(len, re.findall(r"r+", rows)), default=1)      # (a chunk's loads stand together; the oldest may be cut short)
                chunks = ahead - 1 if nm == 1 else ahead - 2
                assert rows.count("r") <= nm * chunks, f"{name}: at {code[i][0]:x}, vmcnt({n}) over {rows}"
            checked += 1
    assert checked >= 10


@pytest.mark.skipif(OBJDUMP is None, reason="needs llvm-objdump")
def test_the_listed_gemv_asks_for_its_weights_in_one_burst():
    # gemv_int4_mfma_kernel<.., FEW, ONE>, but for the form of neither: six groups of weights and two scales and biases, none of which waits for another or
    # for the input rows' products. Of more than four input rows (not FEW) the burst stands behind the turn of all twelve pieces of 16 bytes.
    checked = 0
    for name, code in kernels("gemv_int4_mfma_kernel").items():
        few, one = re.search(r"ILb[01]ELb[01]ELb[01]ELb[01]ELb([01])ELb([01])E", name).groups()
        if "1" not in few + one:
            continue
        ops = [op for _, op, _ in code]
        front = ops[:next(i for i, op in enumerate(ops) if op.startswith("v_mfma"))]
        at = [i for i, op in enumerate(front) if re.match(r"global_load_(dwordx2|ushort) ", op)]
        assert len(at) == 10, f"{name}: {len(at)} of 10 requests in front of the first product"
        assert not any("vmcnt" in op for op in front[at[0]:at[-1]]), name
        assert sum(op.startswith("ds_bpermute") for op in front[:at[0]]) == (0 if few == "1" else 48), name
        checked += 1
    assert checked == 36


@pytest.mark.skipif(OBJDUMP is None, reason="needs llvm-objdump")
def test_the_one_row_down_launch_refills_nothing():
    # A wave of decode_down_combine_kernel walks one tile row: no slot of its ring is wanted twice. A refill named all the same is dropped by
    # the compiler, but its fences stay and hold the arithmetic of a step in its place, for 218 registers instead of 176. What a wave cannot do
    # without at once is eleven groups of weights (6 registers) and of its row (8), i.e. 154; 192 leaves room for addresses and sums.
    for name, code in kernels("decode_down_combine_kernel").items():
        registers = [int(n) for _, op, _ in code for n in re.findall(r"\bv\[?(?:\d+:)?(\d+)", op)]
        assert max(registers) < 192, f"{name}: {max(registers) + 1} registers"

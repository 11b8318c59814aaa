"""Waits that the sources promise by count, looked up in the built library's code for every way through a kernel: data that asynchronous
loads and copies bring must have arrived before it is touched.  The compiler does not see these orders, so another compiler, another register budget or
another epilogue can break them without a warning, and a run on the GPU need not show it."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

VMEM = re.compile(r"(buffer|global|flat|scratch)_(load|store|atomic)")


def code_objects(tmp_path):
    """The gfx950 code objects in libsglq.so, a file each."""
    from sglang_amd import build

    path = build.LIB_PATH if build.LIB_PATH.exists() else build.build()
    data, magic, at = Path(path).read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            name, entry = data[entry + 24:entry + 24 + length], entry + 24 + length
            if name.endswith(b"gfx950"):
                out = tmp_path / f"{at:x}.co"
                out.write_bytes(data[at + offset:at + offset + size])
                yield out
        at += len(magic)


def kernels(tmp_path, pattern):
    """name -> basic blocks {address: ([(op, operands)], [successors])} of the kernels whose name matches."""
    bin_dir = next((d for d in (Path("/opt/rocm/llvm/bin"), Path("/opt/rocm/lib/llvm/bin")) if (d / "llvm-objdump").exists()), None)
    if bin_dir is None:
        pytest.skip("no llvm-objdump")
    found = {}
    for co in code_objects(tmp_path):
        symbols = subprocess.run([bin_dir / "llvm-readelf", "-s", "--wide", co], capture_output=True, text=True, check=True).stdout
        names = {w[-1] for w in map(str.split, symbols.splitlines()) if len(w) >= 8 and w[3] == "FUNC" and re.search(pattern, w[-1])}
        if not names:
            continue
        text = subprocess.run([bin_dir / "llvm-objdump", "-d", "--mcpu=gfx950", "--disassemble-symbols=" + ",".join(names), co],
                              capture_output=True, text=True, check=True).stdout
        for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
            head = re.match(r"([0-9a-f]+) <(\S+)>:", part)
            if head and head[2] in names:
                found[head[2]] = blocks(part, int(head[1], 16))
    return found


def blocks(text, base):
    code = []
    for line in text.splitlines():
        m = re.match(r"\s+(\w+)\s*(.*?)\s*// ([0-9A-F]+):(.*)", line)
        if m:
            target = re.search(r"<\S+?(?:\+0x([0-9a-f]+))?>", m[4]) if m[1].startswith(("s_branch", "s_cbranch")) else None
            code.append((int(m[3], 16), m[1], m[2], base + int(target[1] or "0", 16) if target else None))
    starts = {code[0][0]} | {t for *_, t in code if t is not None}
    starts |= {code[i + 1][0] for i, c in enumerate(code[:-1]) if c[3] is not None or c[1] == "s_endpgm"}
    result, current = {}, None
    for i, (addr, op, operands, target) in enumerate(code):
        assert op not in ("s_setpc_b64", "s_swappc_b64"), "no calls are followed"
        if addr in starts:
            if current is not None and not result[current][2]:
                result[current][1].append(addr)
            current = addr
            result[current] = ([], [], [])
        result[current][0].append((op, operands))
        if target is not None or op == "s_endpgm":
            result[current][2].append(True)
            if target is not None:
                result[current][1].append(target)
            if op.startswith("s_cbranch"):
                result[current][1].append(code[i + 1][0])
    return {a: (ins, succ) for a, (ins, succ, _) in result.items()}


def vmcnt(op, operands):
    m = re.search(r"vmcnt\((\d+)\)", operands) if op == "s_waitcnt" else None
    return int(m[1]) if m else None


def walk(code, start, step, meet):
    """Forward data flow: step(state, op, operands) -> state, meet(old or None, new) -> state, until nothing changes."""
    first = min(code)
    at, todo = {first: start}, [first]
    while todo:
        a = todo.pop()
        state = at[a]
        for op, operands in code[a][0]:
            state = step(state, op, operands)
        for s in code[a][1]:
            merged = meet(at.get(s), state)
            if merged != at.get(s):
                at[s] = merged
                todo.append(s)


def registers(operands):
    out = set()
    for a, b in re.findall(r"\bv(?:\[(\d+):(\d+)\])", operands):
        out |= set(range(int(a), int(b) + 1))
    return out | {int(r) for r in re.findall(r"\bv(\d+)\b", operands)}


def test_linears_touch_no_activation_before_it_has_arrived(tmp_path):
    """gemm_stream_quant_kernel and gemm_stream_tokenquant_kernel load their activations into registers behind the compiler's back."""
    found = kernels(tmp_path, r"gemm_stream_(token)?quant_kernel")
    assert len(found) == 96
    for name, code in found.items():
        loads = [0]

        def step(state, op, operands):  # state: register -> the fewest vector-memory operations younger than its load
            count = vmcnt(op, operands)
            if count is not None:
                return {r: c for r, c in state.items() if c < count}
            touched = registers(operands)
            load = op == "buffer_load_dwordx4" and not operands.endswith("lds")
            fresh = registers(operands.split(",")[0]) if load else set()
            assert not touched & set(state) - fresh, f"{name}: {op} {operands}"
            if VMEM.match(op):
                state = {r: min(c + 1, 64) for r, c in state.items()}
            loads[0] += load
            return {**state, **{r: 0 for r in fresh}}

        walk(code, {}, step, lambda old, new: new if old is None else {r: min(old.get(r, 64), new.get(r, 64)) for r in old.keys() | new.keys()})
        assert loads[0] >= 16


def test_gathered_rows_are_named_before_they_are_read(tmp_path):
    """PIPE_GATHERED's row maps, copied into LDS by waves 0 to 3 and read by all: the copy is waited for, then a barrier.  Two places in turn: a read with
    no barrier since the copy is one of the place that is not being written.  A tile has sixteen stores and then steps with
    barriers.  Ways with another number of stores mix them with the guarded ones of tiles cut by N, which end in a wait for everything, and ways from tile to
    tile without a barrier take none of the tile's heights: neither is followed."""
    found = kernels(tmp_path, r"gemm_pipe_kernelILi0ELi[01]ELi5ELi256E")
    assert len(found) == 2
    for name, code in found.items():
        seen = {"copy": 0, "read": 0}
        header = min(((t - a, t) for a, (_, succ) in code.items() for t in succ if t < a))[1]  # of the walk over tiles, the longest loop
        code[header][0].insert(0, ("next tile", ""))

        def one(state, op, operands):  # operations younger than the copy (None: handed over); it has landed; barriers since; stores, and another tile, since the last barrier
            younger, landed, barrier, stores, tile = state
            count = vmcnt(op, operands)
            if count is not None:
                return (younger, landed or (younger is not None and count <= younger), barrier, stores, tile)
            if op == "buffer_load_dword" and operands.endswith("lds") and ", 0 offen" in operands:
                seen["copy"] += 1
                return (0, False, False, stores, tile)
            if op.startswith("ds_read2st64_b32"):
                seen["read"] += 1
                assert younger is None or not barrier, f"{name}: {op} {operands} behind a barrier, the copy and {younger} younger operations in flight"
            if op == "next tile":
                return None if tile else (younger, landed, barrier, stores, True)
            if op == "s_barrier":
                if younger is None or landed:
                    return (None, False, False, 0, False)
                return (younger, False, True, 0, False) if barrier or stores == 16 else None
            if VMEM.match(op):
                return (younger if younger is None else min(younger + 1, 64), landed, barrier, min(stores + op.startswith("buffer_store"), 17), tile)
            return state

        step = lambda states, op, operands: frozenset(filter(None, (one(s, op, operands) for s in states)))
        walk(code, frozenset([(None, False, False, 0, False)]), step, lambda old, new: new if old is None else old | new)
        assert seen["copy"] >= 2 and seen["read"] >= 18  # (two reads a map: in front of the walk, and at two steps of each of the four heights)


@pytest.mark.parametrize("mode,tile_stores,inner_barriers", [(7, 16, 0), (9, 5, 1)])
def test_walked_rows_are_named_before_they_are_read(tmp_path, mode, tile_stores, inner_barriers):
    """The same of PIPE_WALKED_GATHERED and of PIPE_SILU_GATHERED, whose tiles have five stores, and a barrier between the copy of the row map and these."""
    found = kernels(tmp_path, rf"gemm_pipe_kernelILi0ELi[01]ELi{mode}ELi256E")
    assert len(found) == 2
    for name, code in found.items():
        seen = {"copy": 0, "read": 0, "handed over": 0}
        header = min(((t - a, t) for a, (_, succ) in code.items() for t in succ if t < a))[1]  # of the walk over tiles, the longest loop
        code[header][0].insert(0, ("next tile", ""))

        def one(state, op, operands):  # operations younger than the copy (None: handed over); it has landed; barriers since (behind the tile's stores); stores; barriers in front of these; another tile
            younger, landed, barrier, stores, inner, tile = state
            count = vmcnt(op, operands)
            if count is not None:
                return (younger, landed or (younger is not None and count <= younger), barrier, stores, inner, tile)
            if op == "buffer_load_dword" and operands.endswith("lds") and ", 0 offen" in operands:
                seen["copy"] += 1
                return (0, False, False, 0, 0, tile)
            if op.startswith("ds_read2st64_b32"):
                seen["read"] += 1
                assert younger is None or not barrier, f"{name}: {op} {operands} behind a barrier, the copy and {younger} younger operations in flight"
            if op.startswith("v_exp_f32") and tile:
                return None  # (the activation's epilogue with none of the tile's heights in front of it)
            if op == "next tile":
                return None if tile else (younger, landed, barrier, stores, inner, True)
            if op == "s_barrier":
                if younger is None or landed:
                    seen["handed over"] += younger is not None
                    return (None, False, False, 0, 0, False)
                if not barrier and stores == 0 and inner < inner_barriers:
                    return (younger, False, False, 0, inner + 1, tile)
                # (ways with another number of stores are none: they mix branches on the same condition)
                return (younger, False, True, 0, inner, False) if barrier or (stores == tile_stores and inner == inner_barriers) else None
            if VMEM.match(op):
                return (younger if younger is None else min(younger + 1, 64), landed, barrier, min(stores + op.startswith("buffer_store"), 17), inner, tile)
            return state

        step = lambda states, op, operands: frozenset(filter(None, (one(s, op, operands) for s in states)))
        walk(code, frozenset([(None, False, False, 0, 0, False)]), step, lambda old, new: new if old is None else old | new)
        assert seen["copy"] >= 2 and seen["read"] >= 18 and seen["handed over"] >= 2

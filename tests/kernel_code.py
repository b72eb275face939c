"""Looks through the machine code of the built kernel library for registers that are used while a load into them is
still on its way, and says what its kernels take of registers, LDS and scratch memory.

The compiler waits for the loads that it knows of.  Loads written in assembly it takes as done where they stand, so that
nothing but the kernel's own waits, and where the compiler happens to keep the values, stands between a load and the
first use of its registers: a copy or a spill in between would read what is not there yet."""

import os
import re
import shutil
import struct
import subprocess

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def disassembler():
    for folder in ("/opt/rocm/llvm/bin", "/opt/rocm/lib/llvm/bin"):
        path = os.path.join(folder, "llvm-objdump")
        if os.path.isfile(path):
            return path
    return shutil.which("llvm-objdump")


def code_objects(library, arch):
    """The device code objects inside a shared library: one ELF image per source file."""
    with open(library, "rb") as handle:
        data = handle.read()
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            name = data[entry + 24:entry + 24 + length].decode()
            entry += 24 + length
            if size and arch in name:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


_LINE = re.compile(r"^\t(\S+)(?:[ ]+(.*?))?\s*// ([0-9A-F]+): (?:[0-9A-F ]+?)(?:<[^>]*?(?:\+0x([0-9a-f]+))?>)?$")
_REGISTER = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")
_WAIT = re.compile(r"(vmcnt|lgkmcnt)\((\d+)\)")
_MEMORY = ("global_", "buffer_", "scratch_", "flat_")


def kernels(listing):
    """(name, [(address within the kernel, operation, operands, branch target or None), ...]) of a disassembly."""
    name, start, code = None, 0, []
    for line in listing.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.+)>:$", line)
        if head:
            if name is not None:
                yield name, code
            name, start, code = head[2], int(head[1], 16), []
            continue
        found = _LINE.match(line)
        if found:
            operation = found[1]
            target = int(found[4] or "0", 16) if operation.startswith(("s_branch", "s_cbranch")) else None
            code.append((int(found[3], 16) - start, operation, found[2] or "", target))
    if name is not None:
        yield name, code


def _registers(text):
    out = []
    for kind, low, high, single in _REGISTER.findall(text):
        first, last = (int(low), int(high)) if low else (int(single), int(single))
        out += [(kind, number) for number in range(first, last + 1)]
    return out


def _decode(operation, operands):
    """(counter of a load or store, registers it fills, all registers it names, waits)"""
    waits = {counter: int(count) for counter, count in _WAIT.findall(operands)} if operation == "s_waitcnt" else {}
    named = _registers(operands)
    counter, fills = None, []
    if operation.startswith(_MEMORY):
        counter = "vmcnt"
        if "load" in operation and "_lds" not in operation and " lds" not in operands:
            fills = _registers(operands.split(",")[0])
    elif operation.startswith("ds_"):
        counter = "lgkmcnt"
        if not operation.startswith(("ds_write", "ds_add_u32", "ds_nop")):
            fills = _registers(operands.split(",")[0])
    if fills:      # (filled again by a load of the same kind, which comes back later; its addresses are uses)
        named = _registers(operands.split(",", 1)[1])
    return counter, fills, named, waits


def early_uses(code):
    """[(address, instruction, register)] where a register is named while a load into it may be on its way.

    Per register that is waited for: how many memory operations of its kind were issued behind it at least (they
    come back in order), over all paths; a wait for N of them to be left ends those with N and more behind them."""
    index_of = {address: index for index, (address, _, _, _) in enumerate(code)}
    decoded = [_decode(operation, operands) for _, operation, operands, _ in code]
    starts = {0} | {index_of[target] for _, _, _, target in code if target is not None}
    starts |= {index + 1 for index, line in enumerate(code) if line[3] is not None}
    states, found, work = {0: {}}, {}, [0]

    def flow(state, index):
        if index >= len(code):
            return
        known = states.get(index)
        merged = dict(state) if known is None else dict(known)
        for key, behind in state.items():
            merged[key] = min(merged.get(key, behind), behind)
        if known is None or merged != known:
            states[index] = merged
            work.append(index)

    while work:
        index = work.pop()
        state = dict(states[index])
        while index < len(code):
            address, operation, operands, target = code[index]
            counter, fills, named, waits = decoded[index]
            if state:
                for name, left in waits.items():
                    state = {key: behind for key, behind in state.items() if key[0] != name or behind < left}
                for register in named:
                    if ("vmcnt", register) in state or ("lgkmcnt", register) in state:
                        found[address] = (address, f"{operation} {operands}", register)
                if counter is not None:      # (a counter holds 63 at most: the one before those has come back)
                    state = {key: behind + (key[0] == counter) for key, behind in state.items()
                             if key[0] != counter or behind < 62}
            for register in fills:
                if ("lgkmcnt" if counter == "vmcnt" else "vmcnt", register) in state:
                    found[address] = (address, f"{operation} {operands}", register)
                state[counter, register] = 0
            if target is not None:
                flow(state, index_of[target])
            if operation in ("s_branch", "s_endpgm", "s_setpc_b64"):
                break
            index += 1
            if index in starts:
                flow(state, index)
                break
    return [found[address] for address in sorted(found)]


def disassemble(image, arch, folder):
    path = os.path.join(str(folder), "kernels.elf")
    with open(path, "wb") as handle:
        handle.write(image)
    return subprocess.run([disassembler(), "-d", f"--mcpu={arch}", path], check=True, stdout=subprocess.PIPE,
                          text=True).stdout


def resources(image, folder):
    """{symbol of a kernel: {"vgpr": registers, "scratch" and "lds": bytes}} of a code object, from the notes that the
    compiler leaves in it."""
    path = os.path.join(str(folder), "kernels.elf")
    with open(path, "wb") as handle:
        handle.write(image)
    notes = subprocess.run([os.path.join(os.path.dirname(disassembler()), "llvm-readelf"), "--notes", path], check=True,
                           stdout=subprocess.PIPE, text=True).stdout
    found = {}
    for part in notes.split("- .agpr_count:")[1:]:
        fields = dict(re.findall(r"^    \.(\w+):\s+(\S+)$", part, re.M))
        found[fields["name"]] = {"vgpr": int(fields["vgpr_count"]), "scratch": int(fields["private_segment_fixed_size"]),
                                 "lds": int(fields["group_segment_fixed_size"])}
    return found

"""The machine code of every kernel of the library: no register is read or written while a load into it is on its way, on any path.

The kernels issue many of their loads in inline assembly and wait for them with counts of their own. The compiler knows of neither: it may
copy, spill or reuse a register between a load and its wait, and the result is then wrong now and then, with no error. So the built code is
followed instruction by instruction over all branches: for every register the youngest load into it that no wait covers, counted in
instructions of its counter issued since (vmcnt: loads, stores and atomics, reported in order; lgkmcnt: LDS operations, scalar loads left
out, which makes a count cover less). Loads from memory into LDS have to be over when a wavefront ends."""
import collections
import os
import re
import subprocess

import pytest

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")
LABEL = re.compile(r"^([0-9a-f]+) <(.+)>:$")
LINE = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-Fa-f]+):(.*)$")
TARGET = re.compile(r"<.+\+0x([0-9a-f]+)>\s*$")
Op = collections.namedtuple("Op", "at text uses vm_dest lgkm_dest vm lgkm wait_vm wait_lgkm next ends")
DMA = "LDS"   # stands for the destination of a load from memory into LDS


def regs(text):
    return [k + str(i) for k, n, lo, hi in REG.findall(text) for i in range(int(n or lo), int(n or hi) + 1)]


def kernels(listing):
    """(name, its instructions as (address, operation, operands, rest)) of an objdump listing."""
    name, start, body = None, 0, []
    for line in listing.splitlines():
        m = LABEL.match(line)
        if m:
            if body:
                yield name, start, body
            name, start, body = m[2], int(m[1], 16), []
            continue
        m = LINE.match(line)
        if m:
            body.append((int(m[3], 16), m[1], m[2], m[4]))
    if body:
        yield name, start, body


def decode(start, body):
    place = {b[0]: i for i, b in enumerate(body)}
    out = []
    for i, (at, op, args, rest) in enumerate(body):
        follow = [i + 1] if i + 1 < len(body) else []
        uses, vm_dest, lgkm_dest, vm, lgkm, wait_vm, wait_lgkm = (), (), (), False, False, None, None
        if op == "s_waitcnt":
            m, n = re.search(r"vmcnt\((\d+)\)", args), re.search(r"lgkmcnt\((\d+)\)", args)
            wait_vm, wait_lgkm = m and int(m[1]), n and int(n[1])
        elif op.startswith("s_cbranch") or op == "s_branch":
            to = place[start + int(TARGET.search(rest)[1], 16)]
            follow = [to] if op == "s_branch" else follow + [to]
        elif op == "s_endpgm":
            follow = []
        else:
            assert not op.startswith(("s_setpc", "s_swappc", "s_call")), op   # (everything is inlined)
            first, _, others = args.partition(",")
            if op.startswith(("global_", "buffer_", "flat_", "scratch_")) and not re.search("wbl2|inv", op):
                vm, lgkm = True, op.startswith("flat_")
                if "_lds_" in op or re.search(r"\blds\b", args):
                    vm_dest = (DMA,)
                elif "_load_" in op or ("_atomic_" in op and re.search(r"\b(sc0|glc)\b", args)):
                    vm_dest = tuple(regs(first))
            elif op.startswith("ds_"):
                lgkm = True
                if re.search("read|permute|swizzle|rtn", op):
                    lgkm_dest = tuple(regs(first))
            # (a second load into a register on its way, whose first result nobody wanted, comes after the first)
            uses = tuple(regs(others) if vm_dest or lgkm_dest else regs(args))
            if vm_dest == (DMA,):
                uses = tuple(regs(args))
        out.append(Op(at, op + " " + args, uses, vm_dest, lgkm_dest, vm, lgkm, wait_vm, wait_lgkm, follow, op == "s_endpgm"))
    return out


def faults(prog):
    """{(address, register): instruction} of the instructions that use a register before a wait covers the load into it."""
    heads = {0} | {t for i, p in enumerate(prog) if p.next != [i + 1] for t in p.next + [i + 1]}
    heads = sorted(h for h in heads if h < len(prog))
    end = dict(zip(heads, heads[1:] + [len(prog)]))
    entry, todo, found = {0: ({}, {})}, collections.deque([0]), {}
    while todo:
        head = todo.popleft()
        vm, lgkm = (dict(s) for s in entry[head])   # register -> instructions of the counter since the load into it
        for p in prog[head:end[head]]:
            if vm or lgkm:
                for r in p.uses:
                    if r in vm or r in lgkm:
                        found[p.at, r] = p.text
                for r in p.vm_dest:
                    if r in lgkm:
                        found[p.at, r] = p.text
                for r in p.lgkm_dest:
                    if r in vm:
                        found[p.at, r] = p.text
                if p.ends and DMA in vm:
                    found[p.at, DMA] = p.text
            if p.wait_vm is not None:
                vm = {r: k for r, k in vm.items() if k < p.wait_vm}
            if p.wait_lgkm is not None:
                lgkm = {r: k for r, k in lgkm.items() if k < p.wait_lgkm}
            if p.vm:
                vm = {r: min(k + 1, 64) for r, k in vm.items()}
                vm.update(dict.fromkeys(p.vm_dest, 0))
            if p.lgkm:
                lgkm = {r: min(k + 1, 16) for r, k in lgkm.items()}
                lgkm.update(dict.fromkeys(p.lgkm_dest, 0))
        for t in prog[end[head] - 1].next:
            if t not in entry:
                entry[t] = (dict(vm), dict(lgkm))
                todo.append(t)
                continue
            changed = False
            for old, new in zip(entry[t], (vm, lgkm)):
                for r, k in new.items():
                    if old.get(r, 99) > k:
                        old[r], changed = k, True
            if changed and t not in todo:
                todo.append(t)
    return found


def _listing(*lines):
    """A kernel of four-byte instructions; `-> n` names the instruction that a branch goes to."""
    out = ["0000000000000100 <k>:"]
    for i, line in enumerate(lines):
        text, _, to = line.partition(" -> ")
        out.append("\t%s // %012X: 00000000%s" % (text, 0x100 + 4 * i, " <k+0x%x>" % (4 * int(to)) if to else ""))
    return "\n".join(out)


@pytest.mark.parametrize("lines,at", [
    (["global_load_dwordx4 v[0:3], v[4:5], off", "s_waitcnt vmcnt(0)", "v_mov_b32_e32 v6, v3", "s_endpgm"], None),
    (["global_load_dwordx4 v[0:3], v[4:5], off", "v_mov_b32_e32 v6, v3", "s_endpgm"], 1),                                # read
    (["global_load_dwordx4 v[0:3], v[4:5], off", "v_mov_b32_e32 v2, v6", "s_endpgm"], 1),                                # written
    (["global_load_dword v0, v[4:5], off", "global_store_dword v[4:5], v7, off", "s_waitcnt vmcnt(1)", "v_mov_b32_e32 v6, v0", "s_endpgm"], None),
    (["global_load_dword v0, v[4:5], off", "global_store_dword v[4:5], v7, off", "s_waitcnt vmcnt(2)", "v_mov_b32_e32 v6, v0", "s_endpgm"], 3),
    (["ds_read_b128 v[0:3], v8", "ds_read_b64_tr_b16 v[4:5], v8", "s_waitcnt lgkmcnt(1)", "v_add_f32_e32 v6, v0, v1", "s_endpgm"], None),
    (["ds_read_b128 v[0:3], v8", "ds_read_b64_tr_b16 v[4:5], v8", "s_waitcnt lgkmcnt(1)", "v_add_f32_e32 v6, v0, v5", "s_endpgm"], 3),
    (["ds_read_b128 v[0:3], v8", "s_waitcnt vmcnt(0)", "v_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], v[4:7], v[16:31]", "s_endpgm"], 2),
    # a way round the wait, and one that comes back in front of the load
    (["global_load_dword v0, v[4:5], off", "s_cbranch_scc1 1 -> 3", "s_waitcnt vmcnt(0)", "v_mov_b32_e32 v6, v0", "s_endpgm"], 3),
    (["v_mov_b32_e32 v6, v0", "global_load_dword v0, v[4:5], off", "s_cbranch_scc1 9 -> 0", "s_waitcnt vmcnt(0)", "s_endpgm"], 0),
    (["global_load_lds_dwordx4 v[4:5], off", "s_waitcnt vmcnt(0)", "s_endpgm"], None),
    (["global_load_lds_dwordx4 v[4:5], off", "v_mov_b32_e32 v4, 0", "s_endpgm"], 2),
])
def test_the_check_itself(lines, at):
    (_, start, body), = kernels(_listing(*lines))
    assert sorted({(a - 0x100) // 4 for a, _ in faults(decode(start, body))}) == ([] if at is None else [at])


def test_no_register_is_used_while_a_load_into_it_is_on_its_way(tmp_path):
    from trainium_frontier_them_bones_amd import build
    if not os.path.exists(build.LIB_PATH):
        pytest.skip("library not built (run __graft_entry__.build())")

    def tool(name, *args):
        return subprocess.run([os.path.join(LLVM, name), *args], check=True, capture_output=True, text=True).stdout

    fat = tmp_path / "fatbin"
    tool("llvm-objcopy", "--dump-section", ".hip_fatbin=%s" % fat, build.LIB_PATH, str(tmp_path / "copy"))
    data = fat.read_bytes()
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)]
    seen, bad = 0, []
    for n, (a, b) in enumerate(zip(starts, starts[1:] + [len(data)])):
        bundle, code = tmp_path / ("bundle%d" % n), tmp_path / ("code%d" % n)
        bundle.write_bytes(data[a:b])
        tool("clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=%s" % bundle, "--output=%s" % code)
        for name, start, body in kernels(tool("llvm-objdump", "-d", str(code))):
            seen += 1
            bad += ["%s: %s at %x: %s" % (name, r, at, text) for (at, r), text in sorted(faults(decode(start, body)).items())[:3]]
    assert seen > 300 and not bad, "\n".join(bad[:20])

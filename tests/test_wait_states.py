"""Wait states of the memory instructions in the built library's gfx950 code. The direct-to-LDS loads of the prefill GEMMs
are inline asm, which the compiler's hazard pass does not look into, so the rules it keeps for its own memory
instructions are checked on the listing, along every path (fall-through and branch edges):
  - an SGPR written by a VALU instruction (v_readfirstlane, the v_readlane of a spilled SGPR, a compare) may be read by a
    memory instruction only five wait states later: an address base read too early is an old one;
  - m0 must be written one wait state before a load to LDS, and not by a VALU instruction within five."""
import collections
import re
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def sgprs(operand):
    m = re.match(r"s\[(\d+):(\d+)\]$", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"s(\d+)$", operand)
    return {int(m[1])} if m else {"vcc"} if operand == "vcc" else {"m0"} if operand == "m0" else set()


def functions(text):
    """name -> [(address, mnemonic, operands, branch target)]"""
    out, name = {}, None
    for line in text.splitlines():
        m = re.match(r"([0-9a-f]{16}) <(.*)>:$", line)
        if m:
            name = m[2]
            out[name], base = [], int(m[1], 16)
            continue
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):(.*)$", line)
        if m and name:
            t = re.search(r"<[^>]*\+0x([0-9a-f]+)>$", m[4]) if m[1].startswith(("s_cbranch", "s_branch")) else None
            out[name].append((int(m[3], 16), m[1], m[2].replace(",", " ").split(), base + int(t[1], 16) if t else None))
    return out


def written(mnemonic, ops):
    w = sgprs(ops[0]) if ops else set()
    return w | sgprs(ops[1]) if "_co_" in mnemonic and len(ops) > 1 else w


def violations(ins):
    at = {a: i for i, (a, *_) in enumerate(ins)}
    preds = collections.defaultdict(list)
    for i, (_, op, _, target) in enumerate(ins):
        if target in at:
            preds[at[target]].append(i)
        if op not in ("s_branch", "s_endpgm"):
            preds[i + 1].append(i)

    def before(i, states, hit):
        """Instructions within `states` wait states before instruction i that hit."""
        found, todo, seen = [], [(p, 0) for p in preds[i]], {}
        while todo:
            p, d = todo.pop()
            if d >= states or seen.get(p, states) <= d:
                continue
            seen[p] = d
            _, op, ops, _ = ins[p]
            if hit(op, ops):
                found.append(f"{op} {' '.join(ops)}")
                continue
            cost = int(ops[0], 0) + 1 if op == "s_nop" else 1
            todo += [(q, d + cost) for q in preds[p]]
        return found

    loads, bad = 0, []
    for i, (addr, op, ops, _) in enumerate(ins):
        if not op.startswith(("global_", "buffer_", "scratch_", "flat_")):
            continue
        need = set().union(*(sgprs(o) for o in ops)) if ops else set()
        to_lds = "_lds_" in op or "lds" in ops
        loads += to_lds
        late = before(i, 5, lambda o, a: o.startswith("v_") and written(o, a) & (need | ({"m0"} if to_lds else set())))
        if to_lds:
            late += before(i, 1, lambda o, a: "m0" in written(o, a))
        bad += [f"{addr:x}: {w} -> {op} {' '.join(ops)}" for w in late]
    return loads, bad


def test_the_check_sees_a_missing_wait():
    """The rules on a listing of three instructions: too close, far enough, and close over a loop edge."""
    listing = """
0000000000001000 <k>:
\tv_readlane_b32 s67, v245, 35     // 000000001000: 00000000
\ts_mov_b64 exec, s[4:5]           // 000000001004: 00000000
{}
\tglobal_load_lds_dwordx4 v195, s[66:67]  // 000000001010: 00000000
"""
    near = violations(functions(listing.format("\ts_nop 1   // 000000001008: 00000000"))["k"])
    far = violations(functions(listing.format("\ts_nop 3   // 000000001008: 00000000"))["k"])
    assert near[0] == far[0] == 1 and len(near[1]) == 1 and not far[1]
    loop = """
0000000000001000 <k>:
\tglobal_load_dword v1, v2, s[8:9]   // 000000001000: 00000000
\ts_nop 7                            // 000000001004: 00000000
\tv_readfirstlane_b32 s8, v3         // 000000001008: 00000000
\ts_cbranch_scc1 65532               // 00000000100C: BF85FFFC <k+0x0>
"""
    assert len(violations(functions(loop)["k"])[1]) == 1


def test_memory_instructions_keep_their_wait_states(tmp_path):
    import gfr_moe
    lib = tmp_path / "libgfr_moe.so"
    lib.write_bytes(open(gfr_moe.LIB_PATH, "rb").read())
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    code = sorted(p for p in tmp_path.iterdir() if p.name.endswith("gfx950"))
    assert code
    loads, bad = 0, []
    for p in code:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", p], check=True, capture_output=True, text=True).stdout
        for name, ins in functions(text).items():
            n, b = violations(ins)
            loads += n
            bad += [f"{name} {line}" for line in b]
    assert loads > 100, "the prefill GEMMs' direct loads are not in the listing"
    assert not bad, "\n".join(bad)

"""Wait states in the built gfx950 code. The compiler inserts those that the hardware asks software for, except around inline assembly,
which it does not look into: the loads that go straight into LDS and the write-through stores of the kernels are inline assembly."""
import collections
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
# scalar instructions whose first operand is no scalar register that they write
READ_ONLY = ("s_cmp", "s_bitcmp", "s_nop", "s_wait", "s_cbranch", "s_branch", "s_barrier", "s_sleep", "s_setprio", "s_endpgm", "s_sendmsg")


def functions(path):
    """(name, [(address, text, whole line)]) of every function of a code object."""
    out = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", path], stdout=subprocess.PIPE, text=True, check=True).stdout
    name, body = None, []
    for line in out.splitlines():
        head = re.match(r"([0-9a-f]+) <(.+)>:", line)
        if head:
            if body:
                yield name, body
            name, body = head.group(2), []
            continue
        at = line.find("// ")
        if at > 0 and line[0] in " \t":
            body.append((int(line[at + 3:at + 15], 16), line[:at].strip(), line))
    if body:
        yield name, body


def registers(text, kind):
    out = set()
    for one, lo, hi in re.findall(r"(?<![a-z0-9_])%s(?:(\d+)|\[(\d+):(\d+)\])" % kind, text):
        out |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    if kind == "s" and re.search(r"\bm0\b", text):
        out.add("m0")
    return out


def written(text):
    """Scalar registers that an instruction writes."""
    op, _, rest = text.partition(" ")
    ops = rest.split(",")
    if op.startswith("v_"):
        w = registers(ops[0], "s")
        if "_co_" in op or op.startswith(("v_div_scale", "v_mad_u64", "v_mad_i64")):
            w |= registers(ops[1], "s")
        return w
    return registers(ops[0], "s") if op.startswith("s_") and not op.startswith(READ_ONLY) else set()


def predecessors(body):
    index = {a: i for i, (a, _, _) in enumerate(body)}
    preds = collections.defaultdict(list)
    for i, (_, text, line) in enumerate(body):
        op = text.split()[0]
        if op.startswith(("s_cbranch", "s_branch")):
            to = re.search(r"<[^>+]*(?:\+0x([0-9a-f]+))?>", line)
            preds[index[body[0][0] + int(to.group(1) or "0", 16)]].append(i)
        if op not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(body):
            preds[i + 1].append(i)
    return preds


def nearest(body, preds, i, limit, writer):
    """Fewest wait states from an earlier instruction for which writer() is "hit" to instruction i, under limit; a path ends where it is
    "stop"."""
    best, stack, seen = None, [(p, 0) for p in preds[i]], {}
    while stack:
        j, w = stack.pop()
        if w >= limit or seen.get(j, limit) <= w:
            continue
        seen[j] = w
        text = body[j][1]
        r = writer(text)
        if r == "hit":
            best = w if best is None else min(best, w)
        elif r != "stop":
            w += int(text.split()[1], 0) + 1 if text.startswith("s_nop") else 1
            stack += [(p, w) for p in preds[j]]
    return best


def scalar_hazards(body):
    """Vector memory instructions within five wait states of a vector instruction that wrote a scalar register which they read (m0
    among them), and loads into LDS right behind the write of m0."""
    preds, found = None, []
    for i, (_, text, _) in enumerate(body):
        op, _, rest = text.partition(" ")
        if not op.startswith(("buffer_load", "buffer_store", "buffer_atomic", "global_", "flat_", "scratch_")):
            continue
        reads = registers(rest, "s")
        to_lds = rest.endswith(" lds")
        if not reads and not to_lds:
            continue
        preds = preds or predecessors(body)
        for reg in reads | ({"m0"} if to_lds else set()):
            def writer(t, reg=reg):
                return None if reg not in written(t) else "hit" if t.startswith("v_") else "stop"
            if nearest(body, preds, i, 5, writer) is not None:
                found.append((reg, text))
        if to_lds and nearest(body, preds, i, 1, lambda t: "hit" if "m0" in written(t) else None) is not None:
            found.append(("m0", text))
    return found


def store_hazards(body):
    """Stores of accumulators before the matrix instruction that writes them is done: up to 19 wait states (16 passes and 3)."""
    preds, found = None, []
    for i, (_, text, _) in enumerate(body):
        op, _, rest = text.partition(" ")
        if "store" not in op or not op.startswith(("buffer_", "global_", "flat_")):
            continue
        ops = rest.split(",")
        data = registers(ops[0] if op.startswith("buffer_") else ops[1], "v")
        preds = preds or predecessors(body)
        passes = nearest(body, preds, i, 19, lambda t: "hit" if t.startswith("v_mfma") and registers(t.split(",")[0].partition(" ")[2], "v") & data else None)
        if passes is not None:
            found.append((passes, text))
    return found


@pytest.mark.parametrize("name", ["k_exl3", "k_exl3_gemm", *(f"k_exl3_rgemm_b{b}" for b in (2, 3, 4, 5, 6, 8)), "k_fp4", "k_bf16", "k_route"])
def test_wait_states(name):
    path = os.path.join(ROOT, "ferrite_amd", "_build", name + ".hsaco")
    assert os.path.exists(path), "build the library first"
    count = 0
    for fn, body in functions(path):
        count += 1
        assert not scalar_hazards(body), (fn, scalar_hazards(body)[:3])
        assert not store_hazards(body), (fn, store_hazards(body)[:3])
    assert count > 0


def test_the_scan_finds_what_it_is_for():
    def body(*text):
        return [(4 * i, t, t) for i, t in enumerate(text)]
    load = "buffer_load_dwordx4 v1, s[0:3], s9 offen lds"
    assert scalar_hazards(body("v_readfirstlane_b32 s9, v0", "s_mov_b32 m0, s5", "s_nop 0", load))
    assert scalar_hazards(body("v_readfirstlane_b32 s2, v0", "s_mov_b32 m0, s5", "s_nop 0", load))
    assert scalar_hazards(body("v_readfirstlane_b32 m0, v0", "s_nop 3", load))
    assert scalar_hazards(body("s_mov_b32 m0, s5", load))
    assert not scalar_hazards(body("v_readfirstlane_b32 s8, v0", "s_mov_b32 m0, s5", "s_mov_b32 s9, s8", load))
    assert not scalar_hazards(body("v_readfirstlane_b32 s9, v0", "s_mov_b32 m0, s5", "s_nop 3", load))
    store = "global_store_dwordx4 v[8:9], v[4:7], off sc1"
    assert store_hazards(body("v_mfma_f32_16x16x32_f16 v[4:7], v[0:3], v[10:13], v[4:7]", "s_nop 6", store))
    assert not store_hazards(body("v_mfma_f32_16x16x32_f16 v[0:3], v[10:13], v[14:17], v[0:3]", store))

"""Products that the kernels issue by asm: the compiler does not know them, so it inserts no wait between a product and what reads its
result, nor between what writes an operand and the product.  The kernels place those waits; this reads the assembly for any that is missing."""
import concurrent.futures as cf
import re
import subprocess

import pytest

from ome_amd import build

PRODUCT = "v_mfma_f32_32x32x16_bf16"   # (by asm only; of the others, which are builtins, the compiler keeps count)
MADE, WRITTEN = 11, 2   # slots between a product of 8 passes and another reader; between the vector ALU's write and a product
REG = re.compile(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def _regs(operand):
    m = REG.search(operand)
    if not m:
        return []
    a, b = (int(m[2]), int(m[3])) if m[2] else (int(m[4]), int(m[4]))
    return [(m[1], r) for r in range(a, b + 1)]


def too_early(assembly):
    """(function, instruction, slots) of what comes too early, along the text: an instruction takes a slot, a loop's way back is not followed."""
    found, at, made, written, function = [], 0, {}, {}, ""
    for line in assembly.splitlines():
        if re.match(r"^_Z\w+:", line):
            function, at, made, written = line.split(":")[0], 0, {}, {}
        m = re.match(r"^\s+([vs]_\w+|ds_\w+|global_\w+|buffer_\w+|scratch_\w+)\s*(.*)", line.split(";")[0])
        if not m:
            continue
        name, ops = m[1], re.split(r",\s*(?![^\[]*\])", m[2])
        if name == "s_nop":
            at += int(ops[0], 0) + 1
            continue
        at += 1
        if name == PRODUCT:
            for i, o in enumerate(ops[1:4]):
                for r in _regs(o):
                    since = [at - written.get(r, -99) if at - written.get(r, -99) <= WRITTEN else 99,
                             at - made.get(r, -99) if i < 2 and at - made.get(r, -99) <= MADE else 99]   # (a sum may go on at once)
                    if min(since) < 99:
                        found.append((function, line.strip(), min(since)))
            for r in _regs(ops[0]):
                made[r] = at
                written.pop(r, None)
        elif name[0] != "s":
            for o in ops:
                for r in _regs(o):
                    if at - made.get(r, -99) <= MADE:
                        found.append((function, line.strip(), at - made.pop(r)))
            if name.startswith("v_") and not name.startswith("v_cmp"):
                for o in ops[:2 if "swap" in name else 1]:
                    for r in _regs(o):
                        written[r] = at
    return found


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm")

    def compile_one(name):
        flags = [f for f in build.HIP_FLAGS if f != "-fPIC"]
        subprocess.run([build._hipcc(), *flags, f"-I{build.CSRC}", "-S", "--offload-device-only", str(build.CSRC / "kernels" / f"{name}.hip"), "-o",
                        str(out / name)], check=True, capture_output=True)
        return (out / name).read_text()

    with cf.ThreadPoolExecutor(2) as ex:
        names = ("mla", "prefill_pair")
        return dict(zip(names, ex.map(compile_one, names)))


@pytest.mark.parametrize("name", ["mla", "prefill_pair"])
def test_waits(assembly, name):
    assert assembly[name].count(PRODUCT) > 100
    assert too_early(assembly[name]) == []


@pytest.mark.parametrize("between,early", [("s_nop 9", 1), ("s_nop 10", 0), ("s_nop 7\n\tv_mov_b32 v9, v8", 1), ("v_mov_b32 v9, v8\n" * 11, 0)])
@pytest.mark.parametrize("reader", ["v_accvgpr_read_b32 v8, a15", "v_accvgpr_mov_b32 a40, a3", "ds_write_b128 v1, a[12:15]",
                                    PRODUCT + " a[16:31], v[0:3], a[0:3], a[16:31]"])
def test_an_early_reader_is_found(between, early, reader):
    text = f"_Z1fv:\n\t{PRODUCT} a[0:15], v[0:3], v[4:7], a[0:15]\n\t{PRODUCT} a[0:15], v[0:3], v[4:7], a[0:15]\n\t{between}\n\t{reader}\n"
    found = too_early(text.replace("\nv_mov", "\n\tv_mov"))
    assert bool(found) == bool(early) and all(f[1] == reader for f in found)


def test_an_operand_written_just_now_is_found():
    text = "_Z1fv:\n\tv_mov_b32 v5, v9\n\t%s" + PRODUCT + " a[0:15], v[0:3], v[4:7], 0\n"
    assert len(too_early(text % "")) == 1 and too_early(text % "s_nop 1\n\t") == []

"""What the compiler made of this repository's kernels, where their source cannot say it
all: waits around matrix products that stand as text, which it does not see, and loads
that would wait for others to be done."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

OPS = Path(__file__).parent.parent / "runbooks_amd" / "ops"
DUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
# wait states that a product's result takes until others may read or write it, of the
# longest products there are
DONE = 20


def _kernels(tmp_path, kernel):
    built = list(OPS.glob("_hip.cpython*.so"))
    if not built or not Path(DUMP).exists():
        pytest.skip("nothing built, or no llvm-objdump")
    so = tmp_path / "hip.so"
    shutil.copy(built[0], so)
    subprocess.run([DUMP, "--offloading", so.name], cwd=tmp_path, check=True,
                   capture_output=True)
    for part in sorted(tmp_path.glob("hip.so.*gfx950*")):
        names = subprocess.run([DUMP, "-t", part], capture_output=True,
                               text=True).stdout
        for name in sorted(set(re.findall(
                rf"\S*{kernel}\S*(?=\n)", names))):
            if "." in name:
                continue
            text = subprocess.run(
                [DUMP, "-d", f"--disassemble-symbols={name}", part],
                capture_output=True, text=True, check=True).stdout
            code = [line.split("//")[0].split()
                    for line in text.splitlines() if line.startswith("\t")]
            yield [(c[0], " ".join(c[1:])) for c in code if c]


def _sums(args):
    """The registers a[..] of an instruction."""
    found = set()
    for a, b in re.findall(r"\ba(?:\[(\d+:\d+)\]|(\d+)\b)", args):
        lo, hi = (map(int, a.split(":")) if a else (int(b), int(b)))
        found.update(range(lo, hi + 1))
    return found


def test_products_as_text_wait(tmp_path):
    seen = 0
    for code in _kernels(tmp_path, "flash_prefill_kernelILi256E"):
        # four products behind a wait of four states
        inside, sums = set(), set()
        for i, (op, args) in enumerate(code):
            if (op, args) == ("s_nop", "3") and all(
                    "mfma" in o and a.startswith("a[")
                    for o, a in code[i + 1:i + 5]):
                inside.update(range(i + 1, i + 5))
                for _, a in code[i + 1:i + 5]:
                    sums |= _sums(a.split(",")[0])
        assert len(sums) == 8 * 16          # of 32 rows and 256 columns
        since = DONE
        for i, (op, args) in enumerate(code):
            touches = bool(_sums(args) & sums)
            if "mfma" in op and touches:
                assert i in inside, f"{op} {args} by itself"
                since = 0
                continue
            assert not touches or since >= DONE, f"{op} {args} after {since}"
            since += int(args) + 1 if op == "s_nop" else 1
        seen += 1
    assert seen == 2                        # by whole and by half keys


def test_blocks_of_8_bits_stay_on_their_way(tmp_path):
    """A load from a pointer that may be one to LDS or to memory waits for all loads
    ahead of it, and so for every block that the ring has asked for."""
    seen = 0
    for code in _kernels(tmp_path, "paged_decode8_kernel"):
        assert not any(op.startswith("flat_load") for op, _ in code)
        seen += 1
    assert seen > 0


def test_loads_of_both_kinds(tmp_path):
    """Past L2 and not: two loads that differ in that alone are one to the compiler
    where it may have them so, and neither."""
    seen = 0
    for code in _kernels(tmp_path, "paged_decode_(?:mfma_)?kernel"):
        wide = [args.split()[-1] == "nt" for op, args in code
                if op == "global_load_dwordx4"]
        if any(wide):
            assert 3 * wide.count(False) > wide.count(True) > wide.count(False) / 3
            seen += 1
    assert seen > 0

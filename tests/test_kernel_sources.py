"""Rules of the kernel sources that a compiler does not check (host only)."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "apt-serve_amd" / "csrc"
SOURCES = sorted(p for p in CSRC.rglob("*") if p.suffix in (".hip", ".h"))


def asm_statements(text):
    """(instructions, rest of the statement) of every inline assembly statement."""
    text = re.sub(r"//[^\n]*", "", text)
    for m in re.finditer(r'\basm\s+volatile\s*\(((?:[^()"]|"(?:\\.|[^"\\])*"|\((?:[^()"]|"(?:\\.|[^"\\])*"|\([^()]*\))*\))*)\)\s*;', text):
        body = m.group(1)
        code = re.match(r'\s*((?:"(?:\\.|[^"\\])*"\s*)+)', body)
        if code:
            yield "".join(re.findall(r'"((?:\\.|[^"\\])*)"', code.group(1))), body[code.end():]


def test_assembly_that_writes_m0_says_so_and_waits():
    """A copy global -> LDS takes its LDS address from m0 and its descriptor from scalar registers.  The compiler keeps
    m0 for its own use unless the statement names it, and it cannot put wait states inside a statement: one is needed
    between a write of m0 and the copy, five between a scalar register written by a vector instruction and the copy."""
    found = 0
    for p in SOURCES:
        for code, rest in asm_statements(p.read_text()):
            ins = [i.strip() for i in re.split(r"\\n|;", code) if i.replace("\\t", "").strip()]
            ins = [i.replace("\\t", " ").strip() for i in ins]
            writes = [i for i, x in enumerate(ins) if re.match(r"s_mov_b32 m0\b", x)]
            if not writes:
                continue
            found += 1
            assert '"m0"' in rest.rsplit(":", 1)[-1], f"{p.name}: m0 is not in the clobber list of {code!r}"
            load = next(i for i, x in enumerate(ins) if x.startswith("buffer_load") or x.startswith("global_load"))
            states = sum(int(x.split()[1]) + 1 if x.startswith("s_nop") else 1 for x in ins[:load])
            assert states >= 5, f"{p.name}: {states} wait states before the copy in {code!r}"
    assert found >= 1


def test_prompt_attention_copies_a_tile_ahead():
    """Its copies into LDS are in flight while the tile before is multiplied.  Issued through the compiler's builtin they
    are waited for before the next LDS read of any stage, so every path issues them from assembly."""
    code = re.sub(r"//[^\n]*", "", (CSRC / "prefill_attention.hip").read_text())
    assert not re.search(r"__builtin_amdgcn_\w*load\w*_lds", code)


def test_one_wavefront_of_a_workgroup_looks_the_sequence_up():
    """The search by rank is some hundred instructions that do not depend on the wavefront: in every wavefront of
    workgroups whose sequences are short it took longer than the attention."""
    text = re.sub(r"//[^\n]*", "", (CSRC / "paged_decode_core.h").read_text())
    calls = [m.start() for m in re.finditer(r"=\s*sequence_of_rank\(", text)]
    assert len(calls) == 1 and re.search(r"if \(wave == 0\) \{\s*seq $", text[:calls[0]])

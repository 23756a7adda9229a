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


def instructions(code):
    return [i.strip() for i in re.split(r"\\n|;", code.replace("\\t", " ")) if i.strip()]


def test_assembly_that_writes_m0_says_so_and_waits():
    """A copy global -> LDS takes its LDS address from m0.  The compiler keeps m0 for its own use unless the statement
    names it, and it cannot put the wait state between a write of m0 and the copy into a statement."""
    found = 0
    for p in SOURCES:
        for code, rest in asm_statements(p.read_text()):
            ins = instructions(code)
            for i, x in enumerate(ins):
                if re.match(r"s_mov_b32 m0\b", x):
                    found += 1
                    assert '"m0"' in rest.rsplit(":", 1)[-1], f"{p.name}: m0 is not in the clobber list of {code!r}"
                    load = next(j for j, y in enumerate(ins) if j > i and re.match(r"(buffer|global)_load", y))
                    assert load > i + 1, f"{p.name}: no wait state after the write of m0 in {code!r}"
    assert found >= 1


def test_copies_from_assembly_take_descriptors_that_scalar_instructions_wrote():
    """Five wait states lie between a vector instruction that writes a scalar register and a memory instruction that reads
    it; the compiler puts none in front of a statement.  Descriptors of copies come from scalar_rsrc alone, which ends
    in scalar instructions."""
    text = {p.name: re.sub(r"//[^\n]*", "", p.read_text()) for p in SOURCES}
    for name, t in text.items():
        for code, rest in asm_statements(t):
            if any(x.startswith("buffer_") for x in instructions(code)):
                assert '"s"(rsrc.words)' in rest, f"{name}: {code!r}"
    made = [(name, m.start()) for name, t in text.items() for m in re.finditer(r"\bScalarRsrc\s*\{\s*u32x4\s*\{", t)]
    assert [name for name, _ in made] == ["mfma_common.h"]
    body = text["mfma_common.h"]
    body = body[body.index("ScalarRsrc scalar_rsrc("):made[0][1]]
    code = "".join(re.findall(r'asm\("((?:\\.|[^"\\])*)"', body))
    assert code and all(x.startswith("s_") for x in instructions(code))


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

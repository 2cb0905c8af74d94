"""Inline assembly of the kernels names what it overwrites: a statement with a scalar instruction that writes SCC lists "scc", or the compiler may keep a comparison's result or a carry there across it."""
import glob
import os
import re

import __graft_entry__ as graft

CSRC = os.path.join(graft.PKG_DIR, "csrc")
_WRITES_SCC = re.compile(r"\bs_(?:(?:add|sub|addc|subb|min|max|and|or|xor|andn1|andn2|orn1|orn2|nand|nor|xnor|not|lshl[1-4]?|lshr|ashr|bfe|wqm|quadmask|bcnt[01]|absdiff|abs|bitcmp[01]|cmp)_\w+|\w+_saveexec\w*)")


def _statements(text):
    """Template and clobbers of every asm statement."""
    for m in re.finditer(r"\basm\s+(?:volatile\s*)?\(", text):
        depth, i, parts, quoted = 1, m.end(), [""], False
        while depth:
            c = text[i]
            if quoted and c == "\\":
                parts[-1] += text[i:i + 2]
                i += 2
                continue
            if c == '"':
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
                if c == ":" and depth == 1:
                    parts.append("")
            parts[-1] += c
            i += 1
        yield parts[0].replace("\\n", " ").replace("\\t", " "), parts[3] if len(parts) > 3 else "", text.count("\n", 0, m.start()) + 1


def test_statements_that_write_scc_say_so():
    seen, bad = 0, []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        with open(path) as f:
            text = f.read()
        for template, clobbers, line in _statements(text):
            seen += 1
            if _WRITES_SCC.search(template) and '"scc"' not in clobbers:
                bad.append(f"{os.path.basename(path)}:{line}: {template.strip()[:80]}")
    assert seen > 50 and not bad, bad


def test_the_scan_tells_them_apart():
    (t, c, _), = _statements('asm volatile("s_mov_b32 m0, %1\\n\\ts_add_u32 m0, m0, 4" : : "v"(x), "s"(f(y)) : "memory", "m0");')
    assert _WRITES_SCC.search(t) and '"scc"' not in c and '"m0"' in c
    assert not _WRITES_SCC.search("s_mov_b32 m0, %0 s_nop 0 s_load_dword %0, %1, 0x0 s_waitcnt lgkmcnt(0) s_barrier s_mul_i32 s_sleep 1")

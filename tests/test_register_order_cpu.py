"""The register phase 1 has no barrier while one thread rewrites the basis
bookkeeping next to the tableau update, so nothing else may touch those words
there: a wave that comes late would read them half written and go on with
another variable's use count.  A run cannot be relied on to show that; the
kernel's text is checked instead."""
import os
import re

from conftest import ROOT

SOURCE = os.path.join(ROOT, "mpqpcudasolver_amd", "csrc", "reg_kernel.hpp")
WORDS = re.compile(r"\bL\.(basis|nonb|where|bcnt|nbcnt)\b")


def _text():
    src = re.sub(r"//[^\n]*", "", open(SOURCE).read())
    return re.sub(r"/\*.*?\*/", "", src, flags=re.S)


def _block(src, at):
    """The braces that open at or after `at`, with what they hold."""
    i = src.index("{", at)
    depth = 0
    for j in range(i, len(src)):
        depth += {"{": 1, "}": -1}.get(src[j], 0)
        if depth == 0:
            return i, j + 1
    raise AssertionError("unbalanced braces")


def _function(src, name):
    at = re.search(r"\b%s\(" % name, src).start()
    i, j = _block(src, at)
    return src[i:j]


def test_one_thread_has_the_bookkeeping_during_the_update():
    body = _function(_text(), "reg_phase1")
    # from the barrier behind which every wave knows the pivot to the one that closes it
    open_at = body.index("q = rfl(sh.q);")
    update = body.index("reg_update(R, L, r, q);", open_at)
    close_at = body.index("__syncthreads();", update)
    part = body[open_at:close_at]
    assert "__syncthreads" not in part
    one_thread = r"threadIdx\.x\s*==\s*\(NW - 1\)\s*\*\s*MPQP_WAVE"
    guard = re.search(r"const bool (\w+) = %s;" % one_thread, part)
    cond = r"if \((?:%s%s)\) \{" % (one_thread, "|" + guard.group(1) if guard else "")
    while True:
        m = re.search(cond, part)
        if not m:
            break
        part = part[:m.start()] + part[_block(part, m.start())[1]:]
    assert WORDS.findall(part) == []


def test_the_update_does_not_read_the_bookkeeping():
    src = _text()
    for name in ("reg_update", "reg_apply", "reg_col_op", "reg_set_row", "reg_lds_col", "reg_min_out"):
        assert WORDS.findall(_function(src, name)) == [], name

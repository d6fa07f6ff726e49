"""The hand-out's constants stand in one vector register, a word per lane (grouped_gemm.hip, Words).  What reads a word has to run with all
lanes of the wavefront on: the compiler takes the register for a value of each lane, so a copy or a reload that it places where some are off
holds the words of the others no longer, and v_readlane then gives whatever the register held before.  No GPU."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "expert_specialization_moe_amd", "csrc", "grouped_gemm.hip")


def _close(text, start, pair):
    """Index behind the bracket that closes the one at `start`."""
    depth = 0
    for i in range(start, len(text)):
        depth += (text[i] == pair[0]) - (text[i] == pair[1])
        if depth == 0:
            return i + 1
    raise AssertionError("unbalanced")


def _divergent_reads(text):
    """Reads of a Words object in a condition on the thread's index, or in what it guards."""
    text = re.sub(r"//[^\n]*", "", text)
    names = set(re.findall(r"\bWords (\w+)\(", text))
    assert names, "no Words object"
    read = re.compile(r"\b(?:%s)\[" % "|".join(sorted(names)))
    found = []
    for m in re.finditer(r"\bif (?:constexpr )?\(", text):
        end = _close(text, m.end() - 1, "()")
        cond = text[m.end():end]
        if not re.search(r"\bthreadIdx\b|\blane\b|\btid\b", cond):
            continue
        rest = text[end:]
        body = rest[:_close(rest, rest.index("{"), "{}")] if re.match(r"\s*\{", rest) else rest[:rest.index(";")]
        if read.search(cond) or read.search(body):
            found.append(text[m.start():end])
    return found


def test_words_are_read_where_every_lane_is_on():
    with open(SRC) as f:
        assert _divergent_reads(f.read()) == []


def test_a_read_behind_a_condition_on_the_thread_is_found():
    for bad in ("const Words hand(&s); if (threadIdx.x == 0 && hand[4] != 1) { f(); }", "const Words w(&s); if (lane == 0) { f(w[8]); }",
                "const Words w(&s); if (tid < 9) g = w[0];"):
        assert _divergent_reads(bad)
    assert not _divergent_reads("const Words w(&s); const int u = w[4]; if (u != 1 && threadIdx.x == 0) { f(); }")

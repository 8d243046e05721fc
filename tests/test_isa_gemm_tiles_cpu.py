"""CPU tier (no GPU): the products of gemm_tiles.h read fragments into registers with asm statements whose wait stands half a k-step later, which hipcc does not
track - on no path may an instruction touch a register whose read is still in flight, and no kernel may keep values in scratch memory."""
import re

import pytest

from test_isa_cpu import _compiled, _registers, pytestmark  # noqa: F401


@pytest.mark.parametrize("src, pattern", [("lm_prefill.hip", "k_gemm_pf_wide"), ("whisper_kernels.hip", "k_gemm_rows")])
def test_no_fragment_in_flight_is_touched(src, pattern):
    text, use = _compiled(src)
    names = re.findall(r"\n(_Z\w*%s\w*):" % pattern, text)
    assert len(names) >= 9
    for name in names:
        assert use[name]["scratch"] == 0, (name, use[name])
        i = text.index("\n" + name + ":")
        lines = [l.split(";")[0].strip() for l in text[i: text.index(".Lfunc_end", i)].split("\n")]
        label = {l[:-1]: k for k, l in enumerate(lines) if re.fullmatch(r"\.LBB\w+:", l)}
        todo, seen, most = [(0, ())], set(), 0
        while todo:
            k, flight = todo.pop()
            while k < len(lines) and (k, flight) not in seen:
                seen.add((k, flight))
                l, k = lines[k], k + 1
                if not re.match(r"[a-z]", l):
                    continue
                op, _, rest = l.partition(" ")
                if op == "s_endpgm":
                    break
                if op == "s_waitcnt":
                    m = re.search(r"lgkmcnt\((\d+)\)", l)
                    flight = flight[max(0, len(flight) - int(m[1])):] if m else flight
                    continue
                if op == "s_branch" or op.startswith("s_cbranch"):
                    todo.append((label[rest.strip()], flight))
                    if op == "s_branch":
                        break
                    continue
                operands = [_registers(t.strip().split(" ")[0]) for t in rest.split(",")]
                assert not any(r & f for r in operands for f in flight), (name, l)
                if op.startswith("ds_read"):
                    flight += (operands[0],)
                    most = max(most, len(flight))
        assert most >= 12, (name, most)                              # a half's fragments in flight under the other half's products

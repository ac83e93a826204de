"""Check of the compiled persistent GEMM: the wait states around its MFMAs.

    python minimax-h3-2xt4_amd/mfma_hazards.py FILE.s FUNCTION-NAME-PART

The kernel issues v_mfma_i32_16x16x64_i8 from inline assembly, where the
compiler neither sees an MFMA nor inserts the wait states it needs. The source
keeps them (operands come straight from LDS reads, whose waits the compiler
does count; explicit s_nop after the accumulators are cleared and before they
are read), and the build checks the assembly it produced here, along every
path of the control flow:

* no VALU instruction writes a register that an MFMA reads within two wait
  states (what the compiler keeps itself for the builtin), none writes EXEC
  within four;
* nothing but an MFMA touches an accumulator within 18 wait states of the MFMA
  that writes it;
* no function uses scratch memory (a reload could stand before an MFMA).
"""
import re
import sys

VALU_WAIT, EXEC_WAIT, RESULT_WAIT = 2, 4, 18

_REG = re.compile(r'\b([va])(?:(\d+)|\[(\d+):(\d+)\])')
_LABEL = re.compile(r'^([.\w$]+):')
_SCRATCH = re.compile(r'^; ScratchSize: (\d+)')


def _regs(operand):
    """Vector registers an operand names: {('v', 12), ('a', 3), ...}."""
    out = set()
    for kind, one, lo, hi in _REG.findall(operand):
        out.update((kind, r) for r in (range(int(one), int(one) + 1) if one else range(int(lo), int(hi) + 1)))
    return out


class _Inst:
    __slots__ = ('text', 'op', 'operands', 'states', 'mfma', 'valu')

    def __init__(self, text):
        self.text = text
        op, _, rest = text.partition(' ')
        self.op = op
        self.operands = [p.strip() for p in rest.split(',')]
        self.states = int(self.operands[0], 0) + 1 if op == 's_nop' else 1
        self.mfma = op.startswith(('v_mfma', 'v_smfmac'))
        self.valu = op.startswith('v_') and not self.mfma

    def touches(self):
        return set().union(*map(_regs, self.operands)) if self.operands else set()

    def writes(self):
        if self.op.startswith(('v_cmp', 'v_readfirstlane', 'v_readlane')):
            return set()
        both = self.op.startswith(('v_swap', 'v_permlane16_swap', 'v_permlane32_swap'))
        return set().union(*map(_regs, self.operands[:2 if both else 1]))


def functions(text, kernel=''):
    """(name, instructions, label -> index, scratch bytes) of the functions
    whose name contains kernel."""
    name, insts, labels = None, [], {}
    for raw in text.splitlines():
        m = _SCRATCH.match(raw)
        if m and name:
            yield name, insts, labels, int(m.group(1))
            name = None
            continue
        line = raw.split(';')[0].strip()
        m = _LABEL.match(line)
        if m:
            if not m.group(1).startswith('.'):
                name, insts, labels = m.group(1) if kernel in m.group(1) else None, [], {}
            labels[m.group(1)] = len(insts)
        elif line and not line.startswith('.') and name:
            insts.append(_Inst(re.sub(r'\s+', ' ', line)))


def _reach(insts, labels, i, states):
    """Instructions reached from instruction i with fewer than `states` wait
    states between, over both ways of every branch."""
    seen, todo = {}, [(i, 0)]
    while todo:
        at, dist = todo.pop()
        op = insts[at].op
        nexts = []
        if op in ('s_branch',) or op.startswith('s_cbranch'):
            target = labels.get(insts[at].operands[0])
            if target is not None:
                nexts.append(target)
        if op not in ('s_branch', 's_endpgm', 's_setpc_b64'):
            nexts.append(at + 1)
        for n in nexts:
            if n < len(insts) and seen.get(n, states) > dist:
                seen[n] = dist
                yield insts[n]
                if dist + insts[n].states < states:
                    todo.append((n, dist + insts[n].states))


def hazards(text, kernel):
    """Descriptions of the hazards in the functions whose name contains kernel."""
    found = []
    checked = 0
    for name, insts, labels, scratch in functions(text, kernel):
        checked += 1
        if scratch:
            found.append(f'{name}: {scratch} bytes of scratch a lane')
        # Only instructions with an MFMA or a branch close behind can matter.
        near, close = 0, [False] * len(insts)
        for i in range(len(insts) - 1, -1, -1):
            close[i] = near > 0
            near = EXEC_WAIT if insts[i].mfma or insts[i].op.startswith(('s_branch', 's_cbranch')) else near - 1
        for i, inst in enumerate(insts):
            if inst.valu and close[i]:
                if inst.op.startswith('v_cmpx'):
                    found += [f'{name}: EXEC written by "{inst.text}" before "{n.text}"'
                              for n in _reach(insts, labels, i, EXEC_WAIT) if n.mfma]
                w = inst.writes()
                if w:
                    found += [f'{name}: "{inst.text}" before "{n.text}"'
                              for n in _reach(insts, labels, i, VALU_WAIT)
                              if n.mfma and w & set().union(*map(_regs, n.operands[1:]))]
            elif inst.mfma:
                acc = _regs(inst.operands[0])
                found += [f'{name}: "{inst.text}" before "{n.text}"'
                          for n in _reach(insts, labels, i, RESULT_WAIT) if not n.mfma and acc & n.touches()]
    if not checked:
        found.append(f'no function named *{kernel}* in the assembly')
    return found


if __name__ == '__main__':
    with open(sys.argv[1]) as f:
        problems = hazards(f.read(), sys.argv[2])
    print('\n'.join(problems[:20]))
    sys.exit(1 if problems else 0)

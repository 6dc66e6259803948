#!/usr/bin/env python3
"""Build check for kernels whose matrix instructions or loads to LDS are inline
assembly.

The compiler does not know that such a statement is a matrix instruction and
counts no wait states behind it: a vector, LDS or memory instruction that
touches the instruction's result registers too soon reads (or is overwritten
by) a result that the matrix core has not written yet.  The kernels put their
own `s_nop` behind the last matrix instruction of a tile; this script reads the
compiler's assembly (`hipcc -S --cuda-device-only`) and fails if any other
instruction touches a matrix instruction's destination registers within
WINDOW instructions of it without such a wait in between -- which is what a
register copy that the compiler decided to insert there would look like.

Nor does it count wait states in front of such a statement.  Reported too are a
load to LDS right behind the write of M0, which says where to (one wait state:
the compiler puts an instruction there for its own), a memory instruction that
reads a scalar register within five wait states of the vector instruction that
wrote it (a descriptor made with v_readfirstlane), and a matrix instruction that
reads a register within two wait states of the vector instruction that wrote it
(an accumulator's zeros, a packed operand).

usage: check_mfma_wait.py file.s
"""
import re
import sys

WINDOW = 20  # instructions; 16 passes need at most 18 wait states
REG = re.compile(r'\b([va])(?:(\d+)\b|\[([^\]]+)\])')
SCALAR_REG = re.compile(r'\b(s)(?:(\d+)\b|\[([^\]]+)\])')
SCALAR_WINDOW = 5  # wait states from a vector write to a memory read
OPERAND_WINDOW = 2  # wait states from a vector write to a matrix instruction's read
MEMORY = ('buffer_', 'global_', 'flat_', 'scratch_')


def _value(expr):
  if not re.fullmatch(r'[0-9a-fx+* ]+', expr):
    raise ValueError(expr)
  return int(eval(expr))  # digits, +, * only (checked above)


def registers(text, kinds=REG):
  """{('v', 3), ...} named in an operand string."""
  out = set()
  for kind, single, inner in kinds.findall(text):
    if single:
      out.add((kind, int(single)))
    elif ':' in inner:
      lo, hi = inner.split(':')
      out.update((kind, r) for r in range(_value(lo), _value(hi) + 1))
    else:
      out.add((kind, _value(inner)))
  return out


def too_soon(path):
  """How many loads and matrix instructions come too soon behind what they read
  (see above)."""
  written = []  # [registers, wait states left]
  m0 = False    # the last instruction wrote it
  bad = 0
  for number, line in enumerate(open(path), 1):
    text = line.split(';')[0].strip()
    if not text or text.startswith('.') or text.endswith(':'):
      continue
    op, _, operands = text.partition(' ')
    waits = 1
    if op.startswith('s_nop'):
      waits += _value(operands.strip())
    elif op.startswith(MEMORY):
      if m0 and re.search(r'\blds\b', operands):
        print(f'{path}:{number}: `{text}` right behind the write of M0')
        bad += 1
      used = registers(operands, SCALAR_REG)
      if any(d & used for d, _ in written):
        print(f'{path}:{number}: `{text}` reads a scalar register written by a '
              f'vector instruction fewer than {SCALAR_WINDOW} wait states before')
        bad += 1
    # (operands are apart at commas outside a[..])
    parts = [p.strip() for p in re.split(r',(?![^\[]*\])', operands)]
    first = parts[0]
    if op.startswith('v_mfma'):
      used = registers(', '.join(parts[1:4]))
      if any(d & used for d, _ in written):
        print(f'{path}:{number}: `{text}` reads a register written by a vector '
              f'instruction fewer than {OPERAND_WINDOW} wait states before')
        bad += 1
    m0 = first == 'm0'
    written = [[d, n - waits] for d, n in written if n > waits]
    if op.startswith('v_') and first.startswith('s'):
      written.append([registers(first, SCALAR_REG), SCALAR_WINDOW])
    elif op.startswith('v_') and not op.startswith('v_mfma'):
      both = ', '.join(parts[:2]) if 'swap' in op else first
      written.append([registers(both), OPERAND_WINDOW])
  return bad


def main(path):
  pending = []  # [destination registers, instructions left]
  bad = too_soon(path)
  for number, line in enumerate(open(path), 1):
    text = line.split(';')[0].strip()
    if not text or text.startswith('.') or text.endswith(':'):
      continue
    op, _, operands = text.partition(' ')
    if op.startswith('s_nop'):
      if _value(operands.strip()) >= 7:
        pending = []
      else:
        pending = [[d, n - 1] for d, n in pending if n > 1]
      continue
    if op.startswith('v_mfma'):
      # a matrix instruction may follow one on the same accumulator at once
      dst = registers(operands.split(',')[0])
      pending = [[d, n - 1] for d, n in pending if n > 1 and not (d & dst)]
      pending.append([dst, WINDOW])
      continue
    touched = registers(operands)
    for d, _ in pending:
      if d & touched:
        print(f'{path}:{number}: `{text}` touches the result of a matrix '
              f'instruction issued fewer than {WINDOW} instructions before it')
        bad += 1
        break
    pending = [[d, n - 1] for d, n in pending if n > 1]
  return 1 if bad else 0


if __name__ == '__main__':
  sys.exit(main(sys.argv[1]))

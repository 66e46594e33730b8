// Whether a Krylov step is enqueued before the result of the one before it has
// been read, in plain C++.
#pragma once

namespace sg {

// precond: the preconditioner's number (see SolverState); res: the residual
// before the step on the stream; rate: what the last finished step multiplied
// it by (0 before the first); target: the residual at which the solve ends.
//
// A step enqueued in vain costs its whole length, one that is not costs the
// device some 20 us.  So the host looks first where two more reductions like the
// last would end the solve, and before the first result of a solve, when
// nothing is known.  Preconditioners 3 and 5 walk the grid line after line: a
// step takes 0.8 ms at 33x25, 3.3 to 3.5 at 97x65, 86 and 117 ms at 545x385,
// beside which 20 us are nothing.  The others take 31 (none) to 122 us at 33x25
// and 0.15 to 0.9 ms (1 and 2: 6.7) at 545x385.
inline bool enqueue_ahead(int precond, double res, double rate, double target) {
  if (precond == 3 || precond == 5) return false;
  return res * rate * rate > target;
}

}  // namespace sg

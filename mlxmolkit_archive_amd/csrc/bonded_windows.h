// Windows of a molecule's bonded terms whose energies a kernel holds in LDS at once. Plain
// constexpr functions: the kernels use them, and a host compiler can check them.
#pragma once

namespace mmff {

// A window that does not reach the last term ends a whole number of 64-term tasks into a type (or
// at the type's end), so it moves on only if the LDS holds the energies of one task.
constexpr int BONDED_WINDOW_MIN = 64;

// LDS floats of the bonded energies in the L-BFGS kernels without helper threads: 12 per atom
// (max_n = 3 max_atoms rounded up to a multiple of 4), and at least one task's
constexpr int lbfgs_eb_floats(int max_n) { return 4 * max_n > BONDED_WINDOW_MIN ? 4 * max_n : BONDED_WINDOW_MIN; }

// End of the window that starts at term s and holds at most eb_n >= BONDED_WINDOW_MIN terms. Type
// k has the numbers base[k] .. base[k + 1] - 1; s is such an end, or 0.
constexpr int bonded_window_end(const int (&base)[6], int s, int eb_n) {
  if (base[5] - s <= eb_n) return base[5];
  const int lim = s + eb_n;
  int end = s;
#pragma unroll
  for (int k = 0; k < 5; k++)
    if (lim > base[k] && s < base[k + 1])
      end = lim >= base[k + 1] ? base[k + 1] : base[k] + ((lim - base[k]) & ~63);
  return end;
}

}  // namespace mmff

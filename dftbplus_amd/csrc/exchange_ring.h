// Rules of the exchange ring of the tridiagonalisation over workgroups (sytrd_resident.hip): which
// words a workgroup publishes, gathers and empties in a column, and when it leaves. Plain
// arithmetic, so that the host model of the protocol runs the rules the kernel runs.
#pragma once

#if defined(__HIPCC__)
#define DH_RING_FN __host__ __device__ inline
#else
#define DH_RING_FN inline
#endif

namespace dftbhip {

constexpr int kRingSlots = 3;   // column k uses slot k mod kRingSlots

// Last row of workgroup p of P over m rows (rows p, p + P, ...)
DH_RING_FN int ring_last_row(int p, int P, int m) { return p + P * ((m - 1 - p) / P); }

// Row `row` has a word in column k: its owner publishes it, every workgroup that gathers the
// column reads it.
DH_RING_FN bool ring_published(int row, int k) { return row > k; }

// Once its workgroup has gathered column k, the owner empties the row's words of column k - 1.
DH_RING_FN bool ring_emptied(int row, int k) { return k > 0 && row >= k; }

// Columns that a workgroup gathers, of the kEnd that are reduced: all of them if one of its rows
// is left over, else those before the column that publishes its last row. It publishes that row
// and leaves: what it still writes of that column is known before the exchange. So a workgroup
// that gathers column k also publishes column k + 1, unless there is none, and whoever has
// gathered column k + 1 knows that all have read column k, whose words may then be emptied.
// Gathering the last published column too would break this: nobody waits for such a workgroup,
// and the words it still polls could be emptied under it for good.
DH_RING_FN int ring_gathers(int lastRow, int kEnd) { return lastRow < kEnd ? lastRow - 1 : kEnd; }

}  // namespace dftbhip

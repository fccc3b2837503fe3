// Row kernel: one workgroup integrates one (system, excitation) instance that
// does not fit the lane kernel, its stage state in LDS and its terms streamed
// in a wave-blocked layout.
//
// A side's rows become UNITS, one per thread and slot: unit u of the side is
// evaluated by lane u % 64 of wave (u / 64) % NW, slot (u / 64) / NW, so 64
// consecutive units (a BLOCK) are one wave's work and every load of a block's
// terms is contiguous.  Order of a side's units:
//   [0, pub)      published rows: some term reads them (forward: or the
//                 adjoint reads them as set points); unit u's stage value is
//                 LDS slot u.  A row of more than kRowSplitTerms terms has no
//                 terms in its unit: pieces of at most kRowPieceTerms terms
//                 (the AUX units, evaluated first) leave their sums in LDS and
//                 the unit adds them.
//   [pub, units)  sink rows (energy probes, gradient accumulators): no term
//                 reads them, so a long one is simply several units, each
//                 integrating its own terms; their sum is taken when the row
//                 is output.  A recompute of the forward path skips them.
// Units of equal term counts are neighbours, so a wave's trip counts (the
// largest of its 64 units, the others padded with terms of value 0 on a slot
// that holds 0) waste little.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace pasif {

constexpr uint32_t kRowSplitTerms = 24;
constexpr uint32_t kRowPieceTerms = 8;
constexpr uint32_t kRowThreads = 1024;
constexpr uint32_t kRowSlots = 8;            // units per thread at most
constexpr uint32_t kRowChunk = 64;           // steps whose forcing is tabulated at once
// terms of each kind a thread can hold in registers (launches of one unit per
// thread whose blocks all stay within these)
constexpr uint32_t kRowRes1 = 8, kRowRes2 = 8, kRowRes3 = 4, kRowRes4 = 2;
constexpr uint32_t kRowNone = 0xFFFFFFFFu;   // unit without a row of its own to output

// One side of one system (offsets into the packed arrays).
struct RowProg {
  uint64_t val, word;      // first term value / index word
  uint64_t blk;            // first block header: {value block, word block, counts, forced}
  uint64_t unit;           // first unit (init, force, row, piece range)
  uint64_t sink;           // first multi-piece sink: {row, first unit, end unit}
  uint32_t units, pub;     // units (padded to whole blocks in the arrays), published ones
  uint32_t aux;            // aux units
  uint32_t nsink;
};

struct RowInst {
  RowProg f, a;
  uint64_t vec_f, vec_a;   // saved unit states (and, forward, running maxima)
  uint64_t ck, seg, path;  // checkpoints, recomputed segment, stored path
  uint32_t waves;          // waves of the workgroup that work
  uint32_t n_f, steps, out_f, out_a;
  // LDS values of each stage buffer, each set-point buffer (adjoint) and the
  // sums: the instance's own, since a launch's instances need not be alike (a
  // long chain's stage buffers and the many pieces of a dense system's rows do
  // not fit beside each other, and either alone does)
  uint32_t ys, xs, ps;
  int32_t exc;
};

template <typename R>
struct RowArgs {
  const RowInst* inst;
  const uint4* blk;
  const R* val;
  const uint32_t* word;
  const R* init;
  const R* force;
  const uint32_t* row;     // row of each unit, kRowNone for a piece of a sink
  const uint32_t* piece;   // split rows: first aux unit | end << 16
  const uint32_t* sink;
  const R* excit;          // [n_exc][exc_len]
  const R* interp;         // [2][interp_w] or null (zero-order hold)
  uint32_t exc_len, interp_w;
  R h, h2, h6;
  R* vec_f;                // per instance [2][units_f]: state, running max, then the
                           // running max of each multi-piece sink
  R* vec_a;                // per instance [units_a]
  R* ckpt;                 // per instance [ceil(steps / K)][n_f]
  R* segbuf;               // recompute: [K + 1][pub] (exact: [K][4][pub]); whole
                           // path (store): [steps + 1][pub] (exact: [steps][4][pub])
  uint32_t store;          // the forward pass writes every step's set points:
                           // no checkpoints, no recompute
  uint32_t* progress;      // [inst][4]: step, phase, segment
  R* out_q;
  R* out_max;
  R* out_grad;
  R* traj;
  uint32_t out_len, save_every, nslots, window;
  uint32_t budget, ck_every, adjoint, exact;
  uint32_t resident;       // every block within kRowRes*
  uint32_t lds_slots;      // LDS values of the instance that needs most
};

// LDS values: two stage buffers, two set-point buffers (adjoint), sums, the
// forcing table
inline size_t row_lds_values(uint32_t ys, uint32_t xs, uint32_t ps) {
  return 2 * size_t(ys) + 2 * size_t(xs) + ps + 3 * kRowChunk;
}

hipError_t launch_rows(const RowArgs<double>& a, uint32_t ninst, uint32_t waves, uint32_t slots,
                       hipStream_t s);
hipError_t launch_rows(const RowArgs<float>& a, uint32_t ninst, uint32_t waves, uint32_t slots,
                       hipStream_t s);

}  // namespace pasif

// Schedule of an NTT pass, free of device code: the phase geometry (register
// windows, executed stages, twiddle chunks) and the value ranges of the u64
// arithmetic with headroom. The kernels, the host table builder and a host test
// of the ranges share it.
#pragma once

#include <cstdint>

namespace cbw {
namespace ntt_detail {

constexpr int kLE = 4;
constexpr int kE = 1 << kLE;

// ---- phase geometry (host and device) ---------------------------------------
//
// A pass butterflies LT transform bits in phases of a 4-bit register window.
// Cooley-Tukey (CT) walks the bits high -> low, windows [LT-4(P+1), LT-4P)
// clamped at 0; Gentleman-Sande (GS) walks low -> high, windows [4P, 4P+4)
// clamped at LT-4. A clamped window re-covers bits of its neighbour; only the
// bits not yet done ("active" stages) are butterflied there. Whole rows of
// 2^13 and 2^14 points (kLongRow) take the CT windows in reverse order for GS
// as well, so the clamped window is the lowest one in both directions and all
// exchanges but one stay inside a wave (Pass::wave_local).

constexpr int num_phases(int lt) { return (lt + kLE - 1) / kLE; }
constexpr int imin(int a, int b) { return a < b ? a : b; }
constexpr int imax(int a, int b) { return a > b ? a : b; }

constexpr int kLongRow = 13;  // one-pass rows from 2^13 points
constexpr int window_start(int lt, bool ct, int p) {
    if (!ct && lt >= kLongRow) return window_start(lt, true, num_phases(lt) - 1 - p);
    return ct ? imax(lt - kLE * (p + 1), 0) : (kLE * p < lt - kLE ? kLE * p : imax(lt - kLE, 0));
}
constexpr int stage_hi(int lt, bool ct, int p) {
    if (!ct && lt >= kLongRow) return stage_hi(lt, true, num_phases(lt) - 1 - p);
    const int ws = window_start(lt, ct, p);
    return ct ? imin(imin(ws + 3, lt - 1), lt - kLE * p - 1) : imin(ws + 3, lt - 1);
}
constexpr int stage_lo(int lt, bool ct, int p) {
    if (!ct && lt >= kLongRow) return stage_lo(lt, true, num_phases(lt) - 1 - p);
    const int ws = window_start(lt, ct, p);
    return ct ? ws : imax(ws, kLE * p);
}
// Stage k of the phase at window ws: its twiddle for register group g is
// table[(head >> (k+1)) + (g & gmask)], head = (prefix << lt) | (window bits
// clear). Distinct entries per thread: 2^min(ws+3-k, lt-1-k). All of a
// phase's entries hang off the block index head >> chunk_shift.
constexpr int stage_count(int lt, int ws, int k) { return 1 << imin(ws + 3 - k, lt - 1 - k); }
constexpr int chunk_shift(int lt, bool ct, int p) { return imin(window_start(lt, ct, p) + kLE, lt); }
// The final GS stage of a transform multiplies by n^-1 (no table entries).
constexpr bool scale_stage(int lt, bool ct, bool last, int k) { return !ct && last && k == lt - 1; }
// k of the s-th executed stage of a phase.
constexpr int exec_stage(int lt, bool ct, int p, int s) { return ct ? stage_hi(lt, ct, p) - s : stage_lo(lt, ct, p) + s; }
constexpr int active_stages(int lt, bool ct, int p) { return stage_hi(lt, ct, p) - stage_lo(lt, ct, p) + 1; }
// Entry offset of the s-th executed stage within the chunk, and the chunk size.
constexpr int chunk_offset(int lt, bool ct, bool last, int p, int s) {
    int off = 0;
    for (int e = 0; e < s; ++e) {
        const int k = exec_stage(lt, ct, p, e);
        if (!scale_stage(lt, ct, last, k)) off += stage_count(lt, window_start(lt, ct, p), k);
    }
    return off;
}
constexpr int chunk_entries(int lt, bool ct, bool last, int p) {
    return chunk_offset(lt, ct, last, p, active_stages(lt, ct, p));
}
// Chunk stride in entries: a multiple of 16 bytes.
constexpr int chunk_stride(int lt, bool ct, bool last, int p, int entry_bytes) {
    const int per16 = 16 / entry_bytes > 0 ? 16 / entry_bytes : 1;
    const int e = chunk_entries(lt, ct, last, p);
    return (e + per16 - 1) / per16 * per16;
}
// Chunks of one phase: one per block of the stage tree at chunk_shift,
// over the 2^(prefix_bits + lt) entries the pass covers.
constexpr std::uint64_t chunk_count(int lt, int prefix_bits, bool ct, int p) {
    return (std::uint64_t{1} << (prefix_bits + lt)) >> chunk_shift(lt, ct, p);
}

// ---- ranges of the headroom arithmetic (host and device) ---------------------
//
// In units of q; values stay below kHeadroomLimit q < 2^64. A forward stage adds
// kGrowth to every value, and a phase that would pass the limit reduces its values
// to kReduced first. Inverse stages double the sums and leave the products at
// kReduced; a pair whose sum would pass the limit is reduced first, and each phase
// ends with every value at kReduced.
constexpr int kGrowth = 3, kHeadroomLimit = 16, kReduced = 3;
// Values entering the first pass: reduced words, or canonical ones (either way
// below 4q).
constexpr int kHeadroomEntry = 4;

constexpr int forward_bound_before(int lt, int p, int bound);
// Bound after phase p of a forward pass whose values enter below `bound`.
constexpr int forward_bound_after(int lt, int p, int bound) {
    const int b = p < 0 ? bound : forward_bound_before(lt, p, bound);
    return p < 0 ? b : b + kGrowth * active_stages(lt, true, p);
}
// Bound entering phase p, after the reduction where it needs one.
constexpr int forward_bound_before(int lt, int p, int bound) {
    const int b = forward_bound_after(lt, p - 1, bound);
    return b + kGrowth * active_stages(lt, true, p) > kHeadroomLimit ? kReduced : b;
}
constexpr bool forward_reduces(int lt, int p, int bound) {
    return forward_bound_after(lt, p - 1, bound) + kGrowth * active_stages(lt, true, p) > kHeadroomLimit;
}
// Bound of the values a forward pass leaves.
constexpr int forward_exit(int lt, int bound) { return forward_bound_after(lt, num_phases(lt) - 1, bound); }

// An inverse phase: for each executed stage and register, whether its pair is
// reduced first and the bound with which it enters the butterfly; then whether
// the register is reduced at the end of the phase. `last`: the pass is the
// transform's last, whose top stage also multiplies its sums by n^-1.
struct InversePhase {
    bool reduce[kLE][kE] = {};
    int enter[kLE][kE] = {};
    bool reduce_last[kE] = {};
    bool pairs_match = true;  // both sides of every pair share a bound
    int largest = kReduced;   // largest bound any sum or difference reaches
    int largest_enter = kReduced;  // largest bound entering a butterfly (after its reduction)
};
constexpr InversePhase inverse_phase(int lt, int p, bool last) {
    InversePhase ph;
    int bound[kE] = {};
    for (int r = 0; r < kE; ++r) bound[r] = kReduced;
    for (int s = 0; s < active_stages(lt, false, p); ++s) {
        const int k = exec_stage(lt, false, p, s);
        const int jb = k - window_start(lt, false, p);
        for (int r = 0; r < kE; ++r) {
            if ((r >> jb) & 1) continue;
            const int r2 = r | (1 << jb);
            if (bound[r] != bound[r2]) ph.pairs_match = false;
            const bool reduce = bound[r] + bound[r2] > kHeadroomLimit;
            if (reduce) bound[r] = bound[r2] = kReduced;
            ph.reduce[s][r] = ph.reduce[s][r2] = reduce;
            ph.enter[s][r] = bound[r];
            ph.enter[s][r2] = bound[r2];
            // The difference's span is the subtrahend's bound: it reaches the sum's.
            ph.largest = imax(ph.largest, bound[r] + bound[r2]);
            ph.largest_enter = imax(ph.largest_enter, bound[r2]);
            bound[r] = scale_stage(lt, false, last, k) ? kReduced : bound[r] + bound[r2];
            bound[r2] = kReduced;
        }
    }
    for (int r = 0; r < kE; ++r) ph.reduce_last[r] = bound[r] > kReduced;
    return ph;
}

}  // namespace ntt_detail
}  // namespace cbw

// seq_layout.h -- sizes of the in-order sums (seqsum.hip) and the reach of
// their loads; plain C++, so that a host test can follow them.
#pragma once

namespace m2d {

constexpr int kSeqSeg = 512;        // terms of a segment: 8 per lane
constexpr int kSeqSegDoubles = 7;   // doubles of a segment's map
// One launch (k_seq_final, every segment from its terms, about 3 us each) up
// to this many terms, three above: 10 us against 13 at 2048 terms, 17 against
// 13 at 4096.
constexpr long kSeqDirect = 2048;

// segments with maps of a sum of n terms
constexpr int seq_segments(long n)
{
    return n <= kSeqDirect ? 0 : (int)((n + kSeqSeg - 1) / kSeqSeg);
}

// Doubles that follow the K arrays of n terms: the maps, and at least one,
// because the one-by-one loads take whole 16-byte pairs and the last may hold
// one double past the terms.
constexpr long seq_scratch(long n, int K)
{
    return seq_segments(n) ? (long)seq_segments(n) * K * kSeqSegDoubles : 1;
}

// The one-by-one loads of n terms read a stream of pairs that starts sh (0 or
// 1) doubles before the first term, on a 16-byte boundary: the position in
// it of the last pair.
constexpr long seq_last_pair(long n, int sh) { return (n + sh - 1) & ~1L; }

}  // namespace m2d

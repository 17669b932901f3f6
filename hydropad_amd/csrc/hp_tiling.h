// hp_tiling.h -- how a sweep's cells are dealt out over waves: chunks of an x
// sweep, pencil segments of a y/z sweep.  Host arithmetic and the index a wave
// derives from it, with no GPU call, so it is checked on the CPU.
#pragma once

#ifdef __HIP__
#define HP_TILING_FN __host__ __device__ inline
#else
#define HP_TILING_FN inline
#endif

namespace hp {

// Chunks of 58 cells each wave of an x sweep (or unit of a batch's) walks: one
// where the box has few, more as it grows, since a wave's first chunk waits for
// its loads and for the box's scalars; 16 only where even those make 48
// thousand waves, as short runs balance the Riemann work.  Measured, us at 1,
// 2, 4, 8, 16: 64^3 comoving [33] 36 47 64 117; 96^3 80 [76] 80 88 121; 128^3
// 165 [163] 169 177 220; 192^3 516 488 [480] 494 512; 256^3 1190 1119 1088
// [1094] 1120; 512x512x64 mixed tube 789 714 637 [627] 638; 512x512x256 tube
// 3978 3494 3004 2938 [2890].
inline int x_chunks_per_wave(long nchunks)
{
    int n = 1;
    for (long most = 12000; nchunks >= most && n < 16; most *= 4) n *= 2;
    return n;
}

// Waves of a y/z sweep the chip holds at once, for each wave its SIMD holds:
// 256 CUs x 4 SIMDs.
constexpr int STREAM_SLOTS = 1024;

// Segments of a pencil that stand side by side in a wave: one where the box
// has more than 32 pencils, else as many as fill its 64 lanes.  Measured, z
// sweep in us, of noise, with a segment to each four waves and as here: 3 x 3
// x 100000 cells 1118 -> 209, 4 x 4 x 20000 315 -> 60, 8 x 8 x 8192 134 -> 67,
// 10 x 10 x 100000 1290 -> 894.
HP_TILING_FN unsigned stream_pack(unsigned npen) { return npen > 32u ? 1u : 64u / npen; }

// Waves of a y/z sweep of npen pencils in nseg segments each.  A box has fewer
// than 2^31 cells, ghosts included, and at least 3 ghost cells on either side,
// so the 64 lanes of these waves number less than 2^32 also where every
// segment is one cell: (npen + 63) nax < 2^31 + 63 x 2^31 / 81.
HP_TILING_FN long stream_items(long npen, long nseg)
{
    const long k = stream_pack((unsigned)npen);
    return k > 1 ? (nseg + k - 1) / k : (npen + 63) / 64 * nseg;
}

// The work of one of stream_items' waves.  Consecutive waves take consecutive
// pencils of one segment, whose rows are consecutive memory, and a segment of
// all pencils comes before the next (one wave's 512 bytes at a time with the
// segments side by side: 512x512x256 tube 1405 -> 1704 us, 256^3 comoving
// 1065 -> 1110).
struct StreamItem {
    unsigned pen, seg;
    bool active;
};
HP_TILING_FN StreamItem stream_item(unsigned wave, unsigned lane, unsigned npen, unsigned nseg)
{
    const unsigned k = stream_pack(npen);
    StreamItem I;
    if (k > 1u) {
        const unsigned part = lane / npen;
        I.seg = wave * k + part;
        I.pen = lane - part * npen;
        I.active = part < k && I.seg < nseg;
    } else {
        const unsigned rows = (npen + 63u) >> 6;
        I.seg = wave / rows;
        I.pen = (wave - I.seg * rows) * 64u + lane;
        I.active = I.pen < npen && I.seg < nseg;
    }
    if (!I.active) I.pen = I.seg = 0u;
    return I;
}

// Segment length of a y/z sweep whose pencils are `nax` cells long and take
// `waves(nseg)` waves when each is split into nseg segments.  A wave walks a
// segment of len cells in len + 6 iterations, the first four of them cheap:
// about len + 4 cells' time, and the waves run in rounds of `slots`.  The
// split with the smallest rounds x (len + 4) is taken, at most 24 cells long:
// short enough that the waves that got the most Newton iterations do not run
// on alone, and that the rows two segments share are still in cache.  Measured, y sweep in us, by length (taken one in brackets):
//   64^3 tube                 64: 155   16: 49   8: 33   [2]: 24
//   96^3 comoving             48: 353   16: 133  7: 94   [5]: 96   4: 107
//   128^3 comoving            64: 448   32: 245  16: 174 [11]: 167  10: 181
//   192^3 comoving            64: 640   28: 503  24: 520 [20]: 475  18: 491
//   256^3 comoving            64: 1053  32: 1010 24: 984 [22]: 1042 16: 1023
//   512^3 tube                128: 3270 64: 3132 32: 2995 [20]: 2854 16: 2811
// A length just past a full round (10 at 128^3, 24 at 192^3) is slower than
// its neighbours.
template <class Waves> inline int stream_seglen(int nax, int slots, Waves waves)
{
    int best = nax;
    long cost = -1;
    for (int most = nax < 24 ? nax : 24; most >= 1; --most) {
        const int shares = (nax + most - 1) / most, len = (nax + shares - 1) / shares;   // even shares
        const long rounds = (waves((nax + len - 1) / len) + slots - 1) / slots;
        const long c = rounds * (len + 4);
        if (cost < 0 || c < cost) { cost = c; best = len; }
    }
    return best;
}

}  // namespace hp

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

// Waves per SIMD that a y/z kernel is built for and its launch fills: what LDS
// holds of its window (three blocks of 53 KB per CU, two of 61 KB with
// gravity), and the registers left after it (at most 168 for three waves: the
// gamma = 5/3 forms need 129 to 168, the general-gamma and the reference-order
// forms 175 to 237).
constexpr int stream_waves(bool g53, bool grav) { return g53 && !grav ? 3 : 2; }

// Waves per SIMD of the batch's x kernels, bound by their registers (four
// waves: 128).
constexpr int batch_x_waves(bool g53, bool mixed) { return (mixed ? 3 : 2) + (g53 ? 1 : 0); }

constexpr int SIMDS = 4;   // per CU

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
// `waves(nseg)` waves when each is split into nseg segments, on `simds` SIMDs
// that hold `resident` waves each.  A wave walks a segment of len cells in
// len + 6 iterations, the first four of them cheap: about len + 4 cells' time.
// The waves run in rounds of simds x resident; a round that puts m waves on a
// SIMD takes 1 + 0.3 (m - 1) of one wave's time alone (96^3 comoving, us per
// cell at one, two and three waves: 6.8, 8.8, 10.9).  The split with the
// shortest time is taken, at most 24 cells long: the waves that got the most
// Newton iterations must not run on alone, and the rows two segments share
// should still be in cache.  Measured, y sweep in us, by length (taken one in
// brackets; over 46 sweeps of 64^3 to 512^3 it is 1.1 % off the best length on
// average, 5.9 % at most):
//   64^3 tube        64: 152   16: 50   8: 33   4: 25   [2]: 23.8   1: 30
//   96^3 comoving    48: 363   16: 137  [7]: 95.5  5: 98.3  4: 109
//   96^3 tube        48: 115   16: 48   [7]: 35.5  5: 36.8  4: 42.7
//   128^3 comoving   64: 463   32: 255  15: 171 [11]: 172  10: 187
//   160^3 comoving   32: 353   [23]: 337  20: 392  13: 323  11: 324  7: 324
//   192^3 comoving   64: 664   32: 591  24: 536 [20]: 494  16: 514  12: 501
//   256^3 comoving   64: 1142  32: 1091 24: 1068 [22]: 1074 16: 1110 12: 1115
//   512^3 tube       128: 3268 64: 3142 32: 3014 24: 2924 [19]: 2858 16: 2813
// 160^3 and 192^3 show what the rounds leave out: one or two of them balance
// the Newton work less well than three or four shorter ones (3 to 6 %).
template <class Waves> inline int stream_seglen(int nax, long simds, int resident, Waves waves)
{
    int best = nax;
    long cost = -1;
    for (int most = nax < 24 ? nax : 24; most >= 1; --most) {
        const int shares = (nax + most - 1) / most, len = (nax + shares - 1) / shares;   // even shares
        const long n = (waves((nax + len - 1) / len) + simds - 1) / simds;   // waves per SIMD
        const long part = n % resident;
        const long c = (len + 4) * (n / resident * (7 + 3 * resident) + (part ? 7 + 3 * part : 0));
        if (cost < 0 || c < cost) { cost = c; best = len; }
    }
    return best;
}

// A box of a batch: its interior and the kernels that sweep it.
struct BatchShape {
    int Nx, Ny, Nz;
    bool g53, mixed;
};
constexpr int BATCH_FORMS = 4;
HP_TILING_FN int batch_form(bool g53, bool mixed) { return 2 * mixed + g53; }

// x chunks per unit and y/z segment length of the boxes of one form: a launch
// holds those, so they are dealt out by the rules of the single-box sweeps on
// their chunks and waves, the latter against a persistent grid of `blocks` of
// four waves, at most three to a CU.  Measured, ms per step, all boxes dealt
// out together and by form: 48^3 and two 64^3 in each of the four forms 1.39
// -> 0.92, 48^3 to 96^3 in both precisions 0.87 -> 0.73.  Three to a CU stands
// for the general-gamma kernels too, though they hold two: with two counted
// the segments came out longer and no batch faster (48^3 to 96^3 0.54 -> 0.58).
struct FormTiling {
    int chunks, len;
};
inline FormTiling form_tiling(const BatchShape* boxes, int n, int form, int blocks, int ncu)
{
    const auto in_form = [&](const BatchShape& X) { return batch_form(X.g53, X.mixed) == form; };
    int nax = 1;
    long nchunks = 0;
    for (int i = 0; i < n; ++i) {
        const BatchShape& X = boxes[i];
        if (!in_form(X)) continue;
        nax = X.Ny > nax ? X.Ny : nax;
        nax = X.Nz > nax ? X.Nz : nax;
        nchunks += ((long)X.Ny * X.Nz * (X.Nx + 6) + 57) / 58;
    }
    const int grid = blocks < 3 * ncu ? blocks : 3 * ncu;
    const int resident = (grid + ncu - 1) / ncu;
    FormTiling T;
    T.chunks = x_chunks_per_wave(nchunks);
    T.len = stream_seglen(nax, (long)grid * SIMDS / resident, resident, [&](int nseg) {
        const int l = (nax + nseg - 1) / nseg;
        long waves = 0;
        for (int i = 0; i < n; ++i)
            if (in_form(boxes[i])) waves += stream_items((long)boxes[i].Nx * boxes[i].Ny, (boxes[i].Nz + l - 1) / l);
        return waves;
    });
    return T;
}

}  // namespace hp

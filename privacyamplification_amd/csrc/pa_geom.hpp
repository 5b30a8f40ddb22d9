// pa_geom.hpp -- block geometry shared by the host planner and the kernels.
//
// A block (n, m, flags) is evaluated as a circular convolution of length L (a power of two, L >= n)
// of the key x (kbits = h+1 bits, h = n-m) with the seed t (n bits, rotated left by m when L > n),
// read at conv indices [out_off, out_off + out_bits).  For power-of-two n, L = n and out_off = 0,
// which is the reference's own circular form y[p] = XOR_j x[j] s[(p-j) mod n].
//
// The four-step path (L > 2^14) evaluates the NEGACYCLIC convolution of length L instead, c[q] =
// sum_j sgn a[j] b[(q - j) mod L], sgn = -1 for j > q: wrapped terms change sign, which no parity
// sees.  The polynomial product mod z^L + 1 is one complex transform of length N = L/2 per operand,
// z[t] = a[t] - i a[t + N], at the quarter-shifted frequencies k + 1/4, whose values are multiplied
// point by point: no real-FFT split, and so no frequency needs a partner from another row.
//   Mean.  a, b are the bits minus 1/2.  With PX(q), PT(q) the inclusive prefix sums of both bit
// sequences up to q and W the sum of both popcounts, sum_j sgn x[j] t[(q-j) mod L] = c[q] + PX(q) +
// PT(q) - (W + q + 1)/2 + L/4.  So round(c[q] - ((W + q + 1) mod 4)/2), plus the parities of PX and PT,
// is the bit; the parities are a bit scan over the inputs (prefix_chunk).
//   Whitening.  The constant part of one operand (its mean, the key's zero pad) times a constant or
// periodic part of the other would give values that grow like n/4, or spectral lines whose rounding errors
// alone reach 1/2.  The key is therefore XORed with R, whole words of zeros and ones in a
// pseudo-random order of long period (white_word): every simple key and its pad then have a flat spectrum, and
// an operand with a flat spectrum multiplies any other to small values, as random keys do.
//   The order is a sum mod 2 of levels: word w has sign s_l[(w / b_l) mod c_l], b = 1, 16, 256.  Each
// level's second half is the complement of its first, so R is balanced and has no line at a frequency that
// a sequence of half its period, or of any power of two below, has.  conv(R, t) mod 2 has R's period,
// follows from the seed words folded to that period (white_table) and is added back by the output stage.
//   N = N1 * N2 (t = t2 + N2*t1, k = k1 + N1*k2):
//   pass A  column FFTs of length N1, 16 columns per workgroup.  L >= 2^25: decimated by D classes of
//           k1 (M = N1/D per class), input from the bit-transposed key/seed; the mid sizes (mid_size:
//           up to 2^24 and every 3 * 2^k), straight from the words (k_mid_fwd, k_mix_fwd);
//   pass B  row FFTs of length N2, complex product, inverse row FFTs;
//   pass A' inverse column FFTs of length N1, rounding; for the mid sizes the output words too.
// L >= 2^23 has N2 = 8192.  Below, N1 is 2^6 .. 2^9 and N2 = N / N1 is 2^8 .. 2^12 (mid_lg1; N1 is 2^9 and 2^10
// at 2^23 and 2^24): as many row and column workgroups as the length allows, because there the time is one
// workgroup's latency -- at N2 = 8192 a row's three transforms alone take 20 us on one compute unit.
// N <= 8192 (L <= 2^14) runs fully on chip in one workgroup (small path).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pa {

constexpr int ROW_LOG = 13;            // N2 = 8192 from L = 2^23 on
constexpr int SMALL_MAX_LOG_N = 13;    // N <= 8192 -> single-workgroup path
constexpr int MAX_L_LOG = 29;          // largest transform served (L = 2^29; the reference stops at 2^27)

// The levels' signs: index i at bit i.  Periods of 16 * 8 words for the mid sizes, where the values are small
// enough, and 16 * 16 * 16 for the others.  Chosen among 60 and 80 random ones by the rounding margin (max
// |v - rint v|) of an all-ones key at 2^24 bits in an FP32 emulation of the passes, against constant seeds, square
// waves and repeated random words: 0.05 and 0.011 at worst, for seeds of exactly R's period.  A constant seed
// at 2^25 bits has 0.0017 with the long period, 0.028 with 128 words and 0.22 with alternating blocks of 256.
// Largest margins measured over constant, 7/8 and random keys and seeds that repeat 1 to 64 words: 0.05 at 2^24,
// 0.008 at 2^26, 0.014 at 2^27, 0.06 at 2^28, 0.13 at 2^29 bits (the seed alone whitened by a word of 32 bits: 0.5
// from 2^26 on).
constexpr uint32_t WHITE_MID = 128, WHITE_BIG = 4096;   // words
constexpr uint32_t WHITE_S0 = 0x946Bu, WHITE_S1 = 0xD629u, WHITE_S2 = 0x15EAu;   // c = 16 each
constexpr uint32_t WHITE_MID_S0 = 0x6699u, WHITE_MID_S1 = 0xC3u;                 // c = 16, 8

// Pass B's output R'[k1][t2] when 2^RT_LG1_MIN <= N1 <= 2^RT_LG1_MAX (transforms of 2^25 to 2^29
// bits) goes to its own buffer in tiles, Rt[((t2 / RT_COLS) N1 + k1) RT_COLS + t2 mod RT_COLS]: pass
// B writes whole 128-byte lines, and a workgroup of pass A' (1 to 8 columns) reads its columns from
// consecutive lines along k1 instead of from rows 8 N2 bytes apart.  At N1 = 2^RT_LG1 pass A' runs
// two 256-thread workgroups per CU.
constexpr int RT_LG1_MIN = 11;
constexpr int RT_LG1 = 13;
constexpr int RT_LG1_MAX = 15;
constexpr int RT_COLS = 16;
__host__ __device__ constexpr bool rt_tiled(uint32_t lg1) {
    return lg1 >= (uint32_t)RT_LG1_MIN && lg1 <= (uint32_t)RT_LG1_MAX;
}

// log2(N1) of a transform of 2^14 <= N <= 2^MID_MAX_LOG_N complex points.
__host__ __device__ constexpr int mid_lg1(int lgN) {
    return lgN >= 23 ? 10 : lgN >= 21 ? 9 : lgN >= 16 ? 8 : lgN - 8;
}
constexpr int MID_MAX_LOG_N = 23;

// Transforms of 3 * 2^k, for blocks of 2^(k+1) < n <= 3 * 2^k bits, which a power of two would pad by a third
// and more: N1 = D * 256 columns points in D = 3 classes, or 6 where N2 = 8192 makes it necessary, whose
// sums over the class bits come from a table (k_mix_fwd), so the factor 3 costs pass A nothing; pass B
// is as ever.  Against the power of two, blocks of 0.7 * 2^k bits, us of one block / a block in a batch of 2^27
// bits: k = 19 22.3 / 2.85 to 21.5 / 2.09, k = 22 43.3 / 22.8 to 42.5 / 16.9, k = 23 66 / 48 to 53 / 33, k = 24 123 /
// 101 to 98 / 70, k = 25 266 / 214 to 174 / 155; on a resident seed k = 19 23.1 / 2.17 to 20 / 1.6, k = 22 32.7 / 16.7 to
// 35.1 / 12.3 (the one loss), k = 25 215 / 171 to 129 / 115.  Below k = 19 the direct product takes single blocks.
constexpr uint32_t MIX_M = 256;
constexpr int MIX_MIN_LOG_L = 19, MIX_MAX_LOG_L = 25;  // ceil(log2 L) of the lengths served
__host__ __device__ constexpr uint32_t mix_classes(int lgL) { return lgL == 25 ? 6u : 3u; }

struct Geom {
    uint32_t n, m, h, kbits;           // block shape; kbits = h + 1
    uint32_t L, N, lgN;                // transform length, half length, ceil(log2 N)
    uint32_t N1, N2, lg1, lg2;         // four-step split (N1 = 1 on the small path); lg1: floor(log2 N1)
    uint32_t M, D;                     // pass A class length / classes (3 or 6: a transform of 3 * 2^k)
    uint32_t out_bits, out_off;        // output window in conv indices
    uint32_t seed_words, seed_rot;     // n/32, rotation of the seed in words (m/32 when L > n); the
                                       // rotated seed repeats with period n up to L
    uint32_t key_hw;                   // h/32: index of the key word masked to its MSB
    uint32_t do_xor, reverse_endian;
    uint32_t white;                    // period of the key's whitening in words (0 on the small path)
    uint32_t scan;                     // words per scan chunk: 1024 << scan
    float inv_N;                       // output normalisation: 1/N; on the small path 1/(8N), with the
                                       // factor of r2c_split / c2r_split
};

// A four-step transform of the mid sizes: no bit masks, no separate output stage.
__host__ __device__ inline bool mixed(const Geom& g) { return g.D % 3u == 0u; }
__host__ __device__ inline bool mid_size(const Geom& g) { return g.N1 > 1u && (g.lgN <= (uint32_t)MID_MAX_LOG_N || mixed(g)); }

// The direct product (k_direct) serves what it finishes sooner than the transform: blocks of the one-
// workgroup sizes, and up to L = 2^DIRECT_MAX_L_LOG one block, or all of a batch's group, of up to
// DIRECT_WORK products of a key word and an output word.  One block: 2^17 bits (3.9 M) 10.3 against 18.0 us,
// 2^18 (15.7 M) 21.8 against 20.8; batches of 128: 2^15 0.34 against 0.27 us a block beside the
// call's fixed 27, 2^16 1.1 against 0.37.
constexpr int DIRECT_MAX_L_LOG = 18;
constexpr uint64_t DIRECT_WORK = 12u << 20;
constexpr uint32_t DIRECT_NT_MAX = 1024;
constexpr uint32_t DIRECT_JPAD_MAX = 8000;  // key and seed words in 64 KB of LDS
// Key words of the direct product, padded to its chunks.
__host__ __device__ inline uint32_t direct_key_words(const Geom& g) { return (g.key_hw + 16u) & ~15u; }
inline uint64_t direct_work(const Geom& g) { return (uint64_t)(g.out_bits >> 5) * direct_key_words(g); }
// work: of the block, or of the blocks that share a launch.
inline bool direct_size(const Geom& g, uint64_t work) {
    return g.N1 == 1u || (g.L <= (1u << DIRECT_MAX_L_LOG) && work <= DIRECT_WORK && direct_key_words(g) <= DIRECT_JPAD_MAX);
}

// Word w of the key's whitening R (zero on the small path).
__host__ __device__ inline uint32_t white_word(const Geom& g, uint32_t w) {
    const bool big = g.white == WHITE_BIG;
    const uint32_t s0 = big ? WHITE_S0 : g.white ? WHITE_MID_S0 : 0u, s1 = big ? WHITE_S1 : g.white ? WHITE_MID_S1 : 0u;
    const uint32_t s = (s0 >> (w & 15u)) ^ (s1 >> ((w >> 4) & (big ? 15u : 7u))) ^ (big ? WHITE_S2 >> ((w >> 8) & 15u) : 0u);
    return 0u - (s & 1u);
}

// Inputs and outputs of the input scan: conv words of the key and the fresh seed (or the resident
// seed's finished prefix words sq); prefix words q, and the block's info words.
struct ScanArgs {
    const uint32_t* key;
    const uint32_t* seed;
    const uint32_t* sq;
    uint32_t* q;
    uint32_t* info;
};
// A block's info buffer: both popcounts; per chunk one byte, its parity; conv(R, t), g.white words; per
// chunk its popcount; the fresh seed's words folded to the whitening's period, in fold_slices parts of
// g.white words: one a chunk for the mid sizes (scan_chunk), else one per 16 values of the bit
// transpose's u.
constexpr int INFO_POPS = 0;    // both popcounts
constexpr int INFO_HEAD = 64;   // words before the parities
__host__ __device__ inline uint32_t scan_chunks(const Geom& g) { return g.L >> (15u + g.scan); }
__host__ __device__ inline uint32_t fold_slices(const Geom& g) { return g.white == WHITE_BIG ? g.M / 16u : scan_chunks(g); }
__host__ __device__ inline uint8_t* scan_parities(uint32_t* info) { return reinterpret_cast<uint8_t*>(info + INFO_HEAD); }
__host__ __device__ inline const uint8_t* scan_parities(const uint32_t* info) { return reinterpret_cast<const uint8_t*>(info + INFO_HEAD); }
__host__ __device__ inline uint32_t info_white(const Geom& g) { return (uint32_t)INFO_HEAD + (scan_chunks(g) + 255u) / 256u * 64u; }
__host__ __device__ inline uint32_t info_pops(const Geom& g) { return info_white(g) + g.white; }
__host__ __device__ inline uint32_t info_fold(const Geom& g) { return info_pops(g) + (scan_chunks(g) + 63u) / 64u * 64u; }
inline uint64_t info_bytes(const Geom& g) { return ((uint64_t)info_fold(g) + (uint64_t)fold_slices(g) * g.white) * 4u; }

// One block of a batched launch: its geometry and device buffers.  The blocks of one launch share
// the transform length L (and so N1, N2, M, D); n, m, flags and the buffers are per block.
struct BlockArgs {
    Geom g;
    const uint32_t* key;
    const uint32_t* seed;   // dynamic seed, or nullptr for a resident one (its words for the direct product)
    const float2* sspec;    // resident spectrum when seed == nullptr
    const uint32_t* ws;     // resident seed popcount partials, and its conv(R, t), when seed == nullptr
    const uint32_t* sq;     // resident seed prefix words when seed == nullptr (four-step path only)
    float2* Yk;             // N values (four-step path only)
    float2* Ys;             // N+1 values (dynamic seed, four-step path only)
    uint32_t* tbk;          // bit masks (not for mid_size)
    uint32_t* tbs;
    float2* Rt;             // R' tiles (rt_tiled(lg1)), else nullptr
    uint8_t* nib;
    uint32_t* info;         // info words (above)
    uint32_t* q;            // prefix words, L / 32 (in nib's upper half)
    uint32_t* out;
    float* margin;          // may be nullptr
};

}  // namespace pa

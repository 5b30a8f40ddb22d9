// pa_kernels.hpp -- host-side launchers of the gfx950 kernels (internal to libpa_hip.so).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pa_geom.hpp"

namespace pa {

enum { ROWS_DYN = 0, ROWS_STATIC = 1, ROWS_SEEDPREP = 2 };
// Row pass: rows per workgroup (a row takes N2 / 16 threads, N2 / 32 at 8192), and those of batched launches
// with at least 1024 such workgroups (four a compute unit), 256 threads each: the twiddle tables that a
// workgroup loads first are 3 KB, as much as half a row of 2^9 points or less.  Us a block with few / many
// rows: 2^18 bits, batch of 256, 1.52 / 1.47, resident 1.15 / 1.07; 2^19 2.95 / 2.84 and 2.25 / 2.12; 733984
// bits, batch of 182, 4.35 / 4.19 and 3.29 / 3.09; 64 of 2^18 on a resident seed 98.8 / 95.0 us a call.
__host__ __device__ constexpr int rows_per_wg(int lg2) { return lg2 == 8 ? 4 : lg2 == 9 ? 2 : 1; }
__host__ __device__ constexpr int rows_per_wg_many(int lg2) { return lg2 >= 12 ? 1 : 4096 >> lg2; }
__host__ __device__ constexpr int rows_threads(int lg2, int rpw) { return lg2 == 13 ? 256 : rpw * (1 << lg2) / 16; }
// Column passes of the mid sizes, powers of two: threads and first radix (16 columns, one second-stage butterfly each).
__host__ __device__ constexpr int mid_threads(int lg1) { return lg1 >= 10 ? 512 : lg1 >= 8 ? 256 : 1 << lg1; }
__host__ __device__ constexpr int mid_r1(int lg1) { return lg1 >= 10 ? 32 : lg1 >= 8 ? 16 : 1 << (lg1 - 4); }
constexpr int TB_NT = 128;        // bit-transpose threads: 32 outputs each
constexpr int TB_SPAN_LOG = 12;   // bit-transpose outputs per workgroup (2^12 of a row of N2 = 2^13)
constexpr int POP_SLOTS = 64; // partial popcounts of a resident seed
constexpr int PACK_NT = 128;  // output stage: threads and word columns of a tile
constexpr int PACK_CW = 16;

// Device twiddle tables: tw14[x] = exp(-2 pi i x / 2^14); lo/hi: exp(-2 pi i x / (2L)) split as
// lo[x mod 2^14] * hi[x >> 14].
// cls: pass A's tables, cls_table_offset(D) onwards, of the class pairs (p, p + D/2), p < D/2.
// The sum over v of z[v] w_D^{v (c + 1/4)} is S_even + S_odd for c = p and S_even - S_odd for
// c = p + D/2, S_even over the even v.  Table q of pair p, entries [(p NB + q) 2^BW + index], BW index
// bits: up to D = 8, q = 0 is S_even and q = 1 S_odd, and the index is the bits of a's D/2 values and
// above them those of a[. + N] (z = a - i a[. + N]).  From D = 16 on the sums of one half's bits are
// split into bytes, q < NB/2 even and the others odd.  a = bit - 1/2; computed in double precision
// and rounded once.
struct Tables {
    const float2* tw14;
    const float2* lo;
    const float2* hi;
    const float2* cls;
};
__host__ __device__ constexpr int cls_bits(int D) { return D < 8 ? D : 8; }
__host__ __device__ constexpr int cls_tables(int D) { return D <= 8 ? 2 : D / 8; }
__host__ __device__ constexpr int cls_table_size(int D) { return D / 2 * cls_tables(D) * (1 << cls_bits(D)); }
__host__ __device__ constexpr int cls_table_offset(int D) {
    return D <= 4 ? 0 : cls_table_offset(D / 2) + cls_table_size(D / 2);
}
constexpr int CLS_TABLE_TOTAL = cls_table_offset(64);  // D = 4 .. 32
// Tables of the transforms of 3 * 2^k, 64 entries a class, behind those: of D = 3 by the class bits of a
// (bits 0 .. 2) and of a[. + N] (3 .. 5), of D = 6 by the bits of either, to be added with a factor -i.
__host__ __device__ constexpr int mix_table_offset(int D) { return CLS_TABLE_TOTAL + (D == 6 ? 3 * 64 : 0); }
constexpr int CLS_TABLES_ALL = CLS_TABLE_TOTAL + 9 * 64;
// Place in a mask word (D = 32: a word per half) of class bit v of half h, in the tables' order.
__host__ __device__ constexpr int mask_bit(int D, int h, int v) {
    return D <= 8 ? (v & 1) * D + h * (D / 2) + v / 2 : (D == 16 ? 16 * h : 0) + (v & 1) * (D / 2) + v / 2;
}

// Columns per workgroup in pass A' and its threads: N1 = 2^11, 2^12 take 8192 / N1 (about 68 KB of LDS)
// and N1 = 8192 takes 2 columns one at a time, so that two workgroups share a compute unit.
__host__ __device__ constexpr int inv_cols_width(int lg1) { return lg1 >= 13 ? 2 : 1 << (13 - lg1); }
__host__ __device__ constexpr int clamp_threads(int t) { return t < 64 ? 64 : (t > 1024 ? 1024 : t); }
__host__ __device__ constexpr int inv_cols_threads(int lg1) { return lg1 == 13 ? 256 : 512; }
// Threads of pass A: 16 columns, one second-stage butterfly each.
__host__ __device__ constexpr int fwd_cols_threads(int lgm) { return 16 << (lgm - 5); }
// Bytes of the nib buffer: pass A''s pieces (one bit per conv value, N/4 bytes), then the prefix
// words (L/8 bytes).
__host__ __device__ constexpr uint64_t nib_bytes(uint32_t N) { return N / 2 + 64; }
inline uint32_t* prefix_words(uint8_t* nib, uint32_t N) { return reinterpret_cast<uint32_t*>(nib + N / 4); }
__host__ __device__ constexpr int small_threads(int lgn) { return clamp_threads(2 * (1 << lgn) / 16); }

// A staging range: `bytes` from src to dst, either side device memory or pinned, device-mapped
// host memory.
struct CopyDesc {
    const uint8_t* src;
    uint8_t* dst;
    uint64_t bytes;
};
// Copies every range of d[0 .. count) in one launch; max_bytes = the longest range.
hipError_t launch_copies(const CopyDesc* d, uint32_t count, uint64_t max_bytes, hipStream_t s);
// Bit masks of `ops` operands from `first` on (0 key, 1 seed); scan != 0: the launch also scans the
// inputs (ScanArgs), which takes every operand of the block.
hipError_t launch_transpose(const uint32_t* key, const uint32_t* seed, uint32_t* tbk, uint32_t* tbs, uint32_t first,
                            uint32_t ops, const Geom& g, const ScanArgs* scan, hipStream_t s);
// Pass A of `ops` operands from `first` on; in: the masks, or for a mid-size transform the words, and
// there the scan as above.
hipError_t launch_fwd_cols(const uint32_t* key_in, const uint32_t* seed_in, float2* Yk, float2* Ys, uint32_t first,
                           uint32_t ops, const Geom& g, const Tables& t, const ScanArgs* scan, hipStream_t s);
// ROWS_SEEDPREP: S <- spectrum of the seed rows held in S (in place, N values).
// ROWS_STATIC:   R' from the key rows in Yk and the seed spectrum S.
// ROWS_DYN:      R' from the key rows in Yk and the seed rows (pass-A output) in S.
// R' goes to Rt in tiles when rt_tiled(g.lg1) (N complex values), else to Yk in place.
// info: finished by the launch (ws: a resident seed's popcount partials; seed_ws: receives them).
hipError_t launch_rows(int mode, float2* Yk, float2* S, float2* Rt, const Geom& g, const Tables& t, uint32_t* info,
                       const uint32_t* ws, uint32_t* seed_ws, hipStream_t s);
// A resident seed's chunk-wise prefix words q[0 .. L/32) finished with its chunks' parities.
hipError_t launch_prefix_apply(uint32_t* q, const uint32_t* info, const Geom& g, hipStream_t s);
// R: pass B's tiles (transformed in place from L = 2^28 on).
hipError_t launch_inv_cols(float2* R, uint8_t* nib, const Geom& g, const uint32_t* info, const Tables& t,
                           float* margin, hipStream_t s);
hipError_t launch_pack(const uint8_t* nib, const uint32_t* key, uint32_t* out, const Geom& g, const uint32_t* info,
                       const uint32_t* q, hipStream_t s);
// Pass A' and the output of a mid-size transform.
hipError_t launch_mid_inv(const float2* R, const uint32_t* key, uint32_t* out, const Geom& g, const uint32_t* info,
                          const uint32_t* q, const Tables& t, float* margin, hipStream_t s);
// A block by the direct product, and `count` of them: words, jpad: the most output words and key words
// (direct_key_words) of a block of the launch.  BlockArgs: g, key, seed and out.
hipError_t launch_direct(const uint32_t* key, const uint32_t* seed, uint32_t* out, const Geom& g, hipStream_t s);
hipError_t launch_batch_direct(const BlockArgs* bt, uint32_t count, uint32_t words, uint32_t jpad, hipStream_t s);
hipError_t launch_small(const uint32_t* key, const uint32_t* seed, const float2* sspec,
                        const uint32_t* ws_ptr, uint32_t* out, const Geom& g, const Tables& t,
                        float* margin, float2* sspec_out, uint32_t* ws_out, hipStream_t s);

// Batched forms: `count` blocks of one transform length in one launch each (grid z = block),
// block b's geometry and buffers in bt[b] (device memory); g0 is any block's geometry.
uint32_t pack_halves(const Geom& g);  // halves of the conv positions (t, t + N) the window touches
// ops: 1 (key) or 2 (key and seed).
hipError_t launch_batch_transpose(const BlockArgs* bt, uint32_t count, const Geom& g0, uint32_t ops, hipStream_t s);
// per: column groups each workgroup of pass A walks (L >= 2^25), a power of two up to 32; 0 picks one.
hipError_t launch_batch_fwd_cols(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, uint32_t ops,
                                 uint32_t per, hipStream_t s);
constexpr uint32_t FWD_PER_MAX = 32;
hipError_t launch_batch_rows(int mode, const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t,
                             hipStream_t s);
hipError_t launch_batch_inv_cols(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, hipStream_t s);
// halves: the most of a block of the launch.
hipError_t launch_batch_pack(const BlockArgs* bt, uint32_t count, const Geom& g0, uint32_t halves, hipStream_t s);
hipError_t launch_batch_mid_inv(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, hipStream_t s);
hipError_t launch_batch_small(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, hipStream_t s);

// Sub-block split (tiles of b x b through the batched engine, XOR-accumulated per band).
hipError_t launch_tile_inputs(const uint32_t* key, const uint32_t* seed, uint32_t n, uint32_t h, uint32_t b,
                              uint32_t nbands, uint32_t j0, uint32_t tiles, uint32_t* tkeys, uint32_t* tseeds,
                              hipStream_t s);
hipError_t launch_tile_xor(uint32_t* acc, const uint32_t* tout, uint32_t nbands, uint32_t wb, uint32_t cols,
                           int first, hipStream_t s);
hipError_t launch_split_finish(const uint32_t* acc, const uint32_t* key, uint32_t* out, uint32_t m, uint32_t h,
                               uint32_t do_xor, uint32_t reverse_endian, hipStream_t s);

// Self-test kernels (pa_selftest.hip): production device functions on closed-form inputs.
hipError_t launch_st_correction(const uint32_t* wk, const uint32_t* ws, uint32_t L, float* out, uint32_t count,
                                hipStream_t s);
hipError_t launch_st_product(const float2* a, const float2* b, float r, float2* prod, const float2* z, float2* zz,
                             uint32_t N, hipStream_t s);
hipError_t launch_st_rows(float2* R, const Geom& g, const float2* base, float4 c, const float2* cols, uint32_t c0,
                          uint32_t nc, hipStream_t s);

}  // namespace pa

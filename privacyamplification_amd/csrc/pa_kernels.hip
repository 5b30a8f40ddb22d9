// pa_kernels.hip -- gfx950 kernels of the Toeplitz-hashing engine and their launchers.
//
// The reference evaluates amp_out with cuFFT/VkFFT and five small kernels, one synchronised
// launch each (binInt2float, calculateCorrectionFloat, setFirstElementToZero, ElementWiseProduct,
// ToBinaryArray; PrivacyAmplification.cu:363-813, mainloop 1819-2042).  Here the same arithmetic
// (FP32 FFT convolution, DC-zeroed spectra, round-mod-2 with the popcount correction) is fused
// into a few HBM passes:
//
//   k_transpose_bits  key/seed RefBits -> per-(class,column) bit masks for pass A
//   k_fwd_cols        pass A: decimated column FFTs of the +-1/2-encoded bits (R2C forward part);
//   k_mid_fwd         its form for L <= 2^24, straight from the key's and the seed's words, and
//   k_mix_fwd         for L = 3 * 2^k.  Their launches (the bit transpose's from 2^25 on) also scan
//                     the inputs' popcounts (binInt2float's popcount,
//                     PrivacyAmplification.cu:570-602) and prefix parities
//   k_rows            pass B: row FFTs, complex product (ElementWiseProduct, :465-481), inverse row FFTs
//   k_inv_cols        pass A': inverse column FFTs + round-mod-2 (ToBinaryArray :739-783)
//   k_pack            output word assembly with the mean's correction (calculateCorrectionFloat
//                     :363-373 and setFirstElementToZero :408-418 remove it spectrally), the key-rest
//                     XOR and byte order (key2StartRest's key_rest :873-878, ToBinaryArray's bswap
//                     XOR :757-762)
//   k_inv_big1, 2     pass A' for L >= 2^28
//   k_mid_inv         pass A' and the output in one for L <= 2^24, and
//   k_mix_inv         for L = 3 * 2^k
//   k_direct          short blocks without a transform
//   k_small           the whole block in one workgroup for L <= 2^14
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <type_traits>

#include "pa_device.hpp"
#include "pa_geom.hpp"
#include "pa_kernels.hpp"

namespace pa {

// ------------------------------------------------------------------ logical bit sources ----
// Word widx of the key sequence x: bits 0..h of the key (key2StartRest's key_start,
// PrivacyAmplification.cu:867-868: word h/32 keeps only its MSB), zero beyond.
__device__ __forceinline__ uint32_t key_word(const uint32_t* __restrict__ key, const Geom& g, uint32_t widx) {
    if (widx < g.key_hw) return key[widx];
    if (widx == g.key_hw) return key[widx] & 0x80000000u;
    return 0u;
}
// Word widx (< L/32) of the seed sequence t: the n seed bits rotated left by seed_rot words and
// repeated with period n up to the transform length L.  The
// output window only reads t[0, n), where the repetition changes nothing; beyond n it keeps the
// +-1/2-encoded sequence free of a constant block.  A zero pad there would become a -1/2 block
// whose convolution with the key's pad swings by about h/4 across positions, far beyond FP32's
// resolution at L = 2^24; the repeated seed leaves every position a random-walk sum of the same
// statistics.
__device__ __forceinline__ uint32_t seed_word(const uint32_t* __restrict__ seed, const Geom& g, uint32_t widx) {
    uint32_t s = widx + g.seed_rot;  // < 3 seed_words: L < 2n when L > n
    if (s >= g.seed_words) s -= g.seed_words;
    if (s >= g.seed_words) s -= g.seed_words;
    return seed[s];
}

// A resident seed's popcount, kept as POP_SLOTS partials.
__device__ __forceinline__ uint32_t pop_total(const uint32_t* __restrict__ c) {
    uint32_t t = 0;
#pragma unroll 8
    for (int i = 0; i < POP_SLOTS; ++i) t += c[i];
    return t;
}


// ------------------------------------------------------------------ staging copies ----
// One launch moves every staging range of a batch: workgroup (i, y) copies chunks y, y + grid.y,
// ... of COPY_CHUNK bytes of range d[i].  Host ranges are pinned, device-mapped memory that the
// kernel reads or writes over the bus, so a batch costs one launch instead of one DMA command
// per key, seed and output.  The descriptors themselves may live in mapped host memory.
constexpr uint32_t COPY_NT = 256;
constexpr uint64_t COPY_CHUNK = 64u * 1024u;
__global__ __launch_bounds__(COPY_NT) void k_copies(const CopyDesc* __restrict__ d) {
    const uint8_t* src = d[blockIdx.x].src;
    uint8_t* dst = d[blockIdx.x].dst;
    const uint64_t bytes = d[blockIdx.x].bytes;
    const uint64_t chunks = (bytes + COPY_CHUNK - 1) / COPY_CHUNK;
    const uint32_t al = (uint32_t)(((uintptr_t)src | (uintptr_t)dst) & 15u);
    for (uint64_t ch = blockIdx.y; ch < chunks; ch += gridDim.y) {
        const uint64_t lo = ch * COPY_CHUNK;
        const uint32_t len = (uint32_t)(bytes - lo < COPY_CHUNK ? bytes - lo : COPY_CHUNK);
        uint32_t body = 0;
        if (al == 0) {  // 16-byte words, four loads in flight per thread
            const uint4* s4 = reinterpret_cast<const uint4*>(src + lo);
            uint4* d4 = reinterpret_cast<uint4*>(dst + lo);
            const uint32_t n16 = len / 16;
            for (uint32_t i = threadIdx.x; i < n16; i += 4 * COPY_NT) {
                uint4 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (i + k * COPY_NT < n16) v[k] = s4[i + k * COPY_NT];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (i + k * COPY_NT < n16) d4[i + k * COPY_NT] = v[k];
            }
            body = n16 * 16;
        } else if ((al & 3u) == 0) {
            const uint32_t* s1 = reinterpret_cast<const uint32_t*>(src + lo);
            uint32_t* d1 = reinterpret_cast<uint32_t*>(dst + lo);
            const uint32_t n4 = len / 4;
            for (uint32_t i = threadIdx.x; i < n4; i += COPY_NT) d1[i] = s1[i];
            body = n4 * 4;
        }
        for (uint32_t i = body + threadIdx.x; i < len; i += COPY_NT) dst[lo + i] = src[lo + i];
    }
}

// ------------------------------------------------------------------ mean correction ----
// The conv value of the +-1/2-encoded sequences differs from the integer it stands for by the
// prefix sums of both bit sequences (see pa_geom.hpp); mod 2 only their parities matter.  A scan
// workgroup takes one chunk of 1024 << g.scan words: inclusive prefix parities of x ^ t inside the
// chunk go to q (bit p of word w: the parity of the chunk's bits up to there; only words up to the
// end of the output window), the chunk's parity to its byte of cp, its popcount (key + seed) to its
// entry; for the mid sizes also the XOR of its seed words per word of the whitening's period (the bit
// transpose has the others').  x is the whitened key.  A resident seed brings its own finished prefix
// words sq; x alone is scanned then.  The scan workgroups ride in the bit transpose's launch (in pass A's for the
// mid sizes); scan_finish, in pass B's, turns the entries into what pass A' and the output stage read.
// (In pass A's launch at 2^27 they cost 15 us: with its 74 KB of LDS only two fit a compute unit.)
__device__ __forceinline__ uint32_t prefix_bits(uint32_t w) {  // bit p: parity of bits 0..p, MSB first
    w ^= w >> 1;
    w ^= w >> 2;
    w ^= w >> 4;
    w ^= w >> 8;
    return w ^ (w >> 16);
}
// NT threads; lds: 2 NT (2 + 128) / 64 words at most.  key == nullptr scans the seed alone.  Per 1024 words a wave takes 64 PER
// consecutive ones, 64 at a time: coalesced, the carry between lanes from a ballot.
template <int NT>
__device__ __forceinline__ void scan_chunk(uint32_t chunk, const ScanArgs& a, const Geom& g, uint32_t* lds) {
    constexpr uint32_t PER = 1024 / NT;
    static_assert(PER * NT == 1024 && NT % 64 == 0, "a thread takes whole words");
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t before = (1ull << lane) - 1ull;
    const uint32_t w_end = (g.out_off + g.out_bits) >> 5;
    uint32_t pops = 0, chunk_par = 0, fold[2] = {0, 0};  // fold: words of lane and 64 + lane mod 128
    for (uint32_t sub = 0; sub < (1u << g.scan); ++sub) {
        const uint32_t w0 = ((chunk << g.scan) + sub) * 1024u + 64u * PER * wave + lane;
        uint32_t w[PER], sw[PER], run = 0;
        // no load is conditional on a lane, so that all are in flight together
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t wi = w0 + 64u * i;
            w[i] = a.key ? a.key[wi < g.key_hw ? wi : g.key_hw] : 0u;
            sw[i] = a.seed ? seed_word(a.seed, g, wi) : 0u;
        }
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t wi = w0 + 64u * i;
            if (a.key) w[i] = (w[i] & (wi < g.key_hw ? ~0u : wi == g.key_hw ? 0x80000000u : 0u)) ^ white_word(g, wi);
            pops += (uint32_t)(__popc(w[i]) + __popc(sw[i]));
            fold[i & 1] ^= sw[i];
            w[i] ^= sw[i];
        }
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            w[i] = prefix_bits(w[i]);
            const uint64_t b = __ballot((w[i] & 1u) != 0u);
            w[i] ^= 0u - ((run + (uint32_t)__popcll(b & before)) & 1u);
            run += (uint32_t)__popcll(b);
        }
        uint32_t carry = chunk_par;
        if (sub) __syncthreads();  // the previous round's reads of lds are done
        if (lane == 0) lds[wave] = run;
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < NT / 64; ++k) {
            const uint32_t t = lds[k];
            if (k < wave) carry += t;
            chunk_par += t;
        }
        chunk_par &= 1u;
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t wi = w0 + 64u * i;
            if (wi < w_end) a.q[wi] = w[i] ^ (0u - (carry & 1u)) ^ (a.sq ? a.sq[wi] : 0u);
        }
    }
    for (int off = 32; off > 0; off >>= 1) pops += __shfl_xor(pops, off);
    if (lane == 0) lds[NT / 64 + wave] = pops;
    const bool folds = a.seed && g.white == WHITE_MID;
    uint32_t* lf = lds + 2 * (NT / 64);
    if (folds) {
        lf[128u * wave + lane] = fold[0];
        lf[128u * wave + 64u + lane] = fold[1];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        pops = 0;
        for (int k = 0; k < NT / 64; ++k) pops += lds[NT / 64 + k];
        a.info[info_pops(g) + chunk] = pops;
        scan_parities(a.info)[chunk] = (uint8_t)chunk_par;
    }
    if (folds)
        for (uint32_t c = threadIdx.x; c < WHITE_MID; c += NT) {
            uint32_t x = 0;
            for (int k = 0; k < NT / 64; ++k) x ^= lf[128u * k + c];
            a.info[info_fold(g) + chunk * WHITE_MID + c] = x;
        }
}
// In-place inclusive prefix parities of the `n` words at a (bit p of word w: of all bits up to there),
// n / NT consecutive words a thread (one for the first n threads where n < NT); returns the parity of all.
// part: NT / 64 words.  Ends with a barrier.
template <int NT>
__device__ __forceinline__ uint32_t prefix_words_lds(uint32_t* a, uint32_t n, uint32_t* part) {
    const uint32_t per = n < (uint32_t)NT ? 1u : n / NT, i0 = threadIdx.x * per;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const bool mine = i0 < n;
    uint32_t par = 0;
    if (mine)
        for (uint32_t i = i0; i < i0 + per; ++i) {
            const uint32_t w = prefix_bits(a[i]);
            a[i] = w ^ (0u - par);
            par ^= w & 1u;
        }
    const uint64_t b = __ballot(par != 0u);
    if (lane == 0) part[wave] = (uint32_t)__popcll(b);
    __syncthreads();
    uint32_t carry = (uint32_t)__popcll(b & ((1ull << lane) - 1ull)), total = 0;
    for (uint32_t k = 0; k < NT / 64; ++k) {
        const uint32_t t = part[k];
        if (k < wave) carry += t;
        total += t;
    }
    if (mine && (carry & 1u))
        for (uint32_t i = i0; i < i0 + per; ++i) a[i] = ~a[i];
    __syncthreads();
    return total & 1u;
}
// One level of conv(R, t): word w (< b c) of conv(s[(. / b) mod c], t) from the prefix words p of t folded to
// that period, tau the parity of t.  The words of one sign are a window of t, the difference of two
// prefixes b words apart, so that the sum has a prefix for each change of sign.
template <uint32_t b, uint32_t c, uint32_t s>
__device__ __forceinline__ uint32_t white_level(const uint32_t* p, uint32_t w, uint32_t tau) {
    uint32_t x = 0u - ((s >> (w / b)) & tau & 1u);
    uint32_t d = s ^ ((s << 1) | (s >> (c - 1u)));
#pragma unroll
    for (uint32_t i = 0; i < c; ++i, d >>= 1)
        if (d & 1u) x ^= p[(w - b * i) & (b * c - 1u)];
    return x;
}
// conv(R, t), g.white words, from the fold slices of t (pa_geom.hpp).  One workgroup; the slices (16 KB each
// from 2^25 bits on, 512 bytes below) are 0.5 to 1 MB and 512 bytes a chunk, read while the other
// workgroups of pass B transform.  lds: 16 + 4 NT + 144 words, or 16 + 4096 + 272 + 272.
template <int NT>
__device__ __forceinline__ void white_table(uint32_t* out, const uint4* fold, const Geom& g, uint32_t* lds) {
    uint32_t* a2 = lds + 16;
    const bool big = g.white == WHITE_BIG;
    const uint32_t vecs = g.white / 4u, total = fold_slices(g) * vecs;  // 16-byte entries
    const uint32_t runs = big ? vecs / NT : 1u;  // a thread's entries are of one class, of `runs` in turn
    for (uint32_t c = 0; c < runs; ++c) {
        uint4 x = make_uint4(0u, 0u, 0u, 0u);
        const uint32_t step = big ? vecs : (uint32_t)NT;
        for (uint32_t e0 = threadIdx.x + NT * c; e0 < total; e0 += 16u * step) {
            uint4 y[16];  // requested together
#pragma unroll
            for (uint32_t k = 0; k < 16; ++k) {
                const uint32_t e = e0 + k * step;
                y[k] = fold[e < total ? e : e0];
                if (e >= total) y[k] = make_uint4(0u, 0u, 0u, 0u);
            }
#pragma unroll
            for (uint32_t k = 0; k < 16; ++k) {
                x.x ^= y[k].x;
                x.y ^= y[k].y;
                x.z ^= y[k].z;
                x.w ^= y[k].w;
            }
        }
        uint32_t* v = a2 + 4u * (threadIdx.x + NT * c);
        v[0] = x.x;
        v[1] = x.y;
        v[2] = x.z;
        v[3] = x.w;
    }
    __syncthreads();
    if (big) {
        uint32_t *a1 = a2 + 4096, *a0 = a1 + 256, *o1 = a0 + 16, *o0 = o1 + 256;
        for (uint32_t w = threadIdx.x; w < 256u; w += NT) {
            uint32_t x = 0;
            for (uint32_t i = 0; i < 16u; ++i) x ^= a2[w + 256u * i];
            a1[w] = x;
        }
        __syncthreads();
        if (threadIdx.x < 16u) {
            uint32_t x = 0;
            for (uint32_t i = 0; i < 16u; ++i) x ^= a1[threadIdx.x + 16u * i];
            a0[threadIdx.x] = x;
        }
        __syncthreads();
        prefix_words_lds<NT>(a0, 16u, lds);
        prefix_words_lds<NT>(a1, 256u, lds);
        const uint32_t tau = prefix_words_lds<NT>(a2, 4096u, lds);
        if (threadIdx.x < 16u) o0[threadIdx.x] = white_level<1, 16, WHITE_S0>(a0, threadIdx.x, tau);
        for (uint32_t w = threadIdx.x; w < 256u; w += NT) o1[w] = white_level<16, 16, WHITE_S1>(a1, w, tau);
        __syncthreads();
        for (uint32_t w = threadIdx.x; w < 4096u; w += NT)
            out[w] = o0[w & 15u] ^ o1[w & 255u] ^ white_level<256, 16, WHITE_S2>(a2, w, tau);
    } else {
        // thread t has the words 4 t mod 128 on, so thread t + 32 k those of thread t too
        uint32_t *a1 = a2 + 4 * NT, *a0 = a1 + 128;
        for (uint32_t w = threadIdx.x; w < 128u; w += NT) {
            uint32_t x = 0;
            for (uint32_t k = 0; k < NT / 32u; ++k) x ^= a2[128u * k + w];
            a1[w] = x;
        }
        __syncthreads();
        if (threadIdx.x < 16u) {
            uint32_t x = 0;
            for (uint32_t i = 0; i < 8u; ++i) x ^= a1[threadIdx.x + 16u * i];
            a0[threadIdx.x] = x;
        }
        __syncthreads();
        prefix_words_lds<NT>(a0, 16u, lds);
        const uint32_t tau = prefix_words_lds<NT>(a1, 128u, lds);
        for (uint32_t w = threadIdx.x; w < 128u; w += NT)
            out[w] = white_level<1, 16, WHITE_MID_S0>(a0, w & 15u, tau) ^ white_level<16, 8, WHITE_MID_S1>(a1, w, tau);
    }
}
// One workgroup of NT threads: info[INFO_POPS] = both popcounts, conv(R, t) (RESIDENT: from ws, a resident
// seed's popcount partials and behind them its conv(R, t)), and the chunks' parities become their exclusive prefix.
// lds: as white_table.
// seed_ws != nullptr (resident seed being prepared): it receives what ws holds.
template <int NT, bool RESIDENT>
__device__ __forceinline__ void scan_finish(uint32_t* info, const Geom& g, const uint32_t* ws, uint32_t* seed_ws,
                                            uint32_t* lds) {
    const uint32_t count = scan_chunks(g), per = (count + NT - 1) / NT, i0 = threadIdx.x * per;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint8_t* cp = scan_parities(info);
    uint32_t par = 0, pops = 0;
#pragma unroll 4
    for (uint32_t i = i0; i < i0 + per && i < count; ++i) {
        par ^= cp[i];
        pops += info[info_pops(g) + i];
    }
    for (int off = 32; off > 0; off >>= 1) pops += __shfl_xor(pops, off);
    const uint64_t b = __ballot(par != 0u);
    uint32_t carry = (uint32_t)__popcll(b & ((1ull << lane) - 1ull));
    if (lane == 0) {
        lds[wave] = (uint32_t)__popcll(b);
        lds[NT / 64 + wave] = pops;
    }
    __syncthreads();
    for (uint32_t i = 0; i < wave; ++i) carry += lds[i];
    carry &= 1u;
    for (uint32_t i = i0; i < i0 + per && i < count; ++i) {
        const uint32_t c = cp[i];
        cp[i] = (uint8_t)carry;
        carry ^= c;
    }
    if (wave == 0) {
        pops = 0;
        for (int i = 0; i < NT / 64; ++i) pops += lds[NT / 64 + i];
        if (lane == 0) info[INFO_POPS] = pops + (ws ? pop_total(ws) : 0u);
        if (seed_ws) seed_ws[lane] = lane == 0 ? pops : 0u;
    }
    uint32_t* white = info + info_white(g);
    if constexpr (RESIDENT) {
        const uint4* src = reinterpret_cast<const uint4*>(ws + POP_SLOTS);
        for (uint32_t i = threadIdx.x; i < g.white / 4u; i += NT) reinterpret_cast<uint4*>(white)[i] = src[i];
    } else {
        __syncthreads();  // lds
        white_table<NT>(seed_ws ? seed_ws + POP_SLOTS : white, reinterpret_cast<const uint4*>(info + info_fold(g)), g, lds);
    }
}
// A resident seed's prefix words once their chunks' exclusive parities are known (pa_seed_put).
__global__ __launch_bounds__(256) void k_prefix_apply(uint32_t* __restrict__ q, const uint32_t* __restrict__ info,
                                                      Geom g) {
    const uint32_t w = blockIdx.x * 256u + threadIdx.x;
    if (scan_parities(info)[w >> (10u + g.scan)]) q[w] = ~q[w];
}

// ------------------------------------------------------------------ bit transpose ----
// One round of the recursive 32 x 32 bit-matrix transpose (rows A[k], column 0 = the MSB): swap
// the off-diagonal J x J blocks of every 2J x 2J block.  Five rounds J = 16, 8, 4, 2, 1 transpose.
template <int J>
__device__ __forceinline__ void bit_transpose_round(uint32_t (&A)[32]) {
    constexpr uint32_t M = J == 16 ? 0x0000FFFFu : J == 8 ? 0x00FF00FFu : J == 4 ? 0x0F0F0F0Fu
                         : J == 2 ? 0x33333333u : 0x55555555u;
#pragma unroll
    for (int b = 0; b < 32; b += 2 * J)
#pragma unroll
        for (int r = 0; r < J; ++r) {
            const uint32_t t = (A[b + r] ^ (A[b + r + J] >> J)) & M;
            A[b + r] ^= t;
            A[b + r + J] ^= t << J;
        }
}

__device__ __forceinline__ void bit_transpose(uint32_t (&A)[32]) {
    bit_transpose_round<16>(A);
    bit_transpose_round<8>(A);
    bit_transpose_round<4>(A);
    bit_transpose_round<2>(A);
    bit_transpose_round<1>(A);
}

// tb[u*N2 + t2] has x[t2 + N2(u + M v)] and x[N + t2 + N2(u + M v)] at bits mask_bit(D, 0, v) and
// mask_bit(D, 1, v) (D = 32: the second half's in the word tb[(M + u) N2 + t2]).
// Workgroup (u, part): thread k covers t2 in [part*TB_SPAN + 32k, +32): for each class v it reads
// the two words holding those bits (coalesced across the workgroup), transposes the 2 D x 32 bits
// in registers, and the workgroup writes its TB_SPAN outputs through LDS.  The launch's first
// `scan_wgs` workgroups scan the inputs, the next ones are operand `first` (0 key, 1 seed), then the
// next operand.
// Batched launches (BATCH = true) take each block's geometry and buffers from bt[blockIdx.z].
template <int D, bool BATCH>
__global__ __launch_bounds__(TB_NT) void k_transpose_bits(const uint32_t* __restrict__ key,
                                                          const uint32_t* __restrict__ seed,
                                                          uint32_t* __restrict__ tbk, uint32_t* __restrict__ tbs,
                                                          uint32_t first, Geom g, ScanArgs scan, uint32_t scan_wgs,
                                                          const BlockArgs* __restrict__ bt) {
    __shared__ uint32_t stage[TB_NT * 33];
    if constexpr (BATCH) {
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        key = a.key;
        seed = a.seed;
        tbk = a.tbk;
        tbs = a.tbs;
        scan = ScanArgs{a.key, a.seed, a.sq, a.q, a.info};
    }
    if (blockIdx.x < scan_wgs) {
        scan_chunk<TB_NT>(blockIdx.x, scan, g, stage);
        return;
    }
    constexpr int PARTS_LOG = ROW_LOG - TB_SPAN_LOG;
    uint32_t b = blockIdx.x - scan_wgs;
    const uint32_t nA = g.M << PARTS_LOG;
    const bool is_seed = first + b / nA == 1u;
    const uint32_t* __restrict__ bits = is_seed ? seed : key;
    uint32_t* __restrict__ tb = is_seed ? tbs : tbk;
    if (BATCH && bits == nullptr) return;  // resident seed: nothing to transpose
    b %= nA;
    const uint32_t u = b >> PARTS_LOG, part = b & ((1u << PARTS_LOG) - 1u);
    const uint32_t t0 = (part << TB_SPAN_LOG) + 32u * threadIdx.x;
    uint32_t w0[D], w1[D];
    // M rows and N positions are whole periods of the whitening: one word of it for all
    const uint32_t white = is_seed ? 0u : white_word(g, (t0 + g.N2 * u) >> 5);
    uint32_t fold = 0;
#pragma unroll
    for (int v = 0; v < D; ++v) {
        const uint32_t widx = (t0 + g.N2 * (u + g.M * (uint32_t)v)) >> 5;
        w0[v] = is_seed ? seed_word(bits, g, widx) : key_word(bits, g, widx) ^ white;
        w1[v] = is_seed ? seed_word(bits, g, widx + (g.N >> 5)) : key_word(bits, g, widx + (g.N >> 5)) ^ white;
        fold ^= w0[v] ^ w1[v];
    }
    if (is_seed) scan.info[info_fold(g) + ((t0 + g.N2 * u) >> 5)] = fold;
    uint32_t* srow = stage + threadIdx.x * 33;
    uint32_t* out = tb + (size_t)u * g.N2 + (part << TB_SPAN_LOG);
    // Row A[31 - i] = the words of bit i, transposed: A[c] then holds bit 31 - c (column t0 + c) of
    // each at its place.
    constexpr int NW = D == 32 ? 2 : 1;
#pragma unroll
    for (int k = 0; k < NW; ++k) {
        uint32_t A[32] = {};
#pragma unroll
        for (int v = 0; v < D; ++v) {
            A[31 - mask_bit(D, k, v)] = k ? w1[v] : w0[v];
            if constexpr (NW == 1) A[31 - mask_bit(D, 1, v)] = w1[v];
        }
        bit_transpose(A);
        if (k) __syncthreads();  // the first half has been written out
#pragma unroll
        for (int i = 0; i < 32; ++i) srow[i] = A[i];
        __syncthreads();
        for (int e = threadIdx.x; e < (1 << TB_SPAN_LOG); e += TB_NT) out[e] = stage[(e >> 5) * 33 + (e & 31)];
        out += (size_t)g.M * g.N2;
    }
}

// ------------------------------------------------------------------ pass A ----
// One launch serves `ops` operands from `first` on (0 key, 1 seed), nA workgroups each (k_mid_fwd: and
// then the scan workgroups).  Where a block is one of a batch, its arguments come from the table.
struct FwdArgs {
    const uint32_t* in[2];  // bit masks (k_mid_fwd: the words themselves) of key and seed
    float2* Y[2];
    uint32_t first, ops, nA;
    ScanArgs scan;
};
template <bool BATCH, bool WORDS>
__device__ __forceinline__ void fwd_batch_args(FwdArgs& a, Geom& g, const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) {
        const BlockArgs& b = bt[blockIdx.z];
        g = b.g;
        a.in[0] = WORDS ? b.key : b.tbk;
        a.in[1] = WORDS ? b.seed : b.tbs;
        a.Y[0] = b.Yk;
        a.Y[1] = b.Ys;
        a.scan = ScanArgs{b.key, b.seed, b.sq, b.q, b.info};
    }
}
// w_4N1^x from the 2^14 table while 4 N1 <= 2^14, else from the two-level table of w_2L (2L = 4 N1 N2).
__device__ __forceinline__ float2 w_4n1(const Geom& g, const float2* __restrict__ tw14, const float2* __restrict__ twlo,
                                        const float2* __restrict__ twhi, uint32_t x) {
    if (4u * g.N1 <= (uint32_t)TW14) return tw14[x * (TW14 / (4u * g.N1))];
    return tw_two_level(twlo, twhi, x * g.N2);
}
__device__ __forceinline__ float2 uniform_f2(float2 v) {
    return make_float2(__uint_as_float(__builtin_amdgcn_readfirstlane((int)__float_as_uint(v.x))),
                       __uint_as_float(__builtin_amdgcn_readfirstlane((int)__float_as_uint(v.y))));
}

// Raw buffer access (vector memory instructions): one per-lane byte offset plus a uniform
// scalar offset, so a run of accesses at fixed strides keeps a single address register.
typedef unsigned int pa_u2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
template <int AUX>
__device__ __forceinline__ void buf_store(float2 v, __amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    const pa_u2v x = {__float_as_uint(v.x), __float_as_uint(v.y)};
    __builtin_amdgcn_raw_buffer_store_b64(x, rs, (int)voff, (int)soff, AUX);  // aux 2: nt
}
__device__ __forceinline__ void buf_store_nt(float2 v, __amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    buf_store<2>(v, rs, voff, soff);
}
__device__ __forceinline__ float2 buf_load_f2(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    const pa_u2v x = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)voff, (int)soff, 0);
    return make_float2(__uint_as_float(x.x), __uint_as_float(x.y));
}
__device__ __forceinline__ uint32_t buf_load_u32(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b32(rs, (int)voff, (int)soff, 0);
}

// Pass A for L >= 2^25: a workgroup has 16 columns (group grp) and a pair of classes of the D, c = p
// and p + D/2, and computes Y[k1][t2] for k1 = c + D k1', at the quarter-shifted frequencies k1 + 1/4
// (c' = c + 1/4):
//   Y = w_N^{t2 (k1 + 1/4)} * FFT_M( w_N1^{u c'} * sum_v z[t2 + N2(u + M v)] w_D^{v c'} ),
// z[t] = a[t] - i a[t + N], a = bit - 1/2.  The sums over the even and the odd v are table lookups by
// the mask's bits (the -1/2 included) and serve both classes: their sum and their difference.
// Plan R1 x 32 with M = 32 R1: M = 512 for N1 <= 2^13 (256 threads, two workgroups per compute unit),
// M = 1024 for 2^14 and 2^15 (512 threads, one: its 16 columns take 135 KB of LDS).
template <int LGM, int D>
struct FwdPlan {
    static constexpr int M = 1 << LGM, R1 = M / 32, NT = fwd_cols_threads(LGM), JT = NT / 16, K1 = 32 / JT;
    static constexpr int NW = D == 32 ? 2 : 1;   // mask words per position (both halves in one up to D = 16)
    static constexpr int BW = cls_bits(D), NB = cls_tables(D);  // index bits of a table, tables of a pair
    static constexpr int SEQS = seq_stride(M);
    static_assert(JT == R1, "one second-stage butterfly per thread");
    using Bits = uint32_t[K1][R1][NW];
    using Sums = float2[K1][R1];
    using Tables = float2[NB][1 << BW];
};
// Pieces of the persistent walk.  Thread (col = t mod 16, jt = t / 16).
// Bit words of column group grp: stage-1 butterflies j = jt + JT i, inputs u = j + 32 r.
template <int LGM, int D>
__device__ __forceinline__ void fwd_load_bits(typename FwdPlan<LGM, D>::Bits& tv, __amdgpu_buffer_rsrc_t rtb, uint32_t N2,
                                              uint32_t t2, int jt) {
    using P = FwdPlan<LGM, D>;
#pragma unroll
    for (int i = 0; i < P::K1; ++i) {
        const uint32_t voff = ((uint32_t)(jt + P::JT * i) * N2 + t2) * 4u;
#pragma unroll
        for (int r = 0; r < P::R1; ++r)
#pragma unroll
            for (int h = 0; h < P::NW; ++h)
                tv[i][r][h] = buf_load_u32(rtb, voff, (uint32_t)(32 * r + P::M * h) * N2 * 4u);
    }
}
// Class sums of p (a) and p + D/2 (d).
template <int LGM, int D>
__device__ __forceinline__ void fwd_sums(typename FwdPlan<LGM, D>::Sums& a, typename FwdPlan<LGM, D>::Sums& d,
                                         const typename FwdPlan<LGM, D>::Bits& tv,
                                         const typename FwdPlan<LGM, D>::Tables& TB) {
    using P = FwdPlan<LGM, D>;
    constexpr uint32_t MASK = (1u << P::BW) - 1u;
#pragma unroll
    for (int i = 0; i < P::K1; ++i)
#pragma unroll
        for (int r = 0; r < P::R1; ++r) {
            const uint32_t w0 = tv[i][r][0], w1 = P::NW == 2 ? tv[i][r][P::NW - 1] : w0 >> 16;
            float2 s[2];
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                if constexpr (D <= 8) {
                    s[o] = TB[o][(w0 >> (D * o)) & MASK];
                } else {
                    constexpr int H = P::NB / 2;
                    float2 e = TB[H * o][(w0 >> (8 * H * o)) & MASK], f = TB[H * o][(w1 >> (8 * H * o)) & MASK];
#pragma unroll
                    for (int q = 1; q < H; ++q) {
                        e = cadd(e, TB[H * o + q][(w0 >> (8 * (H * o + q))) & MASK]);
                        f = cadd(f, TB[H * o + q][(w1 >> (8 * (H * o + q))) & MASK]);
                    }
                    s[o] = make_float2(e.x + f.y, e.y - f.x);
                }
            }
            a[i][r] = cadd(s[0], s[1]);
            d[i][r] = csub(s[0], s[1]);
        }
}
// Table entries of the output twiddles w_2L^{t2 (4 k1 + 1)}, k1 = c + D (jt + R1 r) = base step^r, with
// anchors w_N^{t2 R1 D 8 (a+1)}: (lo, hi) pairs of the base for c = p, step, anchor 0..2 and the base for
// p + D/2.  The products are formed where they are used, so that gathering them never waits on other
// loads.
template <int LGM, int D>
__device__ __forceinline__ void fwd_load_tw(float2 (&tw)[12], const float2* __restrict__ lo,
                                            const float2* __restrict__ hi, uint32_t L, uint32_t p, uint32_t t2, int jt) {
    constexpr uint32_t R1 = FwdPlan<LGM, D>::R1;
    const uint32_t L2m = 2u * L - 1u;
    uint32_t x[6];
    x[0] = (t2 * (4u * (p + (uint32_t)D * (uint32_t)jt) + 1u)) & L2m;
    x[1] = (t2 * (4u * R1 * (uint32_t)D)) & L2m;
#pragma unroll
    for (int a = 0; a < 3; ++a) x[2 + a] = (t2 * (4u * R1 * (uint32_t)D * 8u * (uint32_t)(a + 1))) & L2m;
    x[5] = (x[0] + t2 * (2u * (uint32_t)D)) & L2m;
#pragma unroll
    for (int e = 0; e < 6; ++e) {
        tw[2 * e] = lo[x[e] & (TW14 - 1)];
        tw[2 * e + 1] = hi[x[e] >> TW14_LOG];
    }
}
// tw1: the first stage's factors for w_N1^{32 c'} (one class pair per workgroup: uniform).
template <int LGM, int D>
__device__ __forceinline__ void fwd_stage1(typename FwdPlan<LGM, D>::Sums& v, float2* seqbuf,
                                           const float2 (&tw1)[FwdPlan<LGM, D>::R1 / 2], int jt) {
    using P = FwdPlan<LGM, D>;
#pragma unroll
    for (int i = 0; i < P::K1; ++i) {
        dft_tw<P::R1>(v[i], tw1);
#pragma unroll
        for (int r = 0; r < P::R1; ++r) seqbuf[padi((jt + P::JT * i) * P::R1 + r)] = v[i][r];
    }
}
// tw2: the second stage's factors, row jt for w_M^jt w_N1^c' (the class twiddle of input j).
template <int LGM, int D>
__device__ __forceinline__ void fwd_stage2(const float2* seqbuf, const float2* tw2, const float2 base,
                                           const float2 (&tw)[12], __amdgpu_buffer_rsrc_t ry, uint32_t N2, uint32_t c,
                                           uint32_t t2, int jt) {
    using P = FwdPlan<LGM, D>;
    float2 F[32];
    stage_last_from_lds_tab<32, P::M>(F, seqbuf, jt, tw2 + jt * stage_row<32>());
    const float2 step = cmul(tw[2], tw[3]);
    const uint32_t voff = ((c + (uint32_t)D * (uint32_t)jt) * N2 + t2) * 8u;
    float2 w = base;
#pragma unroll
    for (int r = 0; r < 32; ++r) {
        if ((r & 7) == 0 && r) w = cmul(base, cmul(tw[2 * (1 + r / 8)], tw[2 * (1 + r / 8) + 1]));
        buf_store_nt(cmul(F[r], w), ry, voff, (uint32_t)(P::R1 * D * r) * N2 * 8u);
        w = cmul(w, step);
    }
}

// Persistent: workgroup L of G keeps one class pair p = L mod D/2 and walks the column groups
// [k per, k per + per), k = L / (D/2), so its tables are loaded once, and each group's stores drain
// while the next group is transformed (its loads were issued before those stores).  The workgroups
// of one k sit on one XCD and walk the same groups in step, so each bit word is fetched into L2 once.
// The class twiddles w_N1^{u c'}, u = j + 32 r, cost nothing: their r part is in the first stage's
// factors, their j part in the second's.
// Both operands at 2^27: 0.277 ms (one class per workgroup: 0.32), of which storing the 1.07 GB in this
// order alone takes 0.237; at 2^29 1.54 ms (2.23), storing alone 0.84, the rest the lookups, 4 a value.
template <int LGM, int D, bool BATCH>
__global__ __launch_bounds__(fwd_cols_threads(LGM), LGM == 9 ? 2 : 1) void k_fwd_cols(
    FwdArgs a, Geom g, const float2* __restrict__ tw14, const float2* __restrict__ twlo, const float2* __restrict__ twhi,
    const float2* __restrict__ cls, uint32_t per, const BlockArgs* __restrict__ bt) {
    fwd_batch_args<BATCH, false>(a, g, bt);
    using P = FwdPlan<LGM, D>;
    constexpr int NT = P::NT, TW2 = P::R1 * stage_row<32>(), R1H = P::R1 / 2;
    constexpr uint32_t MASK = (1u << P::BW) - 1u;
    __shared__ float2 buf[16 * P::SEQS];
    __shared__ float2 tw2[2 * TW2];
    __shared__ float2 tw1s[2 * R1H];
    __shared__ typename P::Tables TB;
    const uint32_t op = blockIdx.x / a.nA;
    const bool is_seed = a.first + op == 1u;
    const uint32_t* __restrict__ tb = is_seed ? a.in[1] : a.in[0];
    float2* __restrict__ Y = is_seed ? a.Y[1] : a.Y[0];
    if (BATCH && tb == nullptr) return;  // resident seed: nothing to transform
    const uint32_t logical = xcd_logical(blockIdx.x - op * a.nA, a.nA);
    const uint32_t p = logical % (D / 2), grp0 = (logical / (D / 2)) * per, N2 = g.N2;
    const __amdgpu_buffer_rsrc_t rtb = make_rsrc(tb, (uint32_t)(P::M * P::NW) * N2 * 4u);
    const __amdgpu_buffer_rsrc_t ry = make_rsrc(Y, g.N1 * N2 * 8u);
    {
        const float2* src = cls + cls_table_offset(D) + (size_t)p * (P::NB << P::BW);
        for (int e = threadIdx.x; e < P::NB << P::BW; e += NT) TB[e >> P::BW][e & (int)MASK] = src[e];
    }
    const uint32_t m4 = 4u * g.N1 - 1u;  // exponents of w_4N1
    {
        static_assert(P::R1 * 16 == NT, "one factor per thread");
        const uint32_t q = threadIdx.x >> 4, i = threadIdx.x & 15u;
        uint32_t s = 2;  // the size of factor i and its index k at that size (dft_tw's order)
        while (s / 2u <= i && i > 0u) s *= 2u;
        const uint32_t k = i ? i - s / 4u : 0u;
#pragma unroll
        for (uint32_t o = 0; o < 2; ++o) {
            const uint32_t f = 4u * (p + o * (D / 2)) + 1u;
            tw2[o * TW2 + q * stage_row<32>() + i] =
                w_4n1(g, tw14, twlo, twhi, ((32u / s) * (4u * (uint32_t)D * q + f) + k * (4u * g.N1 / s)) & m4);
            if (q == 0 && i < (uint32_t)R1H)
                tw1s[o * R1H + i] = w_4n1(g, tw14, twlo, twhi, ((P::R1 / s) * 32u * f + k * (4u * g.N1 / s)) & m4);
        }
    }
    const int col = threadIdx.x & 15, jt = threadIdx.x >> 4;
    float2* seqbuf = buf + col * P::SEQS;
    typename P::Bits tv;
    float2 tw[12], twn[12];
    uint32_t t2 = grp0 * 16u + (uint32_t)col;
    fwd_load_bits<LGM, D>(tv, rtb, N2, t2, jt);
    fwd_load_tw<LGM, D>(tw, twlo, twhi, g.L, p, t2, jt);
    __syncthreads();  // tables
    // The first stage's factors: in scalar registers where they fit, else read again for each use.
    float2 f0[R1H], f1[R1H];
    auto factors = [&](float2 (&f)[R1H], int o) {
#pragma unroll
        for (int i = 0; i < R1H; ++i) f[i] = tw1s[o * R1H + i];
    };
    if constexpr (P::R1 <= 16) {
        factors(f0, 0);
        factors(f1, 1);
#pragma unroll
        for (int i = 0; i < R1H; ++i) {
            f0[i] = uniform_f2(f0[i]);
            f1[i] = uniform_f2(f1[i]);
        }
    }
    typename P::Sums va, vd;
    // One column group; more: the next one's loads are issued before its last stores.
    auto group = [&](bool more) {
        fwd_sums<LGM, D>(va, vd, tv, TB);
        if constexpr (P::R1 > 16) factors(f0, 0);
        fwd_stage1<LGM, D>(va, seqbuf, f0, jt);
        __syncthreads();
        fwd_stage2<LGM, D>(seqbuf, tw2, cmul(tw[0], tw[1]), tw, ry, N2, p, t2, jt);
        __syncthreads();
        if constexpr (P::R1 > 16) factors(f1, 1);
        fwd_stage1<LGM, D>(vd, seqbuf, f1, jt);
        __syncthreads();
        if (more) {
            fwd_load_bits<LGM, D>(tv, rtb, N2, t2 + 16u, jt);
            fwd_load_tw<LGM, D>(twn, twlo, twhi, g.L, p, t2 + 16u, jt);
        }
        fwd_stage2<LGM, D>(seqbuf, tw2 + TW2, cmul(tw[10], tw[11]), tw, ry, N2, p + D / 2, t2, jt);
    };
    // The first group is peeled: every entry into the loop then has the same memory-operation
    // history (next group's loads, then this group's stores), so the compiler's waits on the
    // prefetched registers count past the stores instead of draining them.
    group(per > 1);
    for (uint32_t it = 1; it < per; ++it) {
        t2 += 16u;
#pragma unroll
        for (int e = 0; e < 12; ++e) tw[e] = twn[e];
        __syncthreads();  // second-stage reads of the previous group are done
        group(it + 1 < per);
    }
}

// Pass A for L <= 2^24 (N1 = 2^6 .. 2^10), straight from the key's and the seed's words: the 16 columns
// of a group are half a word of every row, so no bit transpose is needed.  Plan R1 x 16 (R1 x 32 from
// 512 on): the quarter shift sits in the stages' factors.
// WALK: a workgroup takes `per` (even) consecutive groups, a pair of them from each word, and requests the
// next pair's words and the next group's twiddles while it transforms; one group per workgroup
// otherwise, for launches that leave compute units idle as it is.
// Loading a group's bits (2 used bytes of each line) and its twiddles took 130 of the 387 us of 2^27
// bits in blocks of 2^20 when every group was a workgroup of its own; now 328, of which storing the
// 1.07 GB alone takes 202.  2^22: 440 to 380; 2^24: 490 to 334.
template <int LG1>
struct MidPlan {
    static constexpr int N1 = 1 << LG1, NT = mid_threads(LG1), R1 = mid_r1(LG1), R2 = N1 / R1, S1 = N1 / R1;
    static constexpr int K1 = 16 * S1 / NT, SEQS = seq_stride(N1), RPT = N1 / NT;
    static_assert(16 * R1 == NT && K1 * R1 == R2, "one second-stage butterfly per thread");
    static_assert(RPT * NT == N1, "a thread loads whole rows' words");
};
template <int LG1, bool BATCH, bool WALK>
__global__ __launch_bounds__(mid_threads(LG1)) void k_mid_fwd(FwdArgs a, Geom g, const float2* __restrict__ tw14,
                                                              const float2* __restrict__ twlo,
                                                              const float2* __restrict__ twhi, uint32_t per,
                                                              const BlockArgs* __restrict__ bt) {
    fwd_batch_args<BATCH, true>(a, g, bt);
    using P = MidPlan<LG1>;
    constexpr int N1 = P::N1, NT = P::NT, R1 = P::R1, R2 = P::R2, NA = R2 / 8;
    __shared__ float2 buf[16 * P::SEQS];
    __shared__ float2 tab[R1 * stage_row<R2>()];
    __shared__ uint32_t bw[N1];  // the group's 16 bits of row u, and of row u + N1 above them
    const uint32_t op = blockIdx.x / a.nA;
    if (op >= a.ops) {
        scan_chunk<NT>(blockIdx.x - a.ops * a.nA, a.scan, g, reinterpret_cast<uint32_t*>(buf));
        return;
    }
    const bool is_seed = a.first + op == 1u;
    const uint32_t* __restrict__ in = is_seed ? a.in[1] : a.in[0];
    float2* __restrict__ Y = is_seed ? a.Y[1] : a.Y[0];
    if (BATCH && in == nullptr) return;
    const uint32_t grp0 = (blockIdx.x - op * a.nA) * (WALK ? per : 1u);
    struct Words {
        uint32_t lo[P::RPT], hi[P::RPT];
    };
    auto load_words = [&](Words& x, uint32_t wc) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < P::RPT; ++i) {
            const uint32_t w = wc + (g.N2 >> 5) * (threadIdx.x + (uint32_t)(NT * i)), wh = w + (g.N >> 5);
            const uint32_t white = is_seed ? 0u : white_word(g, w);  // N positions are whole periods
            x.lo[i] = is_seed ? seed_word(in, g, w) : key_word(in, g, w) ^ white;
            x.hi[i] = is_seed ? seed_word(in, g, wh) : key_word(in, g, wh) ^ white;
        }
    };
    auto pack = [&](const Words& x, uint32_t grp) __attribute__((always_inline)) {
        const uint32_t sh = (grp & 1u) ? 0u : 16u;
#pragma unroll
        for (int i = 0; i < P::RPT; ++i)
            bw[threadIdx.x + NT * i] = ((x.lo[i] >> sh) & 0xFFFFu) | ((x.hi[i] >> sh) << 16);
    };
    const int col = threadIdx.x & 15, jt = threadIdx.x >> 4;
    const uint32_t L2m = 2u * g.L - 1u;
    // (lo, hi) entries of w_2L^{t2 (4 k1 + 1)}, k1 = jt + R1 r = anchor step^(r mod 8): the anchors, then
    // the step; their products are formed where they are used
    using Tw = float2[2 * (NA + 1)];
    auto load_tw = [&](Tw& x, uint32_t grp) __attribute__((always_inline)) {
        const uint32_t t2 = 16u * grp + (uint32_t)col;
#pragma unroll
        for (int i = 0; i <= NA; ++i) {
            const uint32_t e = (t2 * (i < NA ? 4u * ((uint32_t)jt + (uint32_t)(8 * R1 * i)) + 1u : 4u * R1)) & L2m;
            x[2 * i] = twlo[e & (TW14 - 1)];
            x[2 * i + 1] = twhi[e >> TW14_LOG];
        }
    };
    Words cur, nxt;
    Tw tw, twn;
    load_words(cur, grp0 >> 1);
    load_tw(tw, grp0);
    // second stage's factors: row q for w_N1^(q + 1/4)
    for (int e = threadIdx.x; e < R1 * (R2 / 2); e += NT) {
        const int q = e / (R2 / 2), i = e % (R2 / 2);
        int s = 2;
        while (s / 2 <= i && i > 0) s *= 2;
        const int k = i ? i - s / 4 : 0;
        tab[q * stage_row<R2>() + i] = tw14[((4 * q + 1) * (TW14 / (4 * R1 * s)) + k * (TW14 / s)) & (TW14 - 1)];
    }
    float2 tw1[R1 / 2];  // first stage: w = exp(-2 pi i / (4 R1)), size s, k: exp(-2 pi i (4k + 1) / (4s))
#pragma unroll
    for (int i = 0; i < R1 / 2; ++i) {
        const int s = i == 0 ? 2 : i == 1 ? 4 : i < 4 ? 8 : i < 8 ? 16 : 32, k = i ? i - s / 4 : 0;
        tw1[i] = uniform_f2(tw14[(4 * k + 1) * (TW14 / (4 * s))]);
    }
    pack(cur, grp0);
    __syncthreads();
    float2* seqbuf = buf + col * P::SEQS;
    const __amdgpu_buffer_rsrc_t ry = make_rsrc(Y, g.N1 * g.N2 * 8u);
    auto stage1 = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < P::K1; ++i) {
            const int j = jt + (NT / 16) * i;
            float2 v[R1];
#pragma unroll
            for (int r = 0; r < R1; ++r) {  // z = (bit - 1/2) - i (bit' - 1/2)
                const uint32_t b = bw[j + P::S1 * r] << (16 + col);
                const uint32_t bh = bw[j + P::S1 * r] << col;
                v[r] = make_float2((int)b < 0 ? 0.5f : -0.5f, (int)bh < 0 ? -0.5f : 0.5f);
            }
            dft_tw<R1>(v, tw1);
#pragma unroll
            for (int r = 0; r < R1; ++r) seqbuf[padi(j * R1 + r)] = v[r];
        }
        __syncthreads();
    };
    auto stage2 = [&](uint32_t grp) __attribute__((always_inline)) {
        float2 F[R2];
        stage_last_from_lds_tab<R2, N1>(F, seqbuf, jt, tab + jt * stage_row<R2>());
        const float2 step = cmul(tw[2 * NA], tw[2 * NA + 1]);
        const uint32_t vo = ((uint32_t)jt * g.N2 + 16u * grp + (uint32_t)col) * 8u;
        float2 w = make_float2(0.f, 0.f);
#pragma unroll
        for (int r = 0; r < R2; ++r) {
            w = (r & 7) == 0 ? cmul(tw[2 * (r / 8)], tw[2 * (r / 8) + 1]) : cmul(w, step);
            buf_store<WALK ? 2 : 0>(cmul(F[r], w), ry, vo, (uint32_t)(R1 * r) * g.N2 * 8u);
        }
    };
    auto advance = [&]() __attribute__((always_inline)) {  // to the next group: its bits are packed, its twiddles loaded
#pragma unroll
        for (int i = 0; i < 2 * (NA + 1); ++i) tw[i] = twn[i];
        __syncthreads();  // packed bits; second-stage reads of the previous group are done
    };
    if constexpr (!WALK) {
        stage1();
        stage2(grp0);
    } else {
        // A pair of groups; more: another pair follows.
        auto pair = [&](uint32_t grp, bool more) __attribute__((always_inline)) {
            if (more) load_words(nxt, (grp >> 1) + 1u);
            stage1();
            pack(cur, grp + 1u);
            load_tw(twn, grp + 1u);
            stage2(grp);
            advance();
            stage1();
            if (more) {
                cur = nxt;
                pack(cur, grp + 2u);
                load_tw(twn, grp + 2u);
            }
            stage2(grp + 1u);
        };
        // the first pair is peeled: see k_fwd_cols
        pair(grp0, per > 2u);
        for (uint32_t it = 2; it < per; it += 2) {
            advance();
            pair(grp0 + it, it + 2u < per);
        }
    }
}

// Transforms of 3 * 2^k: pass A and pass A' of N1 = D 256 points, D = 3 or 6 (pa_geom.hpp), 16 columns per
// workgroup like the passes of the powers of two.
// Stage factors of the 256-point transforms over u with inputs times w_N1^{u f / 4} (f / 4 = c + 1/4 in
// pass A, the residue q in pass A'): tw2 row j for w_256^j w_N1^{f/4}, tw1 for w_N1^{16 f / 4}; exponents
// in units of w_4N1.
constexpr int MIX_TW2 = 16 * stage_row<16>(), MIX_TW1 = 8;
template <int D, int NC, int NT>
__device__ __forceinline__ void mix_factors(float2* tw2, float2* tw1, uint32_t f0, uint32_t fstep, const Geom& g,
                                            const float2* __restrict__ twlo, const float2* __restrict__ twhi) {
    for (uint32_t e = threadIdx.x; e < NC * 136u; e += NT) {
        const uint32_t c = e / 136u, r = e % 136u, q = r >> 3, i = r & 7u, f = f0 + fstep * c;
        uint32_t s = 2;  // the size of factor i and its index k at that size (dft_tw's order)
        while (s / 2u <= i && i > 0u) s *= 2u;
        const uint32_t k = i ? i - s / 4u : 0u, x = (16u / s) * (q < 16u ? 4u * D * q + f : 16u * f) + k * (4u * D * MIX_M / s);
        const float2 w = tw_two_level(twlo, twhi, x * g.N2);
        if (q < 16u) tw2[c * MIX_TW2 + q * stage_row<16>() + i] = w;
        else tw1[c * MIX_TW1 + i] = w;
    }
}

// Y[k1][t2], k1 = c + D k1', at the quarter-shifted frequencies: the sum over v < D of
// z[t2 + N2 (u + 256 v)] w_D^{v (c + 1/4)} by the class bits, then 256 points over u (16 x 16).
// A workgroup takes PER consecutive column groups (2: both of a word, streaming stores) and every class of
// them, so bits, indexes and twiddles are fetched once per group; PER = 0: one group and one class, for
// launches of few groups, which are bound by one workgroup's latency.  A batch's launch is bound by its
// stores: 11 blocks of 11.7 M bits, key and seed, take 0.24 ms for 1.11 GB (4.6 TB/s; the 1.48 GB of the
// power of two took 0.33).  No kernel of the served lengths may spill: scratch memory is given to a stream's
// queue at a launch's first use and stalls the streams in flight (17 registers spilled here at D = 6, with
// three workgroups a unit, and 2 in k_rows: p99.9 of a served stream 1.2 to 8 ms).
template <int D, int PER, bool BATCH>
__global__ __launch_bounds__(256, PER == 0 ? 4 : D == 6 ? 2 : 3) void k_mix_fwd(FwdArgs a, Geom g, const float2* __restrict__ twlo,
                                                                   const float2* __restrict__ twhi,
                                                                   const float2* __restrict__ cls,
                                                                   const BlockArgs* __restrict__ bt) {
    fwd_batch_args<BATCH, true>(a, g, bt);
    constexpr bool SPLIT = PER == 0;
    constexpr uint32_t per = SPLIT ? 1u : PER;
    constexpr int NT = 256, M = (int)MIX_M, SEQS = seq_stride(M), NC = SPLIT ? 1 : D;
    __shared__ float2 buf[16 * SEQS];
    __shared__ float2 tw2[NC * MIX_TW2];
    __shared__ float2 tw1s[NC * MIX_TW1];
    __shared__ float2 TB[NC * 64];
    __shared__ uint32_t bw[D * M];  // per row u + 256 v: 16 columns' bits, and those of a[. + N] above them
    const uint32_t op = blockIdx.x / a.nA;
    if (op >= a.ops) {
        scan_chunk<NT>(blockIdx.x - a.ops * a.nA, a.scan, g, reinterpret_cast<uint32_t*>(buf));
        return;
    }
    const bool is_seed = a.first + op == 1u;
    const uint32_t* __restrict__ in = is_seed ? a.in[1] : a.in[0];
    float2* __restrict__ Y = is_seed ? a.Y[1] : a.Y[0];
    if (BATCH && in == nullptr) return;
    const uint32_t b = blockIdx.x - op * a.nA, grp0 = SPLIT ? b / D : b * per, c0 = SPLIT ? b % D : 0u;
    uint32_t lo[D], hi[D];
    auto load_words = [&](uint32_t wc) __attribute__((always_inline)) {
        // M rows and N positions are whole periods of the whitening
        const uint32_t white = is_seed ? 0u : white_word(g, wc + (g.N2 >> 5) * threadIdx.x);
#pragma unroll
        for (int v = 0; v < D; ++v) {
            const uint32_t w = wc + (g.N2 >> 5) * (threadIdx.x + (uint32_t)(M * v)), wh = w + (g.N >> 5);
            lo[v] = is_seed ? seed_word(in, g, w) : key_word(in, g, w) ^ white;
            hi[v] = is_seed ? seed_word(in, g, wh) : key_word(in, g, wh) ^ white;
        }
    };
    const int col = threadIdx.x & 15, jt = threadIdx.x >> 4;
    // (lo, hi) entries of w_2L^{t2 (4 k1 + 1)}, k1 = c + D (jt + 16 r): of jt at c = 0, and the factors of r = 8,
    // of r and of c
    auto load_tw = [&](float2 (&x)[8], uint32_t grp) __attribute__((always_inline)) {
        const uint32_t t2 = 16u * grp + (uint32_t)col;
        const uint32_t f[4] = {4u * D * (uint32_t)jt + 1u, 4u * D * 128u, 4u * D * 16u, 4u};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[2 * i] = twlo[(t2 * f[i]) & (TW14 - 1)];
            x[2 * i + 1] = twhi[(t2 * f[i]) >> TW14_LOG];
        }
    };
    float2 tw[8];
    load_words(grp0 >> 1);
    load_tw(tw, grp0);
    for (uint32_t e = threadIdx.x; e < NC * 64; e += NT) TB[e] = cls[mix_table_offset(D) + 64u * c0 + e];
    mix_factors<D, NC, NT>(tw2, tw1s, 4u * c0 + 1u, 4u, g, twlo, twhi);
    float2* seqbuf = buf + col * SEQS;
    const __amdgpu_buffer_rsrc_t ry = make_rsrc(Y, g.N1 * g.N2 * 8u);
    for (uint32_t it = 0; it < per; ++it) {
        const uint32_t grp = grp0 + it, sh = (grp & 1u) ? 0u : 16u;
#pragma unroll
        for (int v = 0; v < D; ++v) bw[threadIdx.x + M * v] = ((lo[v] >> sh) & 0xFFFFu) | ((hi[v] >> sh) << 16);
        __syncthreads();  // bits (and tables); second-stage reads of the last group are done
        uint32_t idx[16];  // class bits of u = jt + 16 r: bit v, and v + 16 of a[. + N]
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            idx[r] = 0;
#pragma unroll
            for (int v = 0; v < D; ++v) idx[r] |= ((bw[jt + 16 * r + M * v] >> (15 - col)) & 0x10001u) << v;
        }
        const float2 a8 = cmul(tw[2], tw[3]), step = cmul(tw[4], tw[5]), cstep = cmul(tw[6], tw[7]);
        float2 base = cmul(tw[0], tw[1]);
        for (uint32_t c = 0; c < c0; ++c) base = cmul(base, cstep);
        if (it + 1u < per) load_tw(tw, grp + 1u);
        for (uint32_t i = 0; i < NC; ++i) {
            const uint32_t c = c0 + i;
            const float2* T = TB + 64u * i;
            float2 z[16], f1[8];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if constexpr (D == 3) {
                    z[r] = T[(idx[r] & 7u) | (idx[r] >> 13)];
                } else {
                    const float2 x = T[idx[r] & 63u], y = T[idx[r] >> 16];
                    z[r] = make_float2(x.x + y.y, x.y - y.x);
                }
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) f1[k] = uniform_f2(tw1s[i * MIX_TW1 + k]);
            dft_tw<16>(z, f1);
            if (i) __syncthreads();  // second-stage reads of the last class are done
#pragma unroll
            for (int r = 0; r < 16; ++r) seqbuf[padi(jt * 16 + r)] = z[r];
            __syncthreads();
            stage_last_from_lds_tab<16, M>(z, seqbuf, jt, tw2 + i * MIX_TW2 + jt * stage_row<16>());
            const uint32_t vo = ((c + (uint32_t)(D * jt)) * g.N2 + 16u * grp + (uint32_t)col) * 8u;
            float2 w = base;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (r == 8) w = cmul(base, a8);
                buf_store<PER == 2 ? 2 : 0>(cmul(z[r], w), ry, vo, (uint32_t)(16 * D * r) * g.N2 * 8u);
                w = cmul(w, step);
            }
            base = cmul(base, cstep);
        }
    }
}

// ------------------------------------------------------------------ pass B ----
// Rows of N2 = 2^LG2 points.  The frequencies k1 + N1 k2 + 1/4 of a row have no partners in other
// rows, so rows are independent:
//   forward plan R1 x 16 x 16 (16 x 16 at N2 = 256): stage 1 straight from global memory, stage 3
//   into registers, where thread j of a row holds k2 = j + NTR h + (N2/16) r (r < 16);
//   the product there;
//   inverse plan 16 x 16 x R1: stage 1 from those registers, stage 3 straight to global memory.
//   ROWS_SEEDPREP: seed rows (pass-A output) -> the seed spectrum S[k1 N2 + k2], in place.
//   ROWS_STATIC:   key rows + resident S -> R'[k1][t2] = w_N^{t2 (k1 + 1/4)} FFT_N2(conj P)[t2], in
//                  place, or into pass A''s tiles (Rt) when rt_tiled(lg1).
//   ROWS_DYN:      key rows + seed rows; S is formed first and held in registers.
// N2 = 8192 runs one row per 256-thread workgroup, 32 points per thread.  With a fresh seed it takes 74 KB of
// LDS and 176 registers, so two share a compute unit and one's memory requests overlap the other's
// transforms.  The other modes pass a row's real and imaginary parts through LDS one after the other
// (row_exchange: half the LDS for twice the barriers), so three do: on a resident seed a block of 2^24 bits
// takes 95 instead of 97.5 us, of 1.5 * 2^23 75 instead of 81 (its 768 rows are one round then), 2^25 208 instead
// of 213, 2^27 710 instead of 715, 2^23 in a batch 35.5 instead of 36.8.  Not with a fresh seed, where the
// seed row's 32 values more spill 23 registers and their reloads wait on the loads in flight: the pass
// takes 0.437 ms instead of 0.397 at 2^27.  Shorter rows take 16
// points per thread, rows_per_wg or rows_per_wg_many rows per workgroup.
// The launch's first workgroup finishes the scan (scan_finish).
// A row of 8192 points between two stages: value e of 32 goes to wi(e), comes back from ri(e), through LDS
// of half the row: real parts, then imaginary parts.  Ends with a barrier.
template <typename W, typename R>
__device__ __forceinline__ void row_exchange(float2 (&x)[32], float* lds, W&& wi, R&& ri) {
    float re[32];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 32; ++e) lds[wi(e)] = x[e].x;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 32; ++e) re[e] = lds[ri(e)];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 32; ++e) lds[wi(e)] = x[e].y;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 32; ++e) x[e] = make_float2(re[e], lds[ri(e)]);
    __syncthreads();
}
// Two radix-16 butterflies with the factors of one table row.
__device__ __forceinline__ void row_stage(float2 (&x)[32], const float2* trow) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float2 y[16], tw[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) tw[r] = trow[r];
#pragma unroll
        for (int r = 0; r < 16; ++r) y[r] = x[16 * h + r];
        dft_tw<16>(y, tw);
#pragma unroll
        for (int r = 0; r < 16; ++r) x[16 * h + r] = y[r];
        __builtin_amdgcn_sched_barrier(0);  // one butterfly's factors at a time
    }
}
template <int LG2, int MODE, bool BATCH, int RPW>
__global__ __launch_bounds__(rows_threads(LG2, RPW), LG2 == 13 ? (MODE == ROWS_DYN ? 2 : 3) : 1) void k_rows(
    float2* __restrict__ Yk, float2* __restrict__ Sst, float2* __restrict__ Rt, Geom g,
    const float2* __restrict__ tw14, const float2* __restrict__ twlo, const float2* __restrict__ twhi,
    uint32_t* __restrict__ info, const uint32_t* __restrict__ ws, uint32_t* __restrict__ seed_ws,
    const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) {
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        Yk = a.Yk;
        Sst = (MODE == ROWS_STATIC) ? const_cast<float2*>(a.sspec) : a.Ys;
        Rt = a.Rt;
        info = a.info;
        ws = a.seed ? nullptr : a.ws;
    }
    constexpr int N2 = 1 << LG2, NT = rows_threads(LG2, RPW), NTR = NT / RPW;
    constexpr int PPT = N2 / NTR, KL = PPT / 16;          // points and radix-16 butterflies per thread
    constexpr int R1 = LG2 == 8 ? 16 : N2 / 256, K1 = PPT / R1;
    constexpr int SEQS = seq_stride(N2);
    constexpr bool HALF = LG2 == 13 && MODE != ROWS_DYN;  // LDS holds one component of the row at a time
    __shared__ float2 buf[HALF ? SEQS / 2 : RPW * SEQS];
    float* fbuf = reinterpret_cast<float*>(buf);
    __shared__ float2 twl[TWL_SIZE];
    __shared__ float2 ttf[LG2 == 8 ? 1 : R1 * stage_row<16>()];  // forward middle stage (radix 16, span R1)
    __shared__ float2 tti[LG2 == 8 ? 1 : 16 * stage_row<16>()];  // inverse middle stage (radix 16, span 16)
    const uint32_t N1 = g.N1;
    if (blockIdx.x == 0) {
        scan_finish<NT, MODE == ROWS_STATIC>(info, g, ws, seed_ws, reinterpret_cast<uint32_t*>(buf));
        return;
    }
    const uint32_t row = (blockIdx.x - 1u) * RPW + threadIdx.x / NTR;
    const int j = threadIdx.x % NTR;
    float2* seqbuf = buf + (threadIdx.x / NTR) * SEQS;
    // buffer loads: one 32-bit offset register per thread
    const uint32_t vrow = (row * N2 + (uint32_t)j) * 8u;
    auto load = [&](const float2* __restrict__ src, float2 (&v)[PPT]) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(src, N1 * N2 * 8u);
#pragma unroll
        for (int e = 0; e < PPT; ++e) v[e] = buf_load_f2(rs, vrow, (uint32_t)(8 * NTR * e));
    };
    float2 v[PPT];
    load(MODE == ROWS_STATIC ? Yk : Sst, v);
    load_twl(twl, tw14, NT);
    if constexpr (LG2 != 8) {
        fill_stage_table<16, R1>(ttf, tw14, NT);
        fill_stage_table<16, 16>(tti, tw14, NT);
    }
    __syncthreads();  // tables
    // forward stages 1 (inputs in v) .. 3; request() runs once stage 1 has consumed v
    auto forward = [&](float2 (&z)[KL][16], auto&& request) __attribute__((always_inline)) {
        if constexpr (HALF) {
            float2 x[32];
#pragma unroll
            for (int r = 0; r < 32; ++r) x[r] = v[r];
            dft<32>(x);
            request();
            const int o = opaque_int(j);  // per-exchange address arithmetic, never kept live
            row_exchange(x, fbuf, [&](int e) { return 33 * j + e; }, [&](int e) { return padi(j + 256 * (e >> 4)) + 528 * (e & 15); });
            row_stage(x, ttf + (j & 31) * stage_row<16>());
            row_exchange(x, fbuf,
                         [&](int e) { const int b = o + 256 * (e >> 4); return padi((b / 32) * 512 + b % 32) + 33 * (e & 15); },
                         [&](int e) { return padi(o + 256 * (e >> 4)) + 528 * (e & 15); });
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float2 tw[8];
                twiddle_set_lds<16>(tw, twl, (j + 256 * h) * (TW14 / N2));
#pragma unroll
                for (int r = 0; r < 16; ++r) z[h][r] = x[16 * h + r];
                dft_tw<16>(z[h], tw);
                __builtin_amdgcn_sched_barrier(0);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < K1; ++i) {
            float2 x[R1];
#pragma unroll
            for (int r = 0; r < R1; ++r) x[r] = v[i + K1 * r];
            stage_first_to_lds<R1>(x, seqbuf, j + NTR * i);
        }
        request();
        __syncthreads();
        if constexpr (LG2 != 8) stockham_stage<16, R1, LG2, RPW, SEQS, NT, true>(buf, ttf);
#pragma unroll
        for (int h = 0; h < KL; ++h) stage_last_from_lds<16, N2>(z[h], seqbuf, j + NTR * h, twl);
        __syncthreads();  // stage-3 reads are done before LDS is overwritten
    };
    float2 S[KL][16];
    if constexpr (MODE == ROWS_SEEDPREP || MODE == ROWS_DYN) {
        forward(S, [&] {
            if constexpr (MODE == ROWS_DYN) load(Yk, v);  // the key row, while the seed row is transformed
        });
        if constexpr (MODE == ROWS_SEEDPREP) {
            // in place: every thread of the workgroup has consumed this row
#pragma unroll
            for (int h = 0; h < KL; ++h)
#pragma unroll
                for (int r = 0; r < 16; ++r) st_nt(&Sst[(size_t)row * N2 + j + NTR * h + (N2 / 16) * r], S[h][r]);
            return;
        }
    }
    float2 z[KL][16];
    forward(z, [&] {
        if constexpr (MODE == ROWS_STATIC) {
            // the resident spectrum is requested now, used after the FFT
            const __amdgpu_buffer_rsrc_t rs = make_rsrc(Sst, N1 * N2 * 8u);
#pragma unroll
            for (int h = 0; h < KL; ++h)
#pragma unroll
                for (int r = 0; r < 16; ++r) S[h][r] = buf_load_f2(rs, vrow, (uint32_t)(8 * NTR * h + (N2 / 2) * r));
        }
    });
    float2 F[PPT];
    if constexpr (HALF) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int r = 0; r < 16; ++r) z[h][r] = conjf2(cmul(z[h][r], S[h][r]));
            dft<16>(z[h]);
#pragma unroll
            for (int r = 0; r < 16; ++r) F[16 * h + r] = z[h][r];
            __builtin_amdgcn_sched_barrier(0);
        }
        row_exchange(F, fbuf, [&](int e) { return padi(16 * (j + 256 * (e >> 4))) + (e & 15); },
                     [&](int e) { return padi(j + 256 * (e >> 4)) + 528 * (e & 15); });
        row_stage(F, tti + (j & 15) * stage_row<16>());
        row_exchange(F, fbuf,
                     [&](int e) {
                         const int b = j + 256 * (e >> 4), r = e & 15;
                         return padi((b / 16) * 256 + b % 16) + 16 * r + (r >> 1);
                     },
                     [&](int e) { return padi(j) + 264 * e; });
        {
            float2 tw[16];
            twiddle_set_lds<32>(tw, twl, opaque_int(j) * (TW14 / N2));
            dft_tw<32>(F, tw);
        }
        __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
        for (int h = 0; h < KL; ++h) {
#pragma unroll
            for (int r = 0; r < 16; ++r) z[h][r] = conjf2(cmul(z[h][r], S[h][r]));
            stage_first_to_lds<16>(z[h], seqbuf, j + NTR * h);
        }
        __syncthreads();
        if constexpr (LG2 != 8) stockham_stage<16, 16, LG2, RPW, SEQS, NT, true>(buf, tti);
#pragma unroll
        for (int i = 0; i < K1; ++i) {
            float2 x[R1];
            stage_last_from_lds<R1, N2>(x, seqbuf, j + NTR * i, twl);
#pragma unroll
            for (int r = 0; r < R1; ++r) F[i + K1 * r] = x[r];
        }
    }
    // R'[row][t2] = F[t2] w_2L^{t2 (4 row + 1)}, t2 = j + NTR e: base step^e, re-anchored every 8
    // steps to bound the recurrence error
    const uint32_t f = 4u * row + 1u;  // f t2 < 2L
    const float2 base = tw_two_level(twlo, twhi, f * (uint32_t)j);
    const float2 step = tw_two_level(twlo, twhi, f * (uint32_t)NTR);
    float2 anchor[PPT / 8 - 1];
#pragma unroll
    for (int a = 0; a < PPT / 8 - 1; ++a)
        anchor[a] = tw_two_level(twlo, twhi, f * (uint32_t)(NTR * 8 * (a + 1)));
    // tiled (N2 = 8192): t2 = j + 256 e -> tile row t2 / RT_COLS = j / RT_COLS + (256 / RT_COLS) e, one
    // scalar offset per e; row-major: in place
    const bool tiled = LG2 == 13 && rt_tiled(g.lg1);
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(tiled ? Rt : Yk, N1 * N2 * 8u);
    const uint32_t vo = tiled ? ((((uint32_t)j / RT_COLS) * N1 + row) * RT_COLS + ((uint32_t)j % RT_COLS)) * 8u : vrow;
    const uint32_t estep = tiled ? (256u / RT_COLS) * N1 * RT_COLS * 8u : (uint32_t)(8 * NTR);  // e -> e + 1
    float2 tw = base;
#pragma unroll
    for (int e = 0; e < PPT; ++e) {
        if ((e & 7) == 0 && e) tw = cmul(base, anchor[e / 8 - 1]);
        buf_store_nt(cmul(F[e], tw), ro, vo, (uint32_t)e * estep);
        tw = cmul(tw, step);
    }
}

// ------------------------------------------------------------------ pass A' ----
// Workgroup grp owns columns [W*grp, W*grp + W): G[t1] = FFT_N1(R'[.][t2])[t1] w_4N1^{t1}, so that the
// conv values of positions t = t2 + N2 t1 and t + N are Re G / N and Im G / N.  R' is in pass B's tiles.
// Rounding: conv - mean_half(column) is an integer; its parity, corrected by the prefix parities (in
// the output stage), is the product's bit.
// A thread holds the outputs t1 = j + (N1/16) e, e < 16, of a column, so their bits are one 16-bit
// piece, bit e: piece[(half N2 + t2) N1/16 + j], half 0 for the positions t and 1 for t + N, each half
// only where the output window touches it.
struct InvOut {
    uint32_t lo, len;        // output window in conv positions
    uint32_t N, N2, S;       // S = N1 / 16
    uint16_t* piece;
    float* margin;
    __device__ __forceinline__ InvOut(const Geom& g, uint8_t* nib, uint32_t S_, float* margin_)
        : lo(g.out_off), len(g.out_bits), N(g.N), N2(g.N2), S(S_), piece(reinterpret_cast<uint16_t*>(nib)),
          margin(margin_) {}
    __device__ __forceinline__ bool low() const { return lo < N; }
    __device__ __forceinline__ bool high() const { return lo + len > N; }
};
// The 16-bit piece of half h from X[e] w_64^e (times the caller's scale: conv + i conv'): rounding by the
// 1.5 2^23 trick, whose last mantissa bit is the parity.  dist: max |v - rint v| inside the window.
template <bool HIGH, bool DIST>
__device__ __forceinline__ uint32_t inv_piece(const float2 (&X)[16], float mean, const InvOut& o, uint32_t t2, uint32_t j,
                                              float& dist) {
    constexpr float MAGIC = 12582912.f;
    const uint32_t i0 = t2 + o.N2 * j + (HIGH ? o.N : 0u) - o.lo;
    uint32_t acc = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const float2 w = w64pow(make_float2(1.f, 0.f), e);  // cos, -sin: constants
        const float v = HIGH ? fmaf(X[e].y, w.x, fmaf(X[e].x, w.y, -mean)) : fmaf(X[e].x, w.x, fmaf(X[e].y, -w.y, -mean));
        const float t = v + MAGIC;
        acc = __builtin_amdgcn_alignbit(__float_as_uint(t), acc, 1);
        if constexpr (DIST) {
            const float d = fabsf(v - (t - MAGIC));
            dist = fmaxf(dist, i0 + o.N2 * o.S * (uint32_t)e < o.len ? d : 0.f);
        }
    }
    return acc >> 16;
}
__device__ __forceinline__ void inv_store(const float2 (&X)[16], float mean, const InvOut& o, uint32_t t2, uint32_t j,
                                          float& dist) {
    uint16_t* p = o.piece + (size_t)t2 * o.S + j;
    const size_t plane = (size_t)o.N2 * o.S;
    if (o.margin) {
        if (o.low()) p[0] = (uint16_t)inv_piece<false, true>(X, mean, o, t2, j, dist);
        if (o.high()) p[plane] = (uint16_t)inv_piece<true, true>(X, mean, o, t2, j, dist);
    } else {
        if (o.low()) p[0] = (uint16_t)inv_piece<false, false>(X, mean, o, t2, j, dist);
        if (o.high()) p[plane] = (uint16_t)inv_piece<true, false>(X, mean, o, t2, j, dist);
    }
}
template <int LG1, bool BATCH>
__global__ __launch_bounds__(inv_cols_threads(LG1), 2) void k_inv_cols(
    const float2* __restrict__ Rp, uint8_t* __restrict__ nib, Geom g, const uint32_t* __restrict__ info,
    const float2* __restrict__ tw14, const float2* __restrict__ twlo, const float2* __restrict__ twhi,
    float* __restrict__ margin, const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) {
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        Rp = a.Rt;
        nib = a.nib;
        info = a.info;
        margin = a.margin;
    }
    constexpr int N1 = 1 << LG1;
    constexpr int W = inv_cols_width(LG1);
    constexpr int NT = inv_cols_threads(LG1);
    constexpr int SEQS = seq_stride(N1);
    constexpr int WL = LG1 == RT_LG1 ? 1 : W;  // columns held in LDS at once
    constexpr int S = N1 / 16;
    __shared__ float2 buf[WL * SEQS];
    __shared__ float2 twl[TWL_SIZE];
    load_twl(twl, tw14, NT);
    const uint32_t grp = xcd_logical(blockIdx.x, gridDim.x);
    const InvOut out(g, nib, S, margin);
    float dist = 0.f;
    // w_4N1^{j} / N from the length-2L table (2L = 4 N1 N2)
    auto out_tw = [&](uint32_t j) { return cscale(tw_two_level(twlo, twhi, j * g.N2), g.inv_N); };
    if constexpr (LG1 == RT_LG1) {
        // One column pair t2 = 2 grp, 2 grp + 1 from pass B's tiles per 256-thread workgroup, one
        // column in LDS at a time (72 KB), so that two workgroups share a compute unit and one's
        // reads overlap the other's transforms.  Thread j loads both columns of row k1 = j + 256 r
        // with one 16-byte load, so a workgroup walks consecutive lines.  Plan 32 x 16 x 16 per
        // column: stage 1 from the loaded registers, stage 2 in LDS, stage 3 into registers for
        // butterflies b = j and j + 256 (t1 = b + 512 r), w_4N1^b / N in its first level.
        // What bounds it is the L1 refill: 16 of each line's 128 bytes per workgroup, 8 times the
        // data in lines; the loads alone take 0.205 ms at 2^27, the transforms alone 0.14.
        static_assert(W == 2 && NT == 256, "tiled column pass expects 2 columns, 256 threads");
        static_assert(RT_COLS % W == 0, "a workgroup's columns lie in one tile");
        __shared__ float2 ttf[32 * stage_row<16>()];
        fill_stage_table<16, 32>(ttf, tw14, NT);
        const int j = threadIdx.x;
        const uint32_t t2 = grp * W;
        float2 v0[32], v1[32];
        {
            const float2* tp = Rp + (size_t)(t2 / RT_COLS) * N1 * RT_COLS + (t2 % RT_COLS);
#pragma unroll
            for (int r = 0; r < 32; ++r) {
                const float4 x = *reinterpret_cast<const float4*>(tp + (size_t)(j + 256 * r) * RT_COLS);
                v0[r] = make_float2(x.x, x.y);
                v1[r] = make_float2(x.z, x.w);
            }
        }
        const uint32_t pops = info[INFO_POPS];
        const float2 wb[2] = {out_tw((uint32_t)j), out_tw((uint32_t)j + 256u)};
        auto column = [&](float2 (&v)[32], uint32_t col) {
            stage_first_to_lds<32>(v, buf, j);
            __syncthreads();
            stockham_stage<16, 32, LG1, 1, SEQS, NT, true>(buf, ttf);
            const float mean = mean_half(pops, col);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float2 G[16], tw[8];
                const int b = j + 256 * h;
                stage_last_read<16, N1>(G, buf, b);
                twiddle_set_lds<16>(tw, twl, b * (TW14 / N1));
                tw[0] = cmul(tw[0], wb[h]);
#pragma unroll
                for (int r = 0; r < 8; ++r) G[r] = cmul(G[r], wb[h]);
                dft_tw<16>(G, tw);
                inv_store(G, mean, out, col, (uint32_t)b, dist);
            }
        };
        __syncthreads();  // twl, ttf
        column(v0, t2);
        __syncthreads();  // the first column's stage-3 reads are done
        column(v1, t2 + 1u);
    } else {
        constexpr int LPT = (W * N1 + NT - 1) / NT;
        static_assert(W * S == NT, "one piece per thread");
        float2 v[LPT];
#pragma unroll
        for (int i = 0; i < LPT; ++i) {
            const int e = threadIdx.x + i * NT;
            const uint32_t k1 = (uint32_t)(e / W), t2 = grp * W + (uint32_t)(e % W);
            v[i] = Rp[((size_t)(t2 / RT_COLS) * N1 + k1) * RT_COLS + t2 % RT_COLS];  // pass B's tiles
        }
#pragma unroll
        for (int i = 0; i < LPT; ++i) {
            const int e = threadIdx.x + i * NT;
            buf[(e % W) * SEQS + padi(e / W)] = v[i];
        }
        __syncthreads();
        lds_fft<LG1, W, SEQS, NT>(buf, twl);
        const int col = threadIdx.x / S, j = threadIdx.x % S;
        const float2 wb = out_tw((uint32_t)j);
        float2 X[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) X[e] = cmul(buf[col * SEQS + padi(j + S * e)], wb);
        const uint32_t t2 = grp * W + (uint32_t)col;
        inv_store(X, mean_half(info[INFO_POPS], t2), out, t2, (uint32_t)j, dist);
    }
    if (margin) margin_publish(dist, margin);
}

// N1 = 2^14, 2^15: a column of 128 or 256 KB leaves a single-pass kernel one or two columns per
// workgroup, which refill L1 with 16 or 8 times the data (0.8 and 3.0 ms at 2^28 and 2^29).  Two
// passes over whole 128-byte lines instead, k1 = j + J i with J = N1 / 1024:
//   k_inv_big1: 1024-point FFTs over i, in place: Z_j[s] = sum_i R'[j + J i] w_1024^{i s} at row j + J s;
//   k_inv_big2: G[s + 1024 b] = sum_j Z_j[s] w_N1^{(j + 1/4)(s + 1024 b)}, J points from J adjacent rows,
//               in registers, then the rounding.
// At 2^29: 0.79 ms (4.3 GB, the card's copy rate) + 0.43 ms (2.1 GB), from 3.02.
template <int LG1, bool BATCH>
__global__ __launch_bounds__(512) void k_inv_big1(float2* __restrict__ Rp, Geom g, const float2* __restrict__ tw14,
                                                  const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) Rp = bt[blockIdx.z].Rt;
    constexpr int N1 = 1 << LG1, J = N1 / 1024, NT = 512, SEQS = seq_stride(1024);
    static_assert(RT_COLS == 16, "a workgroup has the columns of a tile");
    __shared__ float2 buf[16 * SEQS];
    __shared__ float2 tab[32 * stage_row<32>()];
    const uint32_t logical = xcd_logical(blockIdx.x, gridDim.x), grp = logical / J, j = logical % J;
    const int col = threadIdx.x & 15, jt = threadIdx.x >> 4;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(Rp, g.N1 * g.N2 * 8u);
    // row j + J i, i = jt + 32 r
    const uint32_t vo = ((grp * (uint32_t)N1 + j + (uint32_t)(J * jt)) * 16u + (uint32_t)col) * 8u;
    float2 v[32];
#pragma unroll
    for (int r = 0; r < 32; ++r) v[r] = buf_load_f2(rs, vo, (uint32_t)(32 * J * r) * 128u);
    fill_stage_table<32, 32>(tab, tw14, NT);
    float2* seqbuf = buf + col * SEQS;
    stage_first_to_lds<32>(v, seqbuf, jt);
    __syncthreads();
    stage_last_from_lds_tab<32, 1024>(v, seqbuf, jt, tab + jt * stage_row<32>());
#pragma unroll
    for (int r = 0; r < 32; ++r) buf_store_nt(v[r], rs, vo, (uint32_t)(32 * J * r) * 128u);
}
template <int LG1, bool BATCH>
__global__ __launch_bounds__(256) void k_inv_big2(const float2* __restrict__ Rp, uint8_t* __restrict__ nib, Geom g,
                                                  const uint32_t* __restrict__ info, const float2* __restrict__ twlo,
                                                  const float2* __restrict__ twhi, float* __restrict__ margin,
                                                  const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) {
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        Rp = a.Rt;
        nib = a.nib;
        info = a.info;
        margin = a.margin;
    }
    constexpr int N1 = 1 << LG1, J = N1 / 1024;
    // 16 columns x 16 values of s per workgroup
    const uint32_t logical = xcd_logical(blockIdx.x, gridDim.x);
    const uint32_t grp = logical / 64u, s = (logical % 64u) * 16u + (threadIdx.x >> 4);
    const uint32_t t2 = grp * 16u + (threadIdx.x & 15u);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(Rp, g.N1 * g.N2 * 8u);
    const uint32_t vo = ((grp * (uint32_t)N1 + (uint32_t)J * s) * 16u + (threadIdx.x & 15u)) * 8u;
    float2 v[J];
#pragma unroll
    for (int j = 0; j < J; ++j) v[j] = buf_load_f2(rs, vo, (uint32_t)(128 * j));
    // w_N1^{j s} in the butterflies, K = w_4N1^s / N on the result; the output factor w_4J^b of b = e
    // (J = 16) is inv_store's w_64^e, of b = 2e and 2e + 1 (J = 32) that and w_128 times it
    const uint32_t u = s * g.N2;  // w_4N1^s = w_2L^u
    const float2 K = cscale(tw_two_level(twlo, twhi, u), g.inv_N);
    float2 pw[5], tw[J / 2];
#pragma unroll
    for (int m = J / 2, l = 0; m >= 1; m /= 2, ++l) pw[l] = tw_two_level(twlo, twhi, (4u * u * (uint32_t)m) & (2u * g.L - 1u));
    twiddle_set<J>(tw, pw);
    tw[0] = cmul(tw[0], K);
#pragma unroll
    for (int j = 0; j < J / 2; ++j) v[j] = cmul(v[j], K);
    dft_tw<J>(v, tw);
    const InvOut out(g, nib, N1 / 16, margin);
    const float mean = mean_half(info[INFO_POPS], t2);
    float dist = 0.f;
    float2 X[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) X[e] = v[J / 16 * e];
    inv_store(X, mean, out, t2, s, dist);
    if constexpr (J == 32) {
#pragma unroll
        for (int e = 0; e < 16; ++e) X[e] = cmul(v[2 * e + 1], make_float2(9.987954562e-01f, -4.906767433e-02f));  // w_128
        inv_store(X, mean, out, t2, s + 1024u, dist);
    }
    if (margin) margin_publish(dist, margin);
}

// ------------------------------------------------------------------ output ----
// The correction of conv word w, MSB first: the prefix parities (q and its chunk's cp), conv(R, t)
// and key_rest word wo = w - out_off / 32 ((key[h/32+wo] << 1) | (key[h/32+wo+1] >> 31),
// key2StartRest PrivacyAmplification.cu:873-878).  No load is conditional on a lane, so that a thread
// with several words has all their operands in flight.
__device__ __forceinline__ uint32_t out_correction(uint32_t w, uint32_t wo, const Geom& g, const uint32_t* __restrict__ q,
                                                   const uint32_t* __restrict__ info,
                                                   const uint32_t* __restrict__ key) {
    uint32_t c = q[w] ^ (0u - (uint32_t)scan_parities(info)[w >> (10u + g.scan)]) ^ info[info_white(g) + (w & (g.white - 1u))];
    if (g.do_xor) {
        const bool in = 32u * wo < g.m;
        const uint32_t k = g.key_hw + (in ? wo : 0u);
        const uint32_t r = (key[k] << 1) | (key[k + 1] >> 31);
        c ^= in ? r : 0u;
    }
    return c;
}
// Pieces (pass A') to output words.  Thread (cw, jp) of a tile of 16 column words x 8 piece pairs takes
// the 32 columns of word cw at rows t1 = j + (N1/16) e, j = 2 jp and 2 jp + 1: a 32 x 32 bit matrix, one
// word per column, transposed in registers to one word per row; through LDS the tile's 256 rows are
// then written as whole 64-byte runs, corrected and byte-swapped for the OutBytes layout
// (ToBinaryArray, PrivacyAmplification.cu:757-762), eight rows' operands in flight per thread.
template <bool BATCH>
__global__ __launch_bounds__(PACK_NT) void k_pack(const uint8_t* __restrict__ nib, const uint32_t* __restrict__ key,
                                                  uint32_t* __restrict__ out, Geom g, const uint32_t* __restrict__ info,
                                                  const uint32_t* __restrict__ q, const BlockArgs* __restrict__ bt) {
    static_assert(PACK_CW * 8 == PACK_NT, "a thread per word column and piece pair");
    __shared__ uint32_t tile[256 * (PACK_CW + 1)];
    if constexpr (BATCH) {  // grid.y covers the most halves of the launch
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        nib = a.nib;
        key = a.key;
        out = a.out;
        info = a.info;
        q = a.q;
    }
    const uint32_t S = g.N1 >> 4, per_half = S / 16u;
    const uint32_t w_lo = g.out_off >> 5, w_hi = (g.out_off + g.out_bits) >> 5;
    const uint32_t half = blockIdx.y / per_half + (g.out_off < g.N ? 0u : 1u);
    if (half > 1u || (half == 1u && 32u * w_hi <= g.N)) return;
    const uint32_t jl = threadIdx.x & 7u, cl = threadIdx.x >> 3;
    const uint32_t jp0 = (blockIdx.y % per_half) * 8u, c0 = blockIdx.x * PACK_CW;
    {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(nib) +
                            ((size_t)half * g.N2 + 32u * (c0 + cl)) * (S / 2u) + jp0 + jl;
        uint32_t A[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) A[k] = p[(size_t)k * (S / 2u)];
        bit_transpose(A);  // A[31 - b]: bit b of every column, first column in the MSB
#pragma unroll
        for (int b = 0; b < 32; ++b) tile[(b * 8 + jl) * (PACK_CW + 1) + cl] = A[31 - b];
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x % PACK_CW;
    const uint8_t* cp = scan_parities(info);
    const uint32_t* white = info + info_white(g);
    for (uint32_t r0 = threadIdx.x / PACK_CW; r0 < 256u; r0 += 64u) {
        // the operands of out_correction for eight words, requested together
        uint32_t w[8], c[8], flip[8], r[8], k0[8], k1[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            const uint32_t row = r0 + 8u * k, b = row >> 3, t1 = 2u * (jp0 + (row & 7u)) + (b >> 4) + S * (b & 15u);
            w[k] = (half * g.N1 + t1) * (g.N2 >> 5) + c0 + lane;  // conv word
            const uint32_t wc = w[k] >= w_lo && w[k] < w_hi ? w[k] : w_lo;
            c[k] = q[wc];
            flip[k] = cp[wc >> (10u + g.scan)];
            r[k] = white[w[k] & (WHITE_BIG - 1u)];
        }
        if (g.do_xor) {
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                const uint32_t wo = w[k] - w_lo, i = g.key_hw + (32u * wo < g.m && w[k] >= w_lo ? wo : 0u);
                k0[k] = key[i];
                k1[k] = key[i + 1];
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            const uint32_t wo = w[k] - w_lo;
            uint32_t cw = tile[(r0 + 8u * k) * (PACK_CW + 1) + lane] ^ c[k] ^ (0u - flip[k]) ^ r[k];
            if (g.do_xor && 32u * wo < g.m) cw ^= (k0[k] << 1) | (k1[k] >> 31);
            if (w[k] >= w_lo && w[k] < w_hi) out[wo] = g.reverse_endian ? __builtin_bswap32(cw) : cw;
        }
    }
}

// Pass A' and the output in one for L <= 2^24: 16 columns per workgroup, plan R1 x 16 (R1 x 32 at 512).
// A wave's 64 lanes are 16 columns x 4 rows, so a ballot is 4 rows' 16 bits: half an output word
// each, corrected and written as 16 bits.
template <int LG1, bool BATCH>
__global__ __launch_bounds__(mid_threads(LG1)) void k_mid_inv(const float2* __restrict__ Rp, const uint32_t* __restrict__ key,
                                                              uint32_t* __restrict__ out, Geom g,
                                                              const uint32_t* __restrict__ info,
                                                              const uint32_t* __restrict__ q,
                                                              const float2* __restrict__ tw14,
                                                              float* __restrict__ margin,
                                                              const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) {
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        Rp = a.Yk;
        key = a.key;
        out = a.out;
        info = a.info;
        q = a.q;
        margin = a.margin;
    }
    constexpr int N1 = 1 << LG1, NT = mid_threads(LG1), R1 = mid_r1(LG1), R2 = N1 / R1, S1 = N1 / R1;
    constexpr int K1 = 16 * S1 / NT, SEQS = seq_stride(N1);
    __shared__ float2 buf[16 * SEQS];
    __shared__ float2 tab[R1 * stage_row<R2>()];
    __shared__ float2 tq[N1];  // w_4N1^{t1} / N
    const int col = threadIdx.x & 15, jt = threadIdx.x >> 4;
    const uint32_t grp = blockIdx.x, t2 = 16u * grp + (uint32_t)col;
    float2 v[K1][R1];
#pragma unroll
    for (int i = 0; i < K1; ++i)
#pragma unroll
        for (int r = 0; r < R1; ++r) v[i][r] = Rp[(size_t)(jt + (NT / 16) * i + S1 * r) * g.N2 + t2];
    fill_stage_table<R2, R1>(tab, tw14, NT);
    for (int e = threadIdx.x; e < N1; e += NT) tq[e] = cscale(tw14[e * (TW14 / (4 * N1))], g.inv_N);
    const uint32_t pops = info[INFO_POPS];
#pragma unroll
    for (int i = 0; i < K1; ++i) stage_first_to_lds<R1>(v[i], buf + col * SEQS, jt + (NT / 16) * i);
    __syncthreads();
    float2 G[R2];
    stage_last_from_lds_tab<R2, N1>(G, buf + col * SEQS, jt, tab + jt * stage_row<R2>());
    const float mean = mean_half(pops, t2);
    const uint32_t RW = g.N2 >> 5, w_lo = g.out_off >> 5, w_hi = (g.out_off + g.out_bits) >> 5;
    const uint32_t lane = threadIdx.x & 63u, sh = (grp & 1u) ? 0u : 16u;
    float dist = 0.f;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (half == 0 ? g.out_off >= g.N : 32u * w_hi <= g.N) continue;
#pragma unroll
        for (int p = 0; p < R2 / 16; ++p) {
            uint32_t mine = 0;  // the 16 bits of row jt + R1 (16 p + col)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t t1 = (uint32_t)jt + (uint32_t)(R1 * (16 * p + e));
                const float2 X = G[16 * p + e], w = tq[t1];
                const float val = half == 0 ? fmaf(X.x, w.x, fmaf(-X.y, w.y, -mean)) : fmaf(X.x, w.y, fmaf(X.y, w.x, -mean));
                float d = 0.f;
                const uint64_t b = __ballot(round_bit(val, d) != 0u);
                const uint32_t pos = t2 + g.N2 * t1 + (half ? g.N : 0u) - g.out_off;
                dist = fmaxf(dist, pos < g.out_bits ? d : 0.f);
                const uint32_t word = (lane & 32u) ? (uint32_t)(b >> 32) : (uint32_t)b;
                mine = col == e ? word >> (lane & 16u) : mine;
            }
            const uint32_t R = (uint32_t)(half * N1 + jt + R1 * (16 * p + col));
            const uint32_t w = R * RW + (grp >> 1);
            if (w >= w_lo && w < w_hi) {
                const uint32_t wo = w - w_lo;
                // bit i of `mine` is column i: MSB first after the reversal
                const uint32_t c16 = (__brev(mine) >> 16) ^ ((out_correction(w, wo, g, q, info, key) >> sh) & 0xFFFFu);
                uint16_t* o = reinterpret_cast<uint16_t*>(out + wo);
                if (g.reverse_endian) o[grp & 1u] = (uint16_t)((c16 >> 8) | (c16 << 8));
                else o[(grp & 1u) ^ 1u] = (uint16_t)c16;
            }
        }
    }
    if (margin) margin_publish(dist, margin);
}

// The same for transforms of 3 * 2^k: rows t1 = q + D s are 256 points over i of
// w_N1^{i q} sum_{r < D} R'[i + 256 r] w_D^{r q}.  D / NQ workgroups per column group, side by side on one XCD;
// NQ = 3: workgroup h has the q of residue h mod D / 3 and forms their three sums of the D inputs in
// registers, then their transforms in turn; NQ = 1 (launches of few groups): one q each.  The registers bound
// it: at D = 6 the inputs of three sums and the second ones in flight take 212, two workgroups a compute unit
// (with three, 90 spilled: 5 blocks of 23.5 M bits 0.30 ms, now 0.19).
template <int D, int NQ, bool BATCH>
__global__ __launch_bounds__(256, NQ == 1 ? 4 : D == 6 ? 2 : 3) void k_mix_inv(
    const float2* __restrict__ Rp, const uint32_t* __restrict__ key, uint32_t* __restrict__ out, Geom g,
    const uint32_t* __restrict__ info, const uint32_t* __restrict__ q, const float2* __restrict__ twlo,
    const float2* __restrict__ twhi, float* __restrict__ margin, const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) {
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        Rp = a.Yk;
        key = a.key;
        out = a.out;
        info = a.info;
        q = a.q;
        margin = a.margin;
    }
    constexpr int H = D / NQ, M = (int)MIX_M, SEQS = seq_stride(M);
    static_assert(NQ == 3 || D == 3, "one q of three or three of D");
    __shared__ float2 buf[16 * SEQS];
    __shared__ float2 tw2[NQ * MIX_TW2];
    __shared__ float2 tw1s[NQ * MIX_TW1];
    const uint32_t logical = xcd_logical(blockIdx.x, gridDim.x);
    const int h = (int)(logical % H), col = threadIdx.x & 15, jt = threadIdx.x >> 4;
    const uint32_t grp = logical / H, t2 = 16u * grp + (uint32_t)col;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(Rp, g.N1 * g.N2 * 8u);
    const uint32_t vo = ((uint32_t)jt * g.N2 + t2) * 8u;
    float2 z[3][16];  // input r of i = jt + 16 e; D = 6: r plus or minus r + 3
#pragma unroll
    for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int r = 0; r < 3; ++r) z[r][e] = buf_load_f2(rs, vo, (uint32_t)(16 * e + M * r) * g.N2 * 8u);
    if constexpr (D == 6) {  // the others four e at a time, so that they never fill the registers
        float2 y[2][12];
        auto load_y = [&](int k) {
#pragma unroll
            for (int i = 0; i < 12; ++i) y[k & 1][i] = buf_load_f2(rs, vo, (uint32_t)(16 * (4 * k + i / 3) + M * (i % 3 + 3)) * g.N2 * 8u);
            __builtin_amdgcn_sched_barrier(0);
        };
        const float sign = h ? -1.f : 1.f;
        __builtin_amdgcn_sched_barrier(0);
        load_y(0);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k < 3) load_y(k + 1);
#pragma unroll
            for (int i = 0; i < 12; ++i) {
                float2& x = z[i % 3][4 * k + i / 3];
                x = make_float2(fmaf(sign, y[k & 1][i].x, x.x), fmaf(sign, y[k & 1][i].y, x.y));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    mix_factors<D, NQ, 256>(tw2, tw1s, 4u * (uint32_t)h, 4u * (uint32_t)H, g, twlo, twhi);
    const uint32_t pops = info[INFO_POPS];
    // sum b of NQ: q = h + H b
    constexpr float S3 = 8.660254038e-01f;
    const float cq = h ? -0.5f : 1.f, sq = h == 1 ? S3 : h ? -S3 : 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        if constexpr (NQ == 1) {  // w_3^q = cq - i sq
            const float2 s = cadd(z[1][e], z[2][e]), d = csub(z[1][e], z[2][e]);
            z[0][e] = make_float2(fmaf(sq, d.y, fmaf(cq, s.x, z[0][e].x)), fmaf(-sq, d.x, fmaf(cq, s.y, z[0][e].y)));
            continue;
        }
        if constexpr (D == 6)
            if (h) {  // odd q: input r times w_6^r
                z[1][e] = cmul(z[1][e], make_float2(0.5f, -S3));
                z[2][e] = cmul(z[2][e], make_float2(-0.5f, -S3));
            }
        const float2 s = cadd(z[1][e], z[2][e]), d = csub(z[1][e], z[2][e]);
        const float2 m = make_float2(fmaf(-0.5f, s.x, z[0][e].x), fmaf(-0.5f, s.y, z[0][e].y));
        z[0][e] = cadd(z[0][e], s);
        z[1][e] = make_float2(fmaf(S3, d.y, m.x), fmaf(-S3, d.x, m.y));
        z[2][e] = make_float2(fmaf(-S3, d.y, m.x), fmaf(S3, d.x, m.y));
    }
    const float mean = mean_half(pops, t2);
    const uint32_t RW = g.N2 >> 5, w_lo = g.out_off >> 5, w_hi = (g.out_off + g.out_bits) >> 5;
    const uint32_t lane = threadIdx.x & 63u, sh = (grp & 1u) ? 0u : 16u;
    float dist = 0.f;
    float2* seqbuf = buf + col * SEQS;
    // w_4N1^{D jt + h} / N, and w_4N1^H for the next b
    float2 K = cscale(tw_two_level(twlo, twhi, (uint32_t)(D * jt + h) * g.N2), g.inv_N);
    const float2 kstep = tw_two_level(twlo, twhi, (uint32_t)H * g.N2);
    __syncthreads();  // tables
#pragma unroll
    for (int b = 0; b < NQ; ++b) {
        const int qr = h + H * b;
        {
            float2 f1[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) f1[i] = uniform_f2(tw1s[b * MIX_TW1 + i]);
            dft_tw<16>(z[b], f1);
        }
        if (b) __syncthreads();  // second-stage reads of the last transform are done
#pragma unroll
        for (int r = 0; r < 16; ++r) seqbuf[padi(jt * 16 + r)] = z[b][r];
        __syncthreads();
        float2 G[16];
        {
            float2 tw[8];
            const float2* trow = tw2 + b * MIX_TW2 + jt * stage_row<16>();
            stage_last_read<16, M>(G, seqbuf, jt);
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                tw[r] = trow[r];
                G[r] = cmul(G[r], K);
            }
            tw[0] = cmul(tw[0], K);
            dft_tw<16>(G, tw);
        }
        K = cmul(K, kstep);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (half == 0 ? g.out_off >= g.N : 32u * w_hi <= g.N) continue;
            uint32_t mine = 0;  // the 16 bits of row qr + D (jt + 16 col)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t t1 = (uint32_t)(qr + D * (jt + 16 * e));
                const float2 X = G[e], w = w64pow(make_float2(1.f, 0.f), e);
                const float val = half == 0 ? fmaf(X.x, w.x, fmaf(-X.y, w.y, -mean)) : fmaf(X.x, w.y, fmaf(X.y, w.x, -mean));
                float d = 0.f;
                const uint64_t bits = __ballot(round_bit(val, d) != 0u);
                const uint32_t pos = t2 + g.N2 * t1 + (half ? g.N : 0u) - g.out_off;
                dist = fmaxf(dist, pos < g.out_bits ? d : 0.f);
                const uint32_t word = (lane & 32u) ? (uint32_t)(bits >> 32) : (uint32_t)bits;
                mine = col == e ? word >> (lane & 16u) : mine;
            }
            const uint32_t R = (uint32_t)half * g.N1 + (uint32_t)(qr + D * (jt + 16 * col));
            const uint32_t w = R * RW + (grp >> 1);
            if (w >= w_lo && w < w_hi) {
                const uint32_t wo = w - w_lo;
                // bit i of `mine` is column i: MSB first after the reversal
                const uint32_t c16 = (__brev(mine) >> 16) ^ ((out_correction(w, wo, g, q, info, key) >> sh) & 0xFFFFu);
                uint16_t* o = reinterpret_cast<uint16_t*>(out + wo);
                if (g.reverse_endian) o[grp & 1u] = (uint16_t)((c16 >> 8) | (c16 << 8));
                else o[(grp & 1u) ^ 1u] = (uint16_t)c16;
            }
        }
    }
    if (margin) margin_publish(dist, margin);
}

// ------------------------------------------------------------------ small path ----
// The whole block in one workgroup: N = 2^LGN <= 8192 complex points per operand in LDS.
// sspec != nullptr: static seed (precomputed split spectrum, N+1 values, popcount *ws_ptr).
// SEEDPREP: only computes the seed's split spectrum into sspec_out and its popcount.
template <int LGN, bool SEEDPREP, bool BATCH>
__global__ __launch_bounds__(small_threads(LGN)) void k_small(
    const uint32_t* __restrict__ key, const uint32_t* __restrict__ seed,
    const float2* __restrict__ sspec, const uint32_t* __restrict__ ws_ptr,
    uint32_t* __restrict__ out, Geom g, const float2* __restrict__ tw14,
    float* __restrict__ margin, float2* __restrict__ sspec_out, uint32_t* __restrict__ ws_out,
    const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) {
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        key = a.key;
        seed = a.seed;
        sspec = a.seed ? nullptr : a.sspec;
        ws_ptr = a.ws;
        out = a.out;
        margin = a.margin;
    }
    constexpr int N = 1 << LGN, L = 2 * N;
    constexpr int NT = small_threads(LGN);
    constexpr int SEQS = seq_stride(N);
    constexpr int PER = (N + NT - 1) / NT;
    __shared__ float2 buf[2 * SEQS];
    __shared__ float2 twl[TWL_SIZE];
    __shared__ uint32_t cnt[2];
    const int tid = threadIdx.x;
    load_twl(twl, tw14, NT);
    const bool dyn = SEEDPREP || (sspec == nullptr);
    if (tid < 2) cnt[tid] = 0u;
    __syncthreads();
    uint32_t ck = 0, cs = 0;
    for (int t = tid; t < N; t += NT) {
        const uint32_t pos = 2u * (uint32_t)t, widx = pos >> 5, sh = pos & 31u;
        if (!SEEDPREP) {
            const uint32_t w = key_word(key, g, widx);
            const uint32_t e = (w >> (31u - sh)) & 1u, o = (w >> (30u - sh)) & 1u;
            ck += e + o;
            buf[padi(t)] = make_float2((float)e - 0.5f, (float)o - 0.5f);
        } else {
            buf[padi(t)] = make_float2(0.f, 0.f);
        }
        if (dyn) {
            const uint32_t w = seed_word(seed, g, widx);
            const uint32_t e = (w >> (31u - sh)) & 1u, o = (w >> (30u - sh)) & 1u;
            cs += e + o;
            buf[SEQS + padi(t)] = make_float2((float)e - 0.5f, (float)o - 0.5f);
        }
    }
    if (ck) atomicAdd(&cnt[0], ck);
    if (cs) atomicAdd(&cnt[1], cs);
    __syncthreads();
    if (SEEDPREP) {
        lds_fft<LGN, 2, SEQS, NT>(buf, twl);  // sequence 0 is unused
    } else if (dyn) {
        lds_fft<LGN, 2, SEQS, NT>(buf, twl);
    } else {
        lds_fft<LGN, 1, SEQS, NT>(buf, twl);
    }
    constexpr int TWS = TW14 / L;
    float2 X[PER];
    float2 PN = make_float2(0.f, 0.f);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int k = tid + i * NT;
        if (k >= N) continue;
        const int kp = (N - k) & (N - 1);
        const float2 wk = tw_lds(twl, k * TWS);
        float2 s, sn = make_float2(0.f, 0.f);
        if (dyn) {
            const float2 zk = buf[SEQS + padi(k)], zp = buf[SEQS + padi(kp)];
            s = r2c_split(zk, zp, wk);
            if (k == 0) {
                sn = r2c_nyquist(zk);
                s = make_float2(0.f, 0.f);
            }
        } else {
            s = sspec[k];
            if (k == 0) sn = sspec[N];
        }
        if (SEEDPREP) {
            sspec_out[k] = s;
            if (k == 0) sspec_out[N] = sn;
            continue;
        }
        const float2 zk = buf[padi(k)], zp = buf[padi(kp)];
        float2 x = r2c_split(zk, zp, wk);
        if (k == 0) {
            PN = cmul(r2c_nyquist(zk), sn);
            x = make_float2(0.f, 0.f);
        }
        X[i] = cmul(x, s);
    }
    if (SEEDPREP) {
        if (tid < POP_SLOTS) ws_out[tid] = (tid == 0) ? cnt[1] : 0u;
        return;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int k = tid + i * NT;
        if (k < N) buf[padi(k)] = X[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int k = tid + i * NT;
        if (k >= N) continue;
        const int kp = (N - k) & (N - 1);
        const float2 pp = (k == 0) ? PN : buf[padi(kp)];
        X[i] = conjf2(c2r_split(X[i], pp, tw_lds(twl, k * TWS)));
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int k = tid + i * NT;
        if (k < N) buf[padi(k)] = X[i];
    }
    __syncthreads();
    lds_fft<LGN, 1, SEQS, NT>(buf, twl);
    const uint32_t ws = dyn ? cnt[1] : pop_total(ws_ptr);
    const float corr = correction(cnt[0], ws, (uint32_t)L);
    const float invN = g.inv_N;
    float dist = 0.f;
    const uint32_t nwords = g.out_bits >> 5;
    for (uint32_t wd = (uint32_t)tid; wd < nwords; wd += NT) {
        const uint32_t t0 = (g.out_off + 32u * wd) >> 1;
        uint32_t cw = 0;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float2 G = buf[padi((int)t0 + j)];
            cw |= round_bit(G.x * invN + corr, dist) << (31 - 2 * j);
            cw |= round_bit(-G.y * invN + corr, dist) << (30 - 2 * j);
        }
        if (g.do_xor && 32u * wd < g.m) cw ^= (key[g.key_hw + wd] << 1) | (key[g.key_hw + wd + 1] >> 31);
        out[wd] = g.reverse_endian ? __builtin_bswap32(cw) : cw;
    }
    if (margin) margin_publish(dist, margin);
}

// ------------------------------------------------------------------ direct product ----
// The product itself for short blocks, 32 bit-products per two integer instructions: no transform and
// no rounding.  Output position p = 32 W + s is the parity of the XOR over the key words j of
//   key word j  AND  window(W - j, s),   window(k, s) bit t = S[32 k + s - 31 + t],
// S the seed sequence (circular in n, rotated by seed_rot words), so that bit 31 - b of the window meets
// key bit b = x[32 j + b].  U_k = the 32 bits from S[32 k - 31] on, staged in LDS; window(k, s) =
// (U_{k+1} : U_k) >> s, one funnel shift per lane s, serves R output words.
// A workgroup has R output words; its half-waves (lanes s) share out the key in chunks of 16 words.
// Bound by the vector ALU from 2^17 bits on (1 T word products a second) and by the launch below: calls of
// 2^10 to 2^16 bits take 4.5 to 5.8 us one after another, where the one-workgroup transform took 18 to 27
// and the three launches of the mid-size one 17 to 18; 3.2 of it is the kernel at 2^12.
template <int R, bool BATCH>
__global__ __launch_bounds__(DIRECT_NT_MAX) void k_direct(const uint32_t* __restrict__ key,
                                                          const uint32_t* __restrict__ seed, uint32_t* __restrict__ out,
                                                          Geom g, const BlockArgs* __restrict__ bt) {
    if constexpr (BATCH) {
        const BlockArgs& a = bt[blockIdx.z];
        g = a.g;
        key = a.key;
        seed = a.seed;
        out = a.out;
    }
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    __shared__ uint32_t part[DIRECT_NT_MAX / 64][R];
    const uint32_t words = g.out_bits >> 5, w0 = blockIdx.x * (uint32_t)R;
    if (w0 >= words) return;
    const uint32_t jpad = direct_key_words(g), NT = blockDim.x;
    uint32_t* kx = lds;         // key words, zero from key_hw + 1 on
    uint32_t* us = lds + jpad;  // U of words base .. base + jpad + R
    const int W0 = (int)((g.out_off >> 5) + w0), base = W0 - (int)jpad + 1;
    for (uint32_t i = threadIdx.x; i < jpad; i += NT) kx[i] = key_word(key, g, i);
    const int nw = (int)g.seed_words;
    auto at = [&](int k) {  // the words off the sequence's range only meet zero key words or unused outputs
        int i = k + (int)g.seed_rot;
        i = i < 0 ? i + nw : i >= nw ? i - nw : i;
        return __brev(seed[min(max(i, 0), nw - 1)]);
    };
    for (uint32_t i = threadIdx.x; i < jpad + (uint32_t)R + 1u; i += NT)
        us[i] = __builtin_amdgcn_alignbit(at(base + (int)i), at(base + (int)i - 1), 1u);
    __syncthreads();
    const uint32_t sh = threadIdx.x & 31u;
    uint32_t acc[R] = {};
    for (uint32_t j0 = 16u * (threadIdx.x >> 5); j0 < jpad; j0 += NT / 2u) {
        constexpr int NU = (16 + R + 3) / 4 * 4;
        uint32_t kw[16], u[NU];
#pragma unroll
        for (int i = 0; i < 16; i += 4) *reinterpret_cast<uint4*>(kw + i) = *reinterpret_cast<const uint4*>(kx + j0 + i);
        const uint32_t* up = us + (jpad - 16u - j0);  // U of word W0 - j0 - 15 on
#pragma unroll
        for (int i = 0; i < NU; i += 4) *reinterpret_cast<uint4*>(u + i) = *reinterpret_cast<const uint4*>(up + i);
#pragma unroll
        for (int a = 0; a < 15 + R; ++a) {
            const uint32_t win = __builtin_amdgcn_alignbit(u[a + 1], u[a], sh);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int j = 15 - a + r;
                if (j >= 0 && j < 16) acc[r] = __builtin_amdgcn_bitop3_b32(acc[r], kw[j], win, 0x78);  // acc ^ (kw & win)
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint64_t b = __ballot(__popc(acc[r]) & 1);
        if ((threadIdx.x & 63u) == 0u) part[threadIdx.x >> 6][r] = (uint32_t)b ^ (uint32_t)(b >> 32);
    }
    __syncthreads();
    const uint32_t wd = w0 + threadIdx.x;
    if (threadIdx.x >= (uint32_t)R || wd >= words) return;
    uint32_t c = 0;
    for (uint32_t i = 0; i < NT / 64u; ++i) c ^= part[i][threadIdx.x];
    c = __brev(c);  // position p at bit 31 - p mod 32
    if (g.do_xor && 32u * wd < g.m) c ^= (key[g.key_hw + wd] << 1) | (key[g.key_hw + wd + 1] >> 31);
    out[wd] = g.reverse_endian ? __builtin_bswap32(c) : c;
}

// ------------------------------------------------------------------ sub-block split ----
// The m x (h+1) Toeplitz product cut into b x b tiles (the tiling of LargeBlocksizeExample,
// LBS/main.cpp:104-124, 313-523): tile (band i, key column j) is the length-2b circular product of
// key bits [jb, jb+b) (bit b zero) with the seed segment S[R, R+b) || S[R-b, R) at R = (i-j)b mod n,
// read at [0, b): z[v] = XOR_u x[jb+u] s[((i-j)b + v - u) mod n].  Tiles of a chunk are consecutive
// key columns j0.., all bands each: tile t = (j - j0) * nbands + i.
__global__ __launch_bounds__(256) void k_tile_inputs(const uint32_t* __restrict__ key,
                                                     const uint32_t* __restrict__ seed, uint32_t n,
                                                     uint32_t h, uint32_t b, uint32_t nbands, uint32_t j0,
                                                     uint32_t* __restrict__ tkeys, uint32_t* __restrict__ tseeds) {
    const uint32_t t = blockIdx.y, i = t % nbands, j = j0 + t / nbands;
    const uint32_t wb = b >> 5, nw = n >> 5, hw = h >> 5;
    const uint32_t R = (uint32_t)(((int64_t)i - (int64_t)j) * (int64_t)b % (int64_t)n + (int64_t)n) % n;
    const uint32_t R2 = (R + n - b % n) % n;
    uint32_t* tk = tkeys + (size_t)t * (wb + 1);
    uint32_t* ts = tseeds + (size_t)t * (2 * wb);
    for (uint32_t w = blockIdx.x * 256u + threadIdx.x; w < 3u * wb + 1u; w += gridDim.x * 256u) {
        if (w <= wb) {  // key words; word wb (bit b) is zero
            const uint32_t kw = j * wb + w;
            uint32_t v = 0;
            if (w < wb) v = kw < hw ? key[kw] : (kw == hw ? key[kw] & 0x80000000u : 0u);
            tk[w] = v;
        } else {
            const uint32_t sw = w - wb - 1u;  // seed word of the tile, < 2 wb
            const uint32_t src = sw < wb ? (R >> 5) + sw : (R2 >> 5) + (sw - wb);
            ts[sw] = seed[src % nw];
        }
    }
}

// acc[w] (=|^=) XOR over the chunk's columns of the tile outputs of band w / wb (32-bit words of
// the engine's output layout, which XOR word for word).
__global__ __launch_bounds__(256) void k_tile_xor(uint32_t* __restrict__ acc, const uint32_t* __restrict__ tout,
                                                  uint32_t nbands, uint32_t wb, uint32_t cols, int first) {
    const uint32_t w = blockIdx.x * 256u + threadIdx.x;
    if (w >= nbands * wb) return;
    const uint32_t i = w / wb, ww = w % wb;
    uint32_t x = first ? 0u : acc[w];
    for (uint32_t c = 0; c < cols; ++c) x ^= tout[(size_t)(c * nbands + i) * wb + ww];
    acc[w] = x;
}

// out word w = acc word w XOR the key rest word ((key[h/32+w] << 1) | (key[h/32+w+1] >> 31),
// key2StartRest PrivacyAmplification.cu:873-878) in the output byte order.
__global__ __launch_bounds__(256) void k_split_finish(const uint32_t* __restrict__ acc,
                                                      const uint32_t* __restrict__ key, uint32_t* __restrict__ out,
                                                      uint32_t m, uint32_t h, uint32_t do_xor, uint32_t reverse_endian) {
    const uint32_t w = blockIdx.x * 256u + threadIdx.x;
    if (w >= (m >> 5)) return;
    uint32_t kr = 0;
    if (do_xor) kr = (key[(h >> 5) + w] << 1) | (key[(h >> 5) + w + 1] >> 31);
    out[w] = acc[w] ^ (reverse_endian ? __builtin_bswap32(kr) : kr);
}

hipError_t launch_tile_inputs(const uint32_t* key, const uint32_t* seed, uint32_t n, uint32_t h, uint32_t b,
                              uint32_t nbands, uint32_t j0, uint32_t tiles, uint32_t* tkeys, uint32_t* tseeds,
                              hipStream_t s) {
    const uint32_t words = 3u * (b >> 5) + 1u;
    k_tile_inputs<<<dim3((words + 255u) / 256u, tiles), 256, 0, s>>>(key, seed, n, h, b, nbands, j0, tkeys, tseeds);
    return hipGetLastError();
}
hipError_t launch_tile_xor(uint32_t* acc, const uint32_t* tout, uint32_t nbands, uint32_t wb, uint32_t cols,
                           int first, hipStream_t s) {
    k_tile_xor<<<(nbands * wb + 255u) / 256u, 256, 0, s>>>(acc, tout, nbands, wb, cols, first);
    return hipGetLastError();
}
hipError_t launch_split_finish(const uint32_t* acc, const uint32_t* key, uint32_t* out, uint32_t m, uint32_t h,
                               uint32_t do_xor, uint32_t reverse_endian, hipStream_t s) {
    k_split_finish<<<((m >> 5) + 255u) / 256u, 256, 0, s>>>(acc, key, out, m, h, do_xor, reverse_endian);
    return hipGetLastError();
}

// ================================================================== launchers ====
namespace {
// f(std::integral_constant<int, lg>) for the mid-size column lengths, row lengths and the others.
template <typename F>
hipError_t by_mid_lg1(uint32_t lg1, F&& f) {
    switch (lg1) {
    case 6: return f(std::integral_constant<int, 6>());
    case 7: return f(std::integral_constant<int, 7>());
    case 8: return f(std::integral_constant<int, 8>());
    case 9: return f(std::integral_constant<int, 9>());
    case 10: return f(std::integral_constant<int, 10>());
    default: return hipErrorInvalidValue;
    }
}
template <typename F>
hipError_t by_classes(uint32_t D, F&& f) {
    return D == 3u ? f(std::integral_constant<int, 3>()) : f(std::integral_constant<int, 6>());
}
template <typename F>
hipError_t by_lg2(uint32_t lg2, F&& f) {
    switch (lg2) {
    case 8: return f(std::integral_constant<int, 8>());
    case 9: return f(std::integral_constant<int, 9>());
    case 10: return f(std::integral_constant<int, 10>());
    case 11: return f(std::integral_constant<int, 11>());
    case 12: return f(std::integral_constant<int, 12>());
    case 13: return f(std::integral_constant<int, 13>());
    default: return hipErrorInvalidValue;
    }
}
template <typename F>
hipError_t by_lg1(uint32_t lg1, F&& f) {
    switch (lg1) {
    case 11: return f(std::integral_constant<int, 11>());
    case 12: return f(std::integral_constant<int, 12>());
    case 13: return f(std::integral_constant<int, 13>());
    case 14: return f(std::integral_constant<int, 14>());
    case 15: return f(std::integral_constant<int, 15>());
    default: return hipErrorInvalidValue;
    }
}

// Column groups a workgroup of k_mid_fwd walks: 4 at N1 = 2^10 (one workgroup per compute unit), else 2, and
// 1 where that would leave compute units idle or, at N1 <= 2^8, where what the launch writes stays in the
// 256 MB cache (64 blocks of 2^18 bits on a resident seed: 100 us with 1, 103 with 2).  Us a block, in batches of 2^27 bits together, with
// 1 / 2 / 4: 2^19 3.24 / 2.95 / 3.03, 2^20 6.22 / 5.62 / 5.75, 2^22 26.7 / 23.9 / 24.5, 2^24 135 / 124 / 114;
// one block: 2^20 26.0 / 26.5 / 29.0, 2^23 67.6 / 66.2 / 70.3, 2^24 133 / 136 / 127.
static uint32_t mid_walk(const Geom& g, uint32_t operands) {
    const uint64_t groups = (uint64_t)(g.N2 / 16u) * operands;
    const uint32_t w = g.lg1 >= 10u ? 4u : 2u;
    return groups / w >= (g.lg1 >= 10u ? 256u : g.lg1 == 9u ? 512u : 8192u) ? w : 1u;
}

// Column groups of a launch below which the passes of 3 * 2^k give each class a workgroup of its own: fewer
// than two a compute unit leave it idle.  One block of 3000032 bits (128 groups an operand): pass A 19.3 to
// 18.4 us, pass A' 12.1 to 8.1.  From 2048 groups on pass A takes two a workgroup and streams its stores:
// us a block in batches of 2^27 bits together with 1 / 2 / 2 streaming / 4, 2^20 bits 4.53 / 4.40 / 4.26 / 4.50,
// 2^22 17.9 / 17.4 / 16.9 / 17.9, 2^24 75.8 / 72.4 / 70.5 / 75.3; one block of 2^25 bits 185 with 1, 185 streaming,
// 181 with 2.
static bool mix_split(uint64_t groups) { return groups < 512u; }

// Pass A of `count` blocks (bt, BATCH) or one (a); per: see launch_batch_fwd_cols.
template <bool BATCH>
hipError_t fwd_cols(FwdArgs a, const Geom& g, const Tables& t, uint32_t per, uint32_t scan_wgs, const BlockArgs* bt,
                    uint32_t count, hipStream_t s) {
    if (mixed(g))
        return by_classes(g.D, [&](auto d) {
            constexpr int D = decltype(d)::value;
            const uint64_t groups = (uint64_t)(g.N2 / 16u) * a.ops * count;
            auto launch = [&](auto per, uint32_t wgs) {
                a.nA = wgs;
                k_mix_fwd<D, decltype(per)::value, BATCH><<<dim3(wgs * a.ops + scan_wgs, 1, count), 256, 0, s>>>(
                    a, g, t.lo, t.hi, t.cls, bt);
                return hipGetLastError();
            };
            if constexpr (D == 3)
                if (mix_split(groups)) return launch(std::integral_constant<int, 0>(), g.N2 / 16u * D);
            if (groups >= 2048u) return launch(std::integral_constant<int, 2>(), g.N2 / 32u);
            return launch(std::integral_constant<int, 1>(), g.N2 / 16u);
        });
    if (mid_size(g))
        return by_mid_lg1(g.lg1, [&](auto lg) {
            constexpr int LG1 = decltype(lg)::value;
            const uint32_t walk = mid_walk(g, a.ops * count);
            a.nA = g.N2 / 16u / walk;
            const dim3 grid(a.nA * a.ops + scan_wgs, 1, count);
            if (walk > 1u) k_mid_fwd<LG1, BATCH, true><<<grid, mid_threads(LG1), 0, s>>>(a, g, t.tw14, t.lo, t.hi, walk, bt);
            else k_mid_fwd<LG1, BATCH, false><<<grid, mid_threads(LG1), 0, s>>>(a, g, t.tw14, t.lo, t.hi, 1u, bt);
            return hipGetLastError();
        });
    return by_lg1(g.lg1, [&](auto lg) {
        constexpr int LG1 = decltype(lg)::value, LGM = LG1 <= 13 ? 9 : 10, D = 1 << (LG1 - LGM);
        a.nA = g.N2 / 16u * (uint32_t)(D / 2) / per;  // N2 / 16 = 512 groups and per divides it
        k_fwd_cols<LGM, D, BATCH><<<dim3(a.nA * a.ops, 1, count), fwd_cols_threads(LGM), 0, s>>>(a, g, t.tw14, t.lo, t.hi,
                                                                                               t.cls, per, bt);
        return hipGetLastError();
    });
}
template <bool BATCH>
hipError_t mix_inv(const float2* R, const uint32_t* key, uint32_t* out, const Geom& g, const uint32_t* info,
                   const uint32_t* q, const Tables& t, float* margin, const BlockArgs* bt, uint32_t count, hipStream_t s) {
    return by_classes(g.D, [&](auto d) {
        constexpr int D = decltype(d)::value;
        if constexpr (D == 3)
            if (mix_split((uint64_t)(g.N2 / 16u) * count)) {
                k_mix_inv<D, 1, BATCH><<<dim3(g.N2 / 16u * D, 1, count), 256, 0, s>>>(R, key, out, g, info, q, t.lo, t.hi, margin, bt);
                return hipGetLastError();
            }
        k_mix_inv<D, 3, BATCH><<<dim3(g.N2 / 16u * (D / 3), 1, count), 256, 0, s>>>(R, key, out, g, info, q, t.lo, t.hi, margin, bt);
        return hipGetLastError();
    });
}
// Pass A' of `count` blocks (bt, BATCH) or one.
template <bool BATCH>
hipError_t inv_cols(float2* R, uint8_t* nib, const Geom& g, const uint32_t* info, const Tables& t, float* margin,
                    const BlockArgs* bt, uint32_t count, hipStream_t s) {
    return by_lg1(g.lg1, [&](auto lg) {
        constexpr int LG1 = decltype(lg)::value;
        if constexpr (LG1 <= RT_LG1) {
            k_inv_cols<LG1, BATCH><<<dim3(g.N2 / (uint32_t)inv_cols_width(LG1), 1, count), inv_cols_threads(LG1), 0, s>>>(
                R, nib, g, info, t.tw14, t.lo, t.hi, margin, bt);
        } else {
            k_inv_big1<LG1, BATCH><<<dim3(g.N2 / 16u * (g.N1 / 1024u), 1, count), 512, 0, s>>>(R, g, t.tw14, bt);
            k_inv_big2<LG1, BATCH><<<dim3(g.N2 / 16u * 64u, 1, count), 256, 0, s>>>(R, nib, g, info, t.lo, t.hi, margin, bt);
        }
        return hipGetLastError();
    });
}
template <bool BATCH>
hipError_t rows(int mode, float2* Yk, float2* S, float2* Rt, const Geom& g, const Tables& t, uint32_t* info,
                const uint32_t* ws, uint32_t* seed_ws, const BlockArgs* bt, uint32_t count, hipStream_t s) {
    return by_lg2(g.lg2, [&](auto lg) {
        constexpr int LG2 = decltype(lg)::value;
        auto launch = [&](auto rpw) {
            constexpr int RPW = decltype(rpw)::value, NT = rows_threads(LG2, RPW);
            const dim3 grid(g.N1 / (uint32_t)RPW + 1u, 1, count);  // + scan_finish
            switch (mode) {
            case ROWS_STATIC:
                k_rows<LG2, ROWS_STATIC, BATCH, RPW><<<grid, NT, 0, s>>>(Yk, S, Rt, g, t.tw14, t.lo, t.hi, info, ws, seed_ws, bt);
                break;
            case ROWS_DYN:
                k_rows<LG2, ROWS_DYN, BATCH, RPW><<<grid, NT, 0, s>>>(Yk, S, Rt, g, t.tw14, t.lo, t.hi, info, ws, seed_ws, bt);
                break;
            case ROWS_SEEDPREP:
                if constexpr (!BATCH) {
                    k_rows<LG2, ROWS_SEEDPREP, false, RPW><<<grid, NT, 0, s>>>(Yk, S, Rt, g, t.tw14, t.lo, t.hi, info, ws, seed_ws, bt);
                    break;
                }
                [[fallthrough]];
            default: return hipErrorInvalidValue;
            }
            return hipGetLastError();
        };
        if constexpr (BATCH && LG2 < 12)
            if ((uint64_t)g.N1 * count >= 1024u * rows_per_wg_many(LG2)) return launch(std::integral_constant<int, rows_per_wg_many(LG2)>());
        return launch(std::integral_constant<int, rows_per_wg(LG2)>());
    });
}
template <bool BATCH>
hipError_t transpose(const uint32_t* key, const uint32_t* seed, uint32_t* tbk, uint32_t* tbs, uint32_t first, uint32_t ops,
                     const Geom& g, const ScanArgs* scan, uint32_t scan_wgs, const BlockArgs* bt, uint32_t count,
                     hipStream_t s) {
    const dim3 grid(scan_wgs + ops * (g.M << (ROW_LOG - TB_SPAN_LOG)), 1, count);
    const ScanArgs sc = scan ? *scan : ScanArgs{};
    switch (g.D) {
    case 4: k_transpose_bits<4, BATCH><<<grid, TB_NT, 0, s>>>(key, seed, tbk, tbs, first, g, sc, scan_wgs, bt); break;
    case 8: k_transpose_bits<8, BATCH><<<grid, TB_NT, 0, s>>>(key, seed, tbk, tbs, first, g, sc, scan_wgs, bt); break;
    case 16: k_transpose_bits<16, BATCH><<<grid, TB_NT, 0, s>>>(key, seed, tbk, tbs, first, g, sc, scan_wgs, bt); break;
    case 32: k_transpose_bits<32, BATCH><<<grid, TB_NT, 0, s>>>(key, seed, tbk, tbs, first, g, sc, scan_wgs, bt); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
template <int LGN>
hipError_t launch_small_t(const uint32_t* key, const uint32_t* seed, const float2* sspec,
                          const uint32_t* ws_ptr, uint32_t* out, const Geom& g, const Tables& t,
                          float* margin, float2* sspec_out, uint32_t* ws_out, hipStream_t s) {
    if (sspec_out)
        k_small<LGN, true, false><<<1, small_threads(LGN), 0, s>>>(key, seed, sspec, ws_ptr, out, g, t.tw14,
                                                                  margin, sspec_out, ws_out, nullptr);
    else
        k_small<LGN, false, false><<<1, small_threads(LGN), 0, s>>>(key, seed, sspec, ws_ptr, out, g, t.tw14,
                                                                   margin, sspec_out, ws_out, nullptr);
    return hipGetLastError();
}
template <int LGN>
hipError_t batch_small_t(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, hipStream_t s) {
    k_small<LGN, false, true><<<dim3(1, 1, count), small_threads(LGN), 0, s>>>(
        nullptr, nullptr, nullptr, nullptr, nullptr, g0, t.tw14, nullptr, nullptr, nullptr, bt);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_copies(const CopyDesc* d, uint32_t count, uint64_t max_bytes, hipStream_t s) {
    if (count == 0) return hipSuccess;
    const uint64_t chunks = (max_bytes + COPY_CHUNK - 1) / COPY_CHUNK;
    const uint32_t y = (uint32_t)(chunks < 1 ? 1 : (chunks > 32 ? 32 : chunks));
    k_copies<<<dim3(count, y), COPY_NT, 0, s>>>(d);
    return hipGetLastError();
}

hipError_t launch_transpose(const uint32_t* key, const uint32_t* seed, uint32_t* tbk, uint32_t* tbs, uint32_t first,
                            uint32_t ops, const Geom& g, const ScanArgs* scan, hipStream_t s) {
    return transpose<false>(key, seed, tbk, tbs, first, ops, g, scan, scan ? scan_chunks(g) : 0u, nullptr, 1, s);
}

// Column groups a workgroup of pass A walks: 8, fewer while that would leave under 512 workgroups per
// operand (two per compute unit).  Fresh seed: 2^25 265 us with 2 and 4, 273 with 8, 325 with 16; 2^26
// 475 with 4, 485 with 2 and 8; 2^27 891 with 8, 906 with 4, 895 with 16; 2^28 and 2^29 within 1%.
static uint32_t default_walk(const Geom& g, uint32_t count) {
    uint32_t per = 8u;
    while (per > 1u && g.N2 / 16u * (g.D / 2u) / per * count < 512u) per >>= 1;
    return per;
}

hipError_t launch_fwd_cols(const uint32_t* key_in, const uint32_t* seed_in, float2* Yk, float2* Ys, uint32_t first,
                           uint32_t ops, const Geom& g, const Tables& t, const ScanArgs* scan, hipStream_t s) {
    FwdArgs a{{key_in, seed_in}, {Yk, Ys}, first, ops, 0u, scan ? *scan : ScanArgs{}};
    return fwd_cols<false>(a, g, t, default_walk(g, 1), scan ? scan_chunks(g) : 0u, nullptr, 1, s);
}

hipError_t launch_rows(int mode, float2* Yk, float2* S, float2* Rt, const Geom& g, const Tables& t, uint32_t* info,
                       const uint32_t* ws, uint32_t* seed_ws, hipStream_t s) {
    return rows<false>(mode, Yk, S, Rt, g, t, info, ws, seed_ws, nullptr, 1, s);
}

hipError_t launch_prefix_apply(uint32_t* q, const uint32_t* info, const Geom& g, hipStream_t s) {
    k_prefix_apply<<<g.L / 32u / 256u, 256, 0, s>>>(q, info, g);
    return hipGetLastError();
}

hipError_t launch_inv_cols(float2* R, uint8_t* nib, const Geom& g, const uint32_t* info, const Tables& t,
                           float* margin, hipStream_t s) {
    return inv_cols<false>(R, nib, g, info, t, margin, nullptr, 1, s);
}

uint32_t pack_halves(const Geom& g) { return (g.out_off < g.N ? 1u : 0u) + (g.out_off + g.out_bits > g.N ? 1u : 0u); }

hipError_t launch_pack(const uint8_t* nib, const uint32_t* key, uint32_t* out, const Geom& g, const uint32_t* info,
                       const uint32_t* q, hipStream_t s) {
    k_pack<false><<<dim3(g.N2 / 32u / PACK_CW, g.N1 / 256u * pack_halves(g)), PACK_NT, 0, s>>>(nib, key, out, g, info, q, nullptr);
    return hipGetLastError();
}

hipError_t launch_mid_inv(const float2* R, const uint32_t* key, uint32_t* out, const Geom& g, const uint32_t* info,
                          const uint32_t* q, const Tables& t, float* margin, hipStream_t s) {
    if (mixed(g)) return mix_inv<false>(R, key, out, g, info, q, t, margin, nullptr, 1, s);
    return by_mid_lg1(g.lg1, [&](auto lg) {
        constexpr int LG1 = decltype(lg)::value;
        k_mid_inv<LG1, false><<<g.N2 / 16u, mid_threads(LG1), 0, s>>>(R, key, out, g, info, q, t.tw14, margin, nullptr);
        return hipGetLastError();
    });
}

// R output words per workgroup: the fewest instruction slots on the busiest of 256 compute units, R + 1
// per key word (R products and a window).  One block of 2^17 bits: 10.4 us with 6 (the rule's), 11.0 with
// 8, 12.6 with 4, 18.5 with 1; of 2^16 7.4 with 3, 9.4 with 1.
template <bool BATCH>
hipError_t direct(const uint32_t* key, const uint32_t* seed, uint32_t* out, const Geom& g, uint32_t words, uint32_t jpad,
                  const BlockArgs* bt, uint32_t count, hipStream_t s) {
    const uint32_t NT = std::min(DIRECT_NT_MAX, (jpad * 2u + 63u) & ~63u);  // a half-wave per chunk of the key
    uint32_t R = 1;
    uint64_t best = ~0ull;
    for (uint32_t r : {1u, 2u, 3u, 4u, 6u, 8u}) {
        const uint64_t wgs = (uint64_t)(words + r - 1u) / r * count, cost = (wgs + 255u) / 256u * (r + 1u);
        if (cost < best) {
            best = cost;
            R = r;
        }
    }
    const size_t lds = (2u * jpad + 12u) * 4u;
    auto go = [&](auto rc) {
        constexpr int RR = decltype(rc)::value;
        k_direct<RR, BATCH><<<dim3((words + RR - 1u) / RR, 1, count), NT, lds, s>>>(key, seed, out, g, bt);
        return hipGetLastError();
    };
    switch (R) {
    case 1: return go(std::integral_constant<int, 1>());
    case 2: return go(std::integral_constant<int, 2>());
    case 3: return go(std::integral_constant<int, 3>());
    case 4: return go(std::integral_constant<int, 4>());
    case 6: return go(std::integral_constant<int, 6>());
    default: return go(std::integral_constant<int, 8>());
    }
}
hipError_t launch_direct(const uint32_t* key, const uint32_t* seed, uint32_t* out, const Geom& g, hipStream_t s) {
    return direct<false>(key, seed, out, g, g.out_bits >> 5, direct_key_words(g), nullptr, 1, s);
}
hipError_t launch_batch_direct(const BlockArgs* bt, uint32_t count, uint32_t words, uint32_t jpad, hipStream_t s) {
    return direct<true>(nullptr, nullptr, nullptr, Geom{}, words, jpad, bt, count, s);
}

hipError_t launch_small(const uint32_t* key, const uint32_t* seed, const float2* sspec,
                        const uint32_t* ws_ptr, uint32_t* out, const Geom& g, const Tables& t,
                        float* margin, float2* sspec_out, uint32_t* ws_out, hipStream_t s) {
    switch (g.lgN) {
    case 5: return launch_small_t<5>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    case 6: return launch_small_t<6>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    case 7: return launch_small_t<7>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    case 8: return launch_small_t<8>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    case 9: return launch_small_t<9>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    case 10: return launch_small_t<10>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    case 11: return launch_small_t<11>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    case 12: return launch_small_t<12>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    case 13: return launch_small_t<13>(key, seed, sspec, ws_ptr, out, g, t, margin, sspec_out, ws_out, s);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------- batched launchers ----
// `count` blocks of one transform length; block b's geometry and buffers are bt[b] (device
// memory) and g0 is any block's geometry (only its L-derived fields are used here).
hipError_t launch_batch_transpose(const BlockArgs* bt, uint32_t count, const Geom& g0, uint32_t ops, hipStream_t s) {
    return transpose<true>(nullptr, nullptr, nullptr, nullptr, 0u, ops, g0, nullptr, scan_chunks(g0), bt, count, s);
}

hipError_t launch_batch_fwd_cols(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, uint32_t ops,
                                 uint32_t per, hipStream_t s) {
    const uint32_t groups = g0.N2 / 16u;
    if (per == 0u) per = default_walk(g0, count);
    if (per > FWD_PER_MAX || (per & (per - 1u)) != 0u || (!mid_size(g0) && groups % per != 0u)) return hipErrorInvalidValue;
    FwdArgs a{};
    a.ops = ops;
    return fwd_cols<true>(a, g0, t, per, scan_chunks(g0), bt, count, s);
}

hipError_t launch_batch_rows(int mode, const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t,
                             hipStream_t s) {
    return rows<true>(mode, nullptr, nullptr, nullptr, g0, t, nullptr, nullptr, nullptr, bt, count, s);
}

hipError_t launch_batch_inv_cols(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, hipStream_t s) {
    return inv_cols<true>(nullptr, nullptr, g0, nullptr, t, nullptr, bt, count, s);
}

hipError_t launch_batch_pack(const BlockArgs* bt, uint32_t count, const Geom& g0, uint32_t halves, hipStream_t s) {
    k_pack<true><<<dim3(g0.N2 / 32u / PACK_CW, g0.N1 / 256u * halves, count), PACK_NT, 0, s>>>(nullptr, nullptr, nullptr, g0, nullptr,
                                                                                  nullptr, bt);
    return hipGetLastError();
}

hipError_t launch_batch_mid_inv(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, hipStream_t s) {
    if (mixed(g0)) return mix_inv<true>(nullptr, nullptr, nullptr, g0, nullptr, nullptr, t, nullptr, bt, count, s);
    return by_mid_lg1(g0.lg1, [&](auto lg) {
        constexpr int LG1 = decltype(lg)::value;
        k_mid_inv<LG1, true><<<dim3(g0.N2 / 16u, 1, count), mid_threads(LG1), 0, s>>>(nullptr, nullptr, nullptr, g0, nullptr,
                                                                                     nullptr, t.tw14, nullptr, bt);
        return hipGetLastError();
    });
}

hipError_t launch_batch_small(const BlockArgs* bt, uint32_t count, const Geom& g0, const Tables& t, hipStream_t s) {
    switch (g0.lgN) {
    case 5: return batch_small_t<5>(bt, count, g0, t, s);
    case 6: return batch_small_t<6>(bt, count, g0, t, s);
    case 7: return batch_small_t<7>(bt, count, g0, t, s);
    case 8: return batch_small_t<8>(bt, count, g0, t, s);
    case 9: return batch_small_t<9>(bt, count, g0, t, s);
    case 10: return batch_small_t<10>(bt, count, g0, t, s);
    case 11: return batch_small_t<11>(bt, count, g0, t, s);
    case 12: return batch_small_t<12>(bt, count, g0, t, s);
    case 13: return batch_small_t<13>(bt, count, g0, t, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pa

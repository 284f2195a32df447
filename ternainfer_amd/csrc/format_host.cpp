// Host-side producer of the compressed ternary weight format (no GPU work).
//
// The format is the one written by the reference's convert/convert_utils.py:52-228 and
// kernels/TernaSpMM.cu:282-439.  This encoder does not walk the matrix in the reference's
// loop nest; it computes, for every bit of every 8x8 bitmap, which original element it
// stands for:
//   bitmap b of tile T:  band = b / 16, g = (b / 4) % 4, sk = (b / 2) % 2, sm = b % 2
//   bit 8*r + c       :  row = 64*tm + 16*band + 8*sk + r
//                        col = 64*tk + 16*g + 4*(c / 2) + 2*sm + (c % 2)
// which folds the 16x16 block permutation (convert_utils.py:9-49) into the index math.
#include <sched.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <system_error>
#include <thread>
#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include "format_host.h"

namespace terna {

namespace {

inline float bf16_to_float(uint16_t h)
{
    uint32_t u = static_cast<uint32_t>(h) << 16;
    float f;
    std::memcpy(&f, &u, sizeof f);
    return f;
}

// The encoders below work on tile rows (64 matrix rows) [tm0, tm1): `sign_words` is where the range's own stream starts,
// tile_off[tile + 1] receives the position (in bits, from that start) behind each tile.  Return: sign words written,
// or -1 for a value outside {-1, 0, 1}.

// Any element type: `at(row, col)` returns <0, 0 or >0 for the element of the ORIGINAL matrix.
template <typename At>
int64_t encode_range(At at, int K, int tm0, int tm1, uint64_t* bitmap, int* tile_off, uint16_t* median_off,
                     uint32_t* sign_words)
{
    const int tiles_k = K / 64;
    int64_t pos = 0;                     // next free sign bit, always a multiple of 32 at tile start
    int64_t tile = static_cast<int64_t>(tm0) * tiles_k;
    for (int tm = tm0; tm < tm1; ++tm) {
        for (int tk = 0; tk < tiles_k; ++tk, ++tile) {
            const int64_t tile_start = pos;
            uint64_t word = 0;           // sign word being filled
            for (int b = 0; b < 64; ++b) {
                const int band = b >> 4, g = (b >> 2) & 3, sk = (b >> 1) & 1, sm = b & 1;
                if (b && (b & 15) == 0) median_off[3 * tile + band - 1] = static_cast<uint16_t>(pos - tile_start);
                const int row0 = 64 * tm + 16 * band + 8 * sk;
                const int col0 = 64 * tk + 16 * g + 2 * sm;
                uint64_t bits = 0;
                for (int r = 0; r < 8; ++r) {
                    for (int c = 0; c < 8; ++c) {
                        const int v = at(row0 + r, col0 + 4 * (c >> 1) + (c & 1));
                        if (v == 0) continue;
                        bits |= 1ull << (8 * r + c);
                        if (v < 0) word |= 1ull << (pos & 31);
                        if ((++pos & 31) == 0) {
                            sign_words[(pos >> 5) - 1] = static_cast<uint32_t>(word);
                            word = 0;
                        }
                    }
                }
                bitmap[tile * 64 + b] = bits;
            }
            if (pos & 31) {              // zero-pad the tile's stream to a whole word
                sign_words[pos >> 5] = static_cast<uint32_t>(word);
                pos = (pos | 31) + 1;
            }
            tile_off[tile + 1] = static_cast<int>(pos);
        }
    }
    return pos >> 5;
}

#if defined(__x86_64__)
#define TERNA_ENCODE_AVX2 1
#define TERNA_AVX2 __attribute__((target("avx2,bmi,bmi2,popcnt")))

// 8 x 8 bytes: byte r of out[j] = byte j of in[r].
TERNA_AVX2 inline void transpose_bytes(const uint64_t in[8], uint64_t out[8])
{
    const __m128i* p = reinterpret_cast<const __m128i*>(in);
    __m128i r[4], t[4];
    for (int i = 0; i < 4; ++i) r[i] = _mm_loadu_si128(p + i);
    for (int i = 0; i < 4; ++i) t[i] = _mm_unpacklo_epi8(r[i], _mm_unpackhi_epi64(r[i], r[i]));   // rows 2i, 2i + 1 by columns
    const __m128i a = _mm_unpacklo_epi16(t[0], t[1]), b = _mm_unpackhi_epi16(t[0], t[1]);          // rows 0 .. 3
    const __m128i c = _mm_unpacklo_epi16(t[2], t[3]), d = _mm_unpackhi_epi16(t[2], t[3]);          // rows 4 .. 7
    __m128i* q = reinterpret_cast<__m128i*>(out);
    _mm_storeu_si128(q + 0, _mm_unpacklo_epi32(a, c));
    _mm_storeu_si128(q + 1, _mm_unpackhi_epi32(a, c));
    _mm_storeu_si128(q + 2, _mm_unpacklo_epi32(b, d));
    _mm_storeu_si128(q + 3, _mm_unpackhi_epi32(b, d));
}

// Bound: reading the matrix.  A 64-column row of a tile becomes two 64-bit masks (nonzero, negative): the bytes of every
// 16 columns are shuffled so that the eight columns of bitmap sm = 0 come first, so byte 2g + sm of a mask is the row's byte
// of bitmap (g, sm), and eight rows are one 8 x 8 byte transposition away from eight bitmaps.  A bitmap's sign bits are the
// negative mask's bits at its set bits (pext), appended 64 at a time.  One core: 13824 x 2560 in 107 ms bit by bit
// (encode_range), 12 ms this way, most of it first touches of the output; 2.4 ms with tile rows spread over eight cores.
TERNA_AVX2 int64_t encode_range_avx2(const int8_t* W, int K, int tm0, int tm1, uint64_t* bitmap, int* tile_off,
                                     uint16_t* median_off, uint32_t* sign_words)
{
    const int tiles_k = K / 64;
    const __m256i order = _mm256_setr_epi8(0, 1, 4, 5, 8, 9, 12, 13, 2, 3, 6, 7, 10, 11, 14, 15,
                                           0, 1, 4, 5, 8, 9, 12, 13, 2, 3, 6, 7, 10, 11, 14, 15);
    const __m256i zero = _mm256_setzero_si256(), one = _mm256_set1_epi8(1);
    __m256i largest = zero;              // of w + 1 as an unsigned byte: at most 2 for a ternary matrix
    uint32_t* out = sign_words;
    int64_t tile = static_cast<int64_t>(tm0) * tiles_k;
    for (int tm = tm0; tm < tm1; ++tm) {
        for (int tk = 0; tk < tiles_k; ++tk, ++tile) {
            const int8_t* w = W + static_cast<int64_t>(64) * tm * K + 64 * tk;
            uint64_t acc = 0;            // sign bits not stored yet
            int fill = 0, count = 0;
            for (int band = 0; band < 4; ++band) {
                uint64_t nz[2][8], ng[2][8];
                for (int sk = 0; sk < 2; ++sk) {
                    uint64_t zrow[8], nrow[8];
                    for (int r = 0; r < 8; ++r, w += K) {
                        const __m256i lo = _mm256_loadu_si256(reinterpret_cast<const __m256i*>(w));
                        const __m256i hi = _mm256_loadu_si256(reinterpret_cast<const __m256i*>(w + 32));
                        largest = _mm256_max_epu8(largest, _mm256_max_epu8(_mm256_add_epi8(lo, one), _mm256_add_epi8(hi, one)));
                        const __m256i l = _mm256_shuffle_epi8(lo, order), h = _mm256_shuffle_epi8(hi, order);
                        const uint32_t zl = _mm256_movemask_epi8(_mm256_cmpeq_epi8(l, zero)), zh = _mm256_movemask_epi8(_mm256_cmpeq_epi8(h, zero));
                        const uint32_t nl = _mm256_movemask_epi8(l), nh = _mm256_movemask_epi8(h);
                        zrow[r] = ~(zl | static_cast<uint64_t>(zh) << 32);
                        nrow[r] = nl | static_cast<uint64_t>(nh) << 32;
                    }
                    transpose_bytes(zrow, nz[sk]);
                    transpose_bytes(nrow, ng[sk]);
                }
                if (band) median_off[3 * tile + band - 1] = static_cast<uint16_t>(count);
                uint64_t* bm = bitmap + tile * 64 + 16 * band;
                for (int b = 0; b < 16; ++b) {
                    const int sk = (b >> 1) & 1, j = 2 * (b >> 2) + (b & 1);
                    const uint64_t bits = nz[sk][j];
                    bm[b] = bits;
                    const uint64_t sign = _pext_u64(ng[sk][j], bits);
                    const int n = static_cast<int>(_mm_popcnt_u64(bits));
                    count += n;
                    acc |= sign << fill;
                    fill += n;
                    if (fill >= 64) {
                        std::memcpy(out, &acc, 8);
                        out += 2;
                        fill -= 64;
                        acc = fill ? sign >> (n - fill) : 0;
                    }
                }
            }
            if (fill > 32) { std::memcpy(out, &acc, 8); out += 2; }      // the tile's stream ends on a whole word
            else if (fill > 0) { std::memcpy(out, &acc, 4); out += 1; }
            tile_off[tile + 1] = static_cast<int>(32 * (out - sign_words));
        }
    }
    const __m256i two = _mm256_set1_epi8(2);
    if (_mm256_movemask_epi8(_mm256_cmpeq_epi8(_mm256_max_epu8(largest, two), two)) != -1) return -1;
    return out - sign_words;
}
#endif

int64_t encode_rows(const int8_t* W, int K, int tm0, int tm1, uint64_t* bitmap, int* tile_off, uint16_t* median_off,
                    uint32_t* sign_words)
{
#ifdef TERNA_ENCODE_AVX2
    static const bool avx2 = __builtin_cpu_supports("avx2") && __builtin_cpu_supports("bmi2") && __builtin_cpu_supports("popcnt");
    if (avx2) return encode_range_avx2(W, K, tm0, tm1, bitmap, tile_off, median_off, sign_words);
#endif
    for (int64_t e = static_cast<int64_t>(64) * tm0 * K; e < static_cast<int64_t>(64) * tm1 * K; ++e)
        if (W[e] < -1 || W[e] > 1) return -1;
    auto at = [=](int row, int col) -> int { return W[static_cast<int64_t>(row) * K + col]; };
    return encode_range(at, K, tm0, tm1, bitmap, tile_off, median_off, sign_words);
}

// Cores for one call: OMP_NUM_THREADS where it is set (what torch and the machine's owner go by), else those the process
// may run on, at most 16; and a megaweight (0.25 ms of work) for each.
int encode_threads(int64_t weights, int tile_rows)
{
    int cores = 0;
    if (const char* env = std::getenv("OMP_NUM_THREADS")) cores = std::atoi(env);
    if (cores < 1) {
        cpu_set_t set;
        cores = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
    }
    const int64_t most = std::min<int64_t>({cores, 16, weights >> 20, tile_rows});
    return static_cast<int>(std::max<int64_t>(most, 1));
}

}  // namespace

int encode_sizes(int N, int K, int64_t* bitmap_len, int64_t* tile_off_len, int64_t* median_len,
                 int64_t* sign_words_capacity)
{
    if (N <= 0 || K <= 0 || N % 64 || K % 64) return -1;
    const int64_t nk = static_cast<int64_t>(N) * K;
    if (bitmap_len) *bitmap_len = nk / 64;
    if (tile_off_len) *tile_off_len = nk / 4096 + 1;
    if (median_len) *median_len = 3 * (nk / 4096);
    if (sign_words_capacity) *sign_words_capacity = nk / 32;
    return 0;
}

// Every thread encodes a run of tile rows into the part of `sign_words` that the worst case would give it (the caller's
// buffer has room for all weights nonzero); then the streams move together, first to last, and the offsets get their base.
int64_t encode_i8(const int8_t* W, int N, int K, uint64_t* bitmap, int* tile_off, uint16_t* median_off,
                  uint32_t* sign_words)
{
    if (N <= 0 || K <= 0 || N % 64 || K % 64) return -1;
    const int rows = N / 64, tiles_k = K / 64;
    const int threads = encode_threads(static_cast<int64_t>(N) * K, rows);
    tile_off[0] = 0;
    if (threads == 1) return encode_rows(W, K, 0, rows, bitmap, tile_off, median_off, sign_words);

    const auto first = [=](int t) { return static_cast<int>(static_cast<int64_t>(rows) * t / threads); };
    const auto room = [=](int t) { return sign_words + static_cast<int64_t>(first(t)) * tiles_k * 128; };
    int64_t words[16];
    const auto work = [&](int t) { words[t] = encode_rows(W, K, first(t), first(t + 1), bitmap, tile_off, median_off, room(t)); };
    std::thread pool[16];
    int started = 0;
    try {
        for (int t = 1; t < threads; ++t, ++started) pool[t] = std::thread(work, t);
    } catch (const std::system_error&) {}                    // no more threads to be had: the rest is done here
    work(0);
    for (int t = started + 1; t < threads; ++t) work(t);
    for (int t = 1; t <= started; ++t) pool[t].join();

    int64_t total = 0;
    for (int t = 0; t < threads; ++t) {
        if (words[t] < 0) return -1;
        if (t) std::memmove(sign_words + total, room(t), 4 * words[t]);
        const int base = static_cast<int>(32 * total);
        for (int64_t tile = static_cast<int64_t>(first(t)) * tiles_k; base && tile < static_cast<int64_t>(first(t + 1)) * tiles_k; ++tile)
            tile_off[tile + 1] += base;
        total += words[t];
    }
    return total;
}

int64_t encode_reordered_bf16(const uint16_t* A, int N, int K, uint64_t* bitmap, int* tile_off,
                              uint16_t* median_off, uint32_t* sign_words, int* max_padded_nnz)
{
    if (N <= 0 || K <= 0 || N % 64 || K % 64) return -1;
    // The caller hands over the matrix AFTER the 16x16 permutation; map original (row, col)
    // to where the permutation put it:  i' = (i&7) + 8*((k>>1)&1),  k' = 8*(i>>3) + 2*(k>>2) + (k&1).
    auto at = [=](int row, int col) -> int {
        const int i = row & 15, k = col & 15;
        const int ri = (i & 7) + 8 * ((k >> 1) & 1);
        const int rk = 8 * (i >> 3) + 2 * (k >> 2) + (k & 1);
        const float f = bf16_to_float(A[static_cast<int64_t>((row & ~15) + ri) * K + (col & ~15) + rk]);
        return f < 0.0f ? -1 : (f != 0.0f ? 1 : 0);
    };
    tile_off[0] = 0;
    const int64_t words = encode_range(at, K, 0, N / 64, bitmap, tile_off, median_off, sign_words);
    *max_padded_nnz = 0;
    for (int64_t tile = 0; tile < static_cast<int64_t>(N / 64) * (K / 64); ++tile)
        *max_padded_nnz = std::max(*max_padded_nnz, tile_off[tile + 1] - tile_off[tile]);
    return words;
}

void reorder_bf16(const uint16_t* W, uint16_t* out, int N, int K)
{
    for (int row = 0; row < N; ++row) {
        const int i = row & 15;
        for (int col = 0; col < K; ++col) {
            const int k = col & 15;
            const int ri = (i & 7) + 8 * ((k >> 1) & 1);
            const int rk = 8 * (i >> 3) + 2 * (k >> 2) + (k & 1);
            out[static_cast<int64_t>((row & ~15) + ri) * K + (col & ~15) + rk] = W[static_cast<int64_t>(row) * K + col];
        }
    }
}

}  // namespace terna

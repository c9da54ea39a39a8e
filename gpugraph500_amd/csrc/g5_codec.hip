// g5_codec.hip -- s4-bp128-d4 on the device, word-for-word the stream that
// CompositeCodec<SIMDBinaryPacking<SIMDIntegratedBlockPacker<CoarseDelta4SIMD,
// true>>, VariableByte<true>> writes (cpu_2d/compression/cpusimd/include/
// codecfactory.h:103-105) into a 16-byte aligned buffer.
//
// Stream (uint32 words):
//   [L = n/128*128, 123456, 123456, 123456]            simdbinarypacking.h:182-183
//   per group of <= 16 miniblocks of 128 values:
//     4 header words, 8-bit widths MSB first            simdbinarypacking.h:195-202
//     per miniblock 4*b words: 4-strided deltas d[k] = x[k] - x[k-4]
//     (x[-4..-1] = previous miniblock's last values, 0 at the start),
//     value k in lane k&3 at bit (k>>2)*b of that lane's word stream;
//     b = 32 stores the raw values, b = 0 stores nothing
//   varint tail of n - L values, deltas restarting at 0, 7-bit groups LSB
//   first, stop bit on the last byte, zero padded to a word (variablebyte.h).
//
// Encode is two launches and decode four to nine, a hop table more for every
// factor of 8 in the groups, so that a level's queue costs launches in proportion
// to what depends on what (short queues, below, one):
//   k_enc_sizes   widths and, per workgroup's miniblocks, their word total
//   k_enc_write   each workgroup adds up the totals before its own, packs its
//                 miniblocks (each lane assembles whole output words from the
//                 deltas staged in LDS, so stores are coalesced and need no
//                 atomics); one more workgroup writes the varint tail
//   k_dec_hop, k_dec_hop8, k_dec_anchors
//                 the group headers: their positions depend on all earlier
//                 widths.  Every word index 4 + 4i is a candidate group start
//                 (groups are 4 + 4 * sum(widths) words); a thread per
//                 candidate follows 8 headers, then tables of 8 hops of the
//                 table before (64, 512, ... groups), until few enough groups
//                 are left for one thread to walk; the walk is then refined
//                 table by table down to every 8th group
//   k_dec_sums    each workgroup finds its miniblocks (at most 7 headers from
//                 an anchor) and their running-sum record: the 4-lane sums
//                 across miniblocks compose as (reset, sums), where b = 32
//                 miniblocks reset the running value to their raw last values
//   k_dec_values  each workgroup composes the records before its own, unpacks
//                 and writes; one more workgroup decodes the varint tail
// Results and counts go to pinned host memory from the last kernel, without a
// copy of their own.  A queue of at most kSmallValues values takes each of
// encode, decode and round trip in one workgroup (k_enc_small, k_dec_small,
// k_rt_small), with the stream in LDS for the decode.
// Latency bounds both: 3001 values encode and decode in 5.7 + 7.3 us of kernels
// (37 us with the calls' launches and waits; 14 launches, three copies and a
// serial tail took 86 us), 7 M values in 31 + 84 us (133 us; 25 launches, a
// serial walk over every 32nd group and a serial tail 234 us).
#include <algorithm>

#include "g5_codec.hpp"

namespace {

constexpr uint32_t kCookie = 123456u;
constexpr int kTile = 64;           // miniblocks a workgroup holds at a time
constexpr int kTileThreads = 512;
constexpr int kTileWaves = kTileThreads / 64;
constexpr int kPerWave = kTile / kTileWaves;
constexpr int64_t kMaxTiles = 1024;  // every workgroup reads the totals before its own

// the miniblocks of a workgroup: whole tiles, at most kMaxTiles workgroups
int64_t per_group(int64_t nblk)
{
    const int64_t tiles = (nblk + kTile - 1) / kTile;
    return std::max<int64_t>(1, (tiles + kMaxTiles - 1) / kMaxTiles) * kTile;
}

struct Carry {
    uint32_t r, v[4];
};

__device__ __forceinline__ Carry comb(const Carry &a, const Carry &b)
{
    if (b.r) return b;
    Carry c = a;
#pragma unroll
    for (int j = 0; j < 4; ++j) c.v[j] += b.v[j];
    return c;
}

// LDS written by some lanes of a wave, then read by others
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// inclusive sum over the lanes of a wave
__device__ __forceinline__ uint32_t scan32(uint32_t v, int l)
{
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(v, d, 64);
        if (l >= d) v += t;
    }
    return v;
}

// ------------------------------------------------------------------ encode

// one miniblock in a wave's registers: lane l holds values l and l + 64 and
// the values 4 before them
struct Mini {
    uint32_t x0, x1, r0, r1;
};

__device__ __forceinline__ Mini load_mini(const uint32_t *__restrict__ in, int64_t i, int l)
{
    const int64_t base = i * 128;
    Mini m;
    m.x0 = in[base + l];
    m.x1 = in[base + l + 64];
    m.r0 = (base + l >= 4) ? in[base + l - 4] : 0u;
    m.r1 = in[base + l + 60];
    return m;
}

// bits of the widest of the wave's values: 6 ballots (a shuffle reduction's 6
// LDS round trips took longer)
__device__ __forceinline__ uint32_t wave_width(uint32_t acc)
{
    uint32_t w = 0;
#pragma unroll
    for (int s = 16; s >= 1; s >>= 1)
        if (__ballot(acc >> s)) {
            acc >>= s;
            w += s;
        }
    return w + (__ballot(acc) ? 1u : 0u);
}

__device__ __forceinline__ uint32_t mini_width(const Mini &m) { return wave_width((m.x0 - m.r0) | (m.x1 - m.r1)); }

// Positions of a tile's miniblocks: s_pos[k] = base + 4 * (widths before k);
// one wave; returns the tile's words
__device__ __forceinline__ uint32_t enc_positions(const uint8_t *s_w, int64_t base, int64_t *s_pos, int l)
{
    const uint32_t w = 4u * s_w[l], inc = scan32(w, l);
    s_pos[l] = base + inc - w;
    return __shfl(inc, 63, 64);
}

// The group headers of a tile whose first miniblock is i0 (a multiple of 64):
// 16 words, one wave
__device__ __forceinline__ void enc_headers(int64_t i0, int cnt, const uint8_t *s_w, const int64_t *s_pos,
                                            uint32_t *__restrict__ out, int l)
{
    if (l < 16 && 16 * (l >> 2) < cnt) {
        uint32_t w = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) w |= (uint32_t)s_w[4 * l + t] << (24 - 8 * t);  // zero past the last miniblock
        const int64_t g = (i0 >> 4) + (l >> 2);
        out[4 + 4 * g + s_pos[16 * (l >> 2)] + (l & 3)] = w;
    }
}

// One miniblock's packed words: one wave, lds = 128 words of its own
__device__ __forceinline__ void enc_pack(const Mini &m, uint32_t b, uint32_t *__restrict__ dst, uint32_t *lds, int l)
{
    if (b == 32) {
        dst[l] = m.x0;
        dst[l + 64] = m.x1;
        return;
    }
    if (b == 0) return;
    lds[l] = m.x0 - m.r0;
    lds[l + 64] = m.x1 - m.r1;
    wave_sync();
    // x / b for x < 1056 and b < 32: x * inv is less than x / 65536 < 1 / 32
    // too large in units of 1
    const uint32_t inv = 65536u / b + 1;
    for (uint32_t t = l; t < 4 * b; t += 64) {
        const uint32_t j = t & 3, lo = 32 * (t >> 2);
        uint32_t word = 0;
        const uint32_t i0 = lo * inv >> 16;
        uint32_t i1 = (lo + 31) * inv >> 16;
        if (i1 > 31) i1 = 31;
        for (uint32_t idx = i0; idx <= i1; ++idx) {
            const int sh = (int)(idx * b) - (int)lo;
            const uint32_t v = lds[4 * idx + j];
            word |= sh >= 0 ? (v << sh) : (v >> (-sh));
        }
        dst[t] = word;
    }
    wave_sync();  // lds is reused by the wave's next miniblock
}

__device__ __forceinline__ uint32_t varint_len(uint32_t v)
{
    return v < (1u << 7) ? 1u : v < (1u << 14) ? 2u : v < (1u << 21) ? 3u : v < (1u << 28) ? 4u : 5u;
}

constexpr int kTailBytes = 128 * 5 + 8;

// stream header + varint tail; one wave (every lane calls it), pn = the
// miniblocks' word total, bytes = kTailBytes of LDS; returns the stream's
// word count
__device__ int64_t enc_tail_wave(const uint32_t *__restrict__ in, int64_t n, int64_t L, int64_t nblk, int64_t pn,
                                 uint32_t *__restrict__ out, uint8_t *bytes, int l)
{
    if (l == 0) {
        out[0] = (uint32_t)L;
        out[1] = out[2] = out[3] = kCookie;
    }
    const int64_t tailpos = 4 + 4 * ((nblk + 15) / 16) + pn;
    const int64_t nt = n - L;
    if (nt == 0) return tailpos;
    for (int k = l; k < kTailBytes; k += 64) bytes[k] = 0;
    wave_sync();
    uint32_t run = 0;
    for (int r = 0; r < 2; ++r) {
        const int k = l + 64 * r;
        uint32_t v = 0, len = 0;
        if (k < nt) {
            v = in[L + k] - (k ? in[L + k - 1] : 0u);
            len = varint_len(v);
        }
        const uint32_t inc = scan32(len, l);
        uint32_t pos = run + inc - len;
        for (uint32_t q = 0; q < len; ++q) {
            const uint32_t last = (q + 1 == len);
            bytes[pos + q] = (uint8_t)(((v >> (7 * q)) & 127u) | (last ? 128u : 0u));
        }
        run += __shfl(inc, 63, 64);
    }
    wave_sync();
    const uint32_t nw = (run + 3) / 4;
    for (uint32_t w = l; w < nw; w += 64)
        out[tailpos + w] = (uint32_t)bytes[4 * w] | ((uint32_t)bytes[4 * w + 1] << 8) |
                           ((uint32_t)bytes[4 * w + 2] << 16) | ((uint32_t)bytes[4 * w + 3] << 24);
    return tailpos + nw;
}

// widths of the workgroup's miniblocks [blockIdx * per, ...) and their words
__global__ __launch_bounds__(kTileThreads) void k_enc_sizes(const uint32_t *__restrict__ in, int64_t nblk,
                                                            int64_t per, uint8_t *__restrict__ width,
                                                            int64_t *__restrict__ total)
{
    __shared__ int64_t s_sum[kTileWaves];
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int64_t first = blockIdx.x * per, last = min(nblk, first + per);
    int64_t sum = 0;
    constexpr int U = 4;  // miniblocks in flight per wave
    for (int64_t i0 = first + wv; i0 < last; i0 += U * kTileWaves) {
        Mini m[U] = {};
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (i0 + k * kTileWaves < last) m[k] = load_mini(in, i0 + k * kTileWaves, l);
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const uint32_t w = mini_width(m[k]);
            if (i0 + k * kTileWaves < last) {
                if (l == 0) width[i0 + k * kTileWaves] = (uint8_t)w;
                sum += 4 * w;
            }
        }
    }
    if (l == 0) s_sum[wv] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t t = 0;
        for (int k = 0; k < kTileWaves; ++k) t += s_sum[k];
        total[blockIdx.x] = t;
    }
}

// sum of total[0 .. n), every thread of the workgroup gets it
__device__ __forceinline__ int64_t sum_before(const int64_t *__restrict__ total, int64_t n)
{
    __shared__ int64_t s_part[kTileWaves];
    int64_t t = 0;
    for (int64_t i = threadIdx.x; i < n; i += kTileThreads) t += total[i];
    t = g5_wave_sum(t);
    if (__lane_id() == 0) s_part[threadIdx.x >> 6] = t;
    __syncthreads();
    t = 0;
    for (int k = 0; k < kTileWaves; ++k) t += s_part[k];
    return t;
}

// Workgroup 0: stream header, varint tail and the stream's length (to nw_out
// and, when given, host memory); workgroup 1 + t: the miniblocks
// [t * per, ...).
__global__ __launch_bounds__(kTileThreads) void k_enc_write(const uint32_t *__restrict__ in, int64_t n, int64_t nblk,
                                                            int64_t per, const uint8_t *__restrict__ width,
                                                            const int64_t *__restrict__ total,
                                                            uint32_t *__restrict__ out, int64_t *__restrict__ nw_out,
                                                            int64_t *__restrict__ host)
{
    __shared__ uint8_t s_bytes[kTailBytes];
    __shared__ uint8_t s_w[kTile];
    __shared__ int64_t s_pos[kTile], s_run;
    __shared__ uint32_t s_d[kTileWaves][128];
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (blockIdx.x == 0) {
        const int64_t pn = sum_before(total, gridDim.x - 1);
        if (wv == 0) {
            const int64_t nw = enc_tail_wave(in, n, nblk * 128, nblk, pn, out, s_bytes, l);
            if (l == 0) {
                *nw_out = nw;
                if (host) *host = nw;
            }
        }
        return;
    }
    const int64_t t = blockIdx.x - 1, first = t * per, last = min(nblk, first + per);
    const int64_t before = sum_before(total, t);
    if (threadIdx.x == 0) s_run = before;
    for (int64_t i0 = first; i0 < last; i0 += kTile) {
        const int cnt = (int)min((int64_t)kTile, last - i0);
        // the next miniblocks' values on their way while positions are found
        Mini m[kPerWave] = {};
#pragma unroll
        for (int k = 0; k < kPerWave; ++k)
            if (wv + k * kTileWaves < cnt) m[k] = load_mini(in, i0 + wv + k * kTileWaves, l);
        if (wv == 0) s_w[l] = l < cnt ? width[i0 + l] : (uint8_t)0;
        __syncthreads();
        if (wv == 0) {
            const int64_t run = s_run;
            const uint32_t words = enc_positions(s_w, run, s_pos, l);
            wave_sync();
            enc_headers(i0, cnt, s_w, s_pos, out, l);
            if (l == 0) s_run = run + words;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPerWave; ++k) {
            const int q = wv + k * kTileWaves;
            if (q < cnt) enc_pack(m[k], s_w[q], out + 8 + 4 * ((i0 + q) >> 4) + s_pos[q], s_d[wv], l);
        }
        __syncthreads();  // s_w and s_pos are rewritten by the next tile
    }
}

// ------------------------------------------------------------------ decode

enum { kMetaL = 0, kMetaGroups = 1, kMetaTailPos = 2, kMetaErr = 3, kMetaTail = 4, kMetaBig = 5, kMetaFlag = 6,
       kMetaNw = 7, kMetaSlots = 8 };

// errors: 1 cookie, 2 the header's L, 3 a width, 4 truncated, 5 more values
// than the capacity
constexpr int32_t kBadWidth = -1, kTruncated = -2;
__device__ __forceinline__ int64_t err_of(int32_t code) { return code == kBadWidth ? 3 : 4; }

// Word position after the group whose header is at p and which holds cnt
// miniblocks (16 but for the stream's last), or kBadWidth / kTruncated if
// there can be none.
__device__ __forceinline__ int64_t after_group(const uint32_t *__restrict__ in, int64_t nwords, int64_t p, int cnt)
{
    if (p + 4 > nwords) return kTruncated;
    int64_t size = 4;
    bool ok = true;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint32_t x = in[p + w];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t b = (x >> (24 - 8 * k)) & 0xFF;
            if (4 * w + k < cnt) {
                ok = ok && b <= 32;
                size += 4 * b;
            }
        }
    }
    if (!ok) return kBadWidth;
    return p + size <= nwords ? p + size : (int64_t)kTruncated;
}

constexpr int kHopLog = 3;      // every table takes 8 hops of the one before
constexpr int kMaxTables = 6;
constexpr int64_t kTopWalk = 16;  // groups the last table leaves to one thread

// hop[i] = the candidate 8 groups after candidate i (word 4 + 4i)
__global__ __launch_bounds__(256) void k_dec_hop(const uint32_t *__restrict__ in, const int64_t *__restrict__ nwp,
                                                 int64_t nwv, int64_t bound, int32_t *__restrict__ hop)
{
    const int64_t nwords = nwp ? *nwp : nwv, ncand = min(bound, (nwords - 4) / 4 + 1);
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < ncand; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t p = 4 + 4 * i;
        for (int k = 0; k < (1 << kHopLog) && p >= 0; ++k) p = after_group(in, nwords, p, 16);
        hop[i] = p < 0 ? (int32_t)p : (int32_t)((p - 4) / 4);
    }
}

// out[i] = 8 hops of `in` from i (errors propagate)
__global__ __launch_bounds__(256) void k_dec_hop8(const int32_t *__restrict__ in, const int64_t *__restrict__ nwp,
                                                  int64_t nwv, int64_t bound, int32_t *__restrict__ out)
{
    const int64_t ncand = min(bound, ((nwp ? *nwp : nwv) - 4) / 4 + 1);
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < ncand; i += (int64_t)gridDim.x * blockDim.x) {
        int32_t a = (int32_t)i;
        for (int k = 0; k < (1 << kHopLog) && a >= 0; ++k) a = a < ncand ? in[a] : kTruncated;
        out[i] = a;
    }
}

struct HopTables {
    const int32_t *t[kMaxTables];
    int n;
};

// One workgroup: the decoder's record is cleared and gets L and the group
// count, after the stream header's checks; anchor[k] = candidate index of
// group 8k, k = 0..(ngroups-1)/8.  Hops from anchor to anchor only cross
// groups before the last one, whose unused widths are not read.
__global__ __launch_bounds__(256) void k_dec_anchors(const uint32_t *__restrict__ in, int64_t cap,
                                                     const int64_t *__restrict__ nwp, int64_t nwv, int64_t bound,
                                                     HopTables hops, int32_t *__restrict__ anchor,
                                                     int64_t *__restrict__ meta)
{
    __shared__ int64_t s_err, s_na;
    const int64_t ncand = min(bound, ((nwp ? *nwp : nwv) - 4) / 4 + 1);
    if (threadIdx.x < kMetaSlots) meta[threadIdx.x] = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int64_t L = in[0], ngroups = (L / 128 + 15) / 16;
        int64_t err = 0;
        if (in[1] != kCookie || in[2] != kCookie || in[3] != kCookie) err = 1;
        if (L % 128 != 0 || L > cap) err = 2;
        if (!err && ngroups > ncand) err = 4;  // more groups than possible starts: truncated
        meta[kMetaL] = L;
        meta[kMetaGroups] = ngroups;
        if (!err && ngroups == 0) meta[kMetaTailPos] = 4;
        const int64_t na = err || ngroups == 0 ? 0 : ((ngroups - 1) >> kHopLog) + 1;  // anchors
        if (na) {
            const int64_t stride = (int64_t)1 << (kHopLog * (hops.n - 1));  // the last table's hop, in anchors
            const int32_t *hop = hops.t[hops.n - 1];
            int32_t a = 0;
            for (int64_t k = 0;; k += stride) {
                anchor[k] = a;
                if (k + stride >= na) break;
                a = a < ncand ? hop[a] : kTruncated;
                if (a < 0) {
                    err = err_of(a);
                    break;
                }
            }
        }
        s_err = err;
        s_na = na;
    }
    __syncthreads();
    const int64_t na = s_na;
    for (int t = hops.n - 2; t >= 0 && na; --t) {
        const bool good = s_err == 0;
        __syncthreads();  // every thread has looked before one sets it below
        if (!good) break;
        const int64_t step = (int64_t)1 << (kHopLog * t);  // anchors from one new anchor to the next
        const int64_t from = step << kHopLog;              // and between the known ones
        for (int64_t k = threadIdx.x * from; k < na; k += blockDim.x * from) {
            int32_t a = anchor[k];
            for (int j = 1; j < (1 << kHopLog) && k + j * step < na; ++j) {
                a = a < ncand ? hops.t[t][a] : kTruncated;
                if (a < 0) {
                    s_err = err_of(a);
                    break;
                }
                anchor[k + j * step] = a;
            }
        }
        __syncthreads();  // also orders the anchors within the workgroup
    }
    if (threadIdx.x == 0 && s_err) meta[kMetaErr] = s_err;
}

// A tile's miniblocks: their widths and data positions from the positions of
// its (at most 4) group headers; one wave, lane = miniblock.
__device__ __forceinline__ void dec_places(const uint32_t *__restrict__ in, const int64_t *s_grp, int cnt,
                                           uint8_t *s_w, int64_t *s_off, int l)
{
    uint32_t w = 0;
    const int64_t hp = 16 * (l >> 4) < cnt ? s_grp[l >> 4] : 0;
    if (l < cnt) w = (in[hp + ((l & 15) >> 2)] >> (24 - 8 * (l & 3))) & 0xFF;
    uint32_t inc = w;  // within the group's 16 lanes
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) {
        const uint32_t t = __shfl_up(inc, d, 16);
        if ((l & 15) >= d) inc += t;
    }
    s_w[l] = (uint8_t)w;
    s_off[l] = hp + 4 + 4 * (int64_t)(inc - w);
}

// Miniblock of width b at o: lane l's deltas (b < 32) or values (b = 32) l
// and l + 64
__device__ __forceinline__ void dec_fetch(const uint32_t *__restrict__ in, int64_t o, uint32_t b, int l, uint32_t &d0,
                                          uint32_t &d1)
{
    if (b == 32) {
        d0 = in[o + l];
        d1 = in[o + l + 64];
        return;
    }
    d0 = d1 = 0;
    if (b == 0) return;
    const uint32_t j = l & 3;
    uint32_t d[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t bit = ((l >> 2) + 16 * h) * b, w = bit >> 5, sh = bit & 31;
        uint64_t v = in[o + 4 * w + j];
        if (sh + b > 32) v |= (uint64_t)in[o + 4 * (w + 1) + j] << 32;
        d[h] = (uint32_t)(v >> sh) & ((1u << b) - 1);
    }
    d0 = d[0];
    d1 = d[1];
}

// The records of a tile composed from its left, one wave, lane = miniblock:
// s_c[k] becomes what precedes miniblock k (start included), the return value
// what follows the tile
__device__ __forceinline__ Carry dec_compose(Carry *s_c, int cnt, const Carry &start, int l)
{
    Carry c{0, {0, 0, 0, 0}};
    if (l < cnt) c = s_c[l];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        Carry p;
        p.r = __shfl_up(c.r, d, 64);
#pragma unroll
        for (int j = 0; j < 4; ++j) p.v[j] = __shfl_up(c.v[j], d, 64);
        if (l >= d) c = comb(p, c);
    }
    const Carry all = comb(start, c);
    Carry ex, end;
    ex.r = __shfl_up(all.r, 1, 64);
    end.r = __shfl(all.r, 63, 64);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        ex.v[j] = __shfl_up(all.v[j], 1, 64);
        end.v[j] = __shfl(all.v[j], 63, 64);
    }
    s_c[l] = l == 0 ? start : ex;
    return end;
}

// Workgroup t: the group positions and the composed record of the miniblocks
// [t * per, ...); the tail's position from the last group.
__global__ __launch_bounds__(kTileThreads) void k_dec_sums(const uint32_t *__restrict__ in,
                                                           const int64_t *__restrict__ nwp, int64_t nwv, int64_t per,
                                                           const int32_t *__restrict__ anchor,
                                                           int64_t *__restrict__ grp, Carry *__restrict__ rec,
                                                           int64_t *__restrict__ meta)
{
    __shared__ int64_t s_grp[kTile / 16], s_off[kTile], s_err;
    __shared__ uint8_t s_w[kTile];
    __shared__ Carry s_c[kTile], s_run;
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int64_t nwords = nwp ? *nwp : nwv;
    const int64_t nblk = meta[kMetaL] / 128, ngroups = meta[kMetaGroups];
    const int64_t first = blockIdx.x * per, last = min(nblk, first + per);
    if (threadIdx.x == 0) {
        s_run = Carry{0, {0, 0, 0, 0}};
        s_err = meta[kMetaErr];
    }
    __syncthreads();
    const bool good = s_err == 0;
    __syncthreads();  // every thread has looked before one sets it below
    if (!good) return;
    for (int64_t i0 = first; i0 < last; i0 += kTile) {
        const int cnt = (int)min((int64_t)kTile, last - i0);
        if (wv == 0) {
            const int64_t g = (i0 >> 4) + l;
            if (l < kTile / 16 && g < ngroups) {
                int64_t p = 4 + 4 * (int64_t)anchor[g >> kHopLog];
                for (int k = (int)(g & ((1 << kHopLog) - 1)); k > 0 && p >= 0; --k) p = after_group(in, nwords, p, 16);
                const int64_t e = p < 0 ? p : after_group(in, nwords, p, (int)min((int64_t)16, nblk - 16 * g));
                if (e < 0) {
                    s_err = err_of((int32_t)e);
                    atomicMax((unsigned long long *)&meta[kMetaErr], (unsigned long long)err_of((int32_t)e));
                } else {
                    s_grp[l] = p;
                    grp[g] = p;
                    if (g == ngroups - 1) meta[kMetaTailPos] = e;
                }
            }
        }
        __syncthreads();
        if (s_err) break;
        if (wv == 0) dec_places(in, s_grp, cnt, s_w, s_off, l);
        __syncthreads();
        uint32_t d0[kPerWave], d1[kPerWave];
#pragma unroll
        for (int k = 0; k < kPerWave; ++k) {
            const int q = wv + k * kTileWaves;
            d0[k] = d1[k] = 0;
            if (q < cnt) dec_fetch(in, s_off[q], s_w[q], l, d0[k], d1[k]);
        }
#pragma unroll
        for (int k = 0; k < kPerWave; ++k) {
            const int q = wv + k * kTileWaves;
            if (q >= cnt) break;
            const bool raw = s_w[q] == 32;
            // raw values: the last four; deltas: sums over lanes of the same class
            uint32_t s = raw ? d1[k] : d0[k] + d1[k];
            if (!raw) {
                s += __shfl_xor(s, 4, 64);
                s += __shfl_xor(s, 8, 64);
                s += __shfl_xor(s, 16, 64);
                s += __shfl_xor(s, 32, 64);
            }
            if (l >= 60) s_c[q].v[l - 60] = s;
            if (l == 60) s_c[q].r = raw ? 1u : 0u;
        }
        __syncthreads();
        if (wv == 0) {
            const Carry end = dec_compose(s_c, cnt, s_run, l);
            wave_sync();
            if (l == 0) s_run = end;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0 && first < last) rec[blockIdx.x] = s_run;
}

// Varint values that start at byte position 0 of the nb bytes at bi, deltas
// from 0, to out (at most cap values); one wave.  Returns the values there
// are; more than cap: -1, after cap were written.
__device__ int64_t dec_tail_wave(const uint8_t *bi, int64_t nb, int64_t cap, uint32_t *__restrict__ out, int l)
{
    int64_t o = 0, start = 0;  // values written, the byte after the last stop
    uint32_t prev = 0;
    for (int64_t q0 = 0; q0 < nb; q0 += 64) {
        const int64_t q = q0 + l;
        const uint32_t c = q < nb ? bi[q] : 0u;
        const uint64_t stops = __ballot((c & 128u) != 0);
        const uint64_t lower = stops & ((1ull << l) - 1);
        // the bytes of the value that stops here; a stream's values have at
        // most 5, more bytes shift out (and in again, as the shifts count
        // modulo 32)
        const int64_t b = lower ? q0 + 64 - __clzll((long long)lower) : start;
        uint32_t v = 0;
        if (c & 128u)
            for (int64_t k = b; k <= q; ++k) v += (uint32_t)(bi[k] & 127u) << ((7 * (k - b)) & 31);
        const uint32_t inc = scan32(v, l);
        const int64_t at = o + __popcll(lower);
        if ((c & 128u) && at < cap) out[at] = prev + inc;
        o += __popcll(stops);
        prev += __shfl(inc, 63, 64);
        if (stops) start = q0 + 64 - __clzll((long long)stops);
        if (o > cap) return -1;
    }
    return o;
}

// The end of a decode, one wave: the tail's values and the record, to
// device memory and, when given, the host's.  n_expect (round trip; else < 0):
// the record's flag slot, or flag when given (never a slot of the record), is
// set to 1 unless the stream held exactly that many values.
__device__ void dec_finish(const uint8_t *stream, int64_t nwords, int64_t err, int64_t L,
                           int64_t tailpos, int64_t cap, uint32_t *__restrict__ out, int64_t n_expect,
                           int64_t *__restrict__ flag, int64_t *__restrict__ meta, int64_t *__restrict__ host, int l)
{
    int64_t n = 0;
    if (!err) {
        n = dec_tail_wave(stream + 4 * tailpos, (nwords - tailpos) * 4, cap - L, out + L, l);
        if (n < 0) {
            err = 5;
            n = 0;
        }
    }
    if (l == 0) {
        const int64_t lost = n_expect >= 0 && (err || L + n != n_expect);
        if (lost && flag) *flag = 1;
        meta[kMetaFlag] = lost;
        meta[kMetaErr] = err;
        meta[kMetaTail] = n;
        meta[kMetaNw] = nwords;
        if (host) {
            host[kMetaL] = L;
            host[kMetaErr] = err;
            host[kMetaTail] = n;
            host[kMetaBig] = 0;
            host[kMetaFlag] = lost;
            host[kMetaNw] = nwords;
        }
    }
}

// Workgroup 0: the varint tail and the record; workgroup 1 + t: the values of
// the miniblocks [t * per, ...).
__global__ __launch_bounds__(kTileThreads) void k_dec_values(const uint32_t *__restrict__ in,
                                                             const int64_t *__restrict__ nwp, int64_t nwv,
                                                             int64_t per, const int64_t *__restrict__ grp,
                                                             const Carry *__restrict__ rec, int64_t cap,
                                                             uint32_t *__restrict__ out, int64_t n_expect,
                                                             int64_t *__restrict__ flag, int64_t *__restrict__ meta,
                                                             int64_t *__restrict__ host)
{
    __shared__ int64_t s_grp[kTile / 16], s_off[kTile];
    __shared__ uint8_t s_w[kTile];
    __shared__ Carry s_c[kTile], s_run;
    __shared__ int s_last;
    __shared__ uint32_t s_sum[4];
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int64_t err = meta[kMetaErr], L = meta[kMetaL];
    if (blockIdx.x == 0) {
        if (wv == 0)
            dec_finish((const uint8_t *)in, nwp ? *nwp : nwv, err, L, meta[kMetaTailPos], cap, out, n_expect, flag,
                       meta, host, l);
        return;
    }
    // workgroup 0 may set err 5 meanwhile: the tail did not fit, the
    // miniblocks do, and either way they are written as far as they go
    if (err && err != 5) return;
    const int64_t nblk = L / 128, ngroups = meta[kMetaGroups];
    const int64_t t = blockIdx.x - 1, first = t * per, last = min(nblk, first + per);
    if (first >= last) return;
    // what precedes the workgroup: the sums since the last reset
    if (threadIdx.x == 0) s_last = -1;
    if (threadIdx.x < 4) s_sum[threadIdx.x] = 0;
    __syncthreads();
    int reset = -1;
    for (int k = threadIdx.x; k < t; k += kTileThreads)
        if (rec[k].r) reset = k;
    if (reset >= 0) atomicMax(&s_last, reset);
    __syncthreads();
    const int from = s_last;
    uint32_t sum[4] = {0, 0, 0, 0};
    for (int k = threadIdx.x; k < t; k += kTileThreads)
        if (k >= from)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[j] += rec[k].v[j];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) sum[j] += __shfl_xor(sum[j], d, 64);
        if (l == 0 && sum[j]) atomicAdd(&s_sum[j], sum[j]);
    }
    __syncthreads();
    if (threadIdx.x == 0) s_run = Carry{0, {s_sum[0], s_sum[1], s_sum[2], s_sum[3]}};
    for (int64_t i0 = first; i0 < last; i0 += kTile) {
        const int cnt = (int)min((int64_t)kTile, last - i0);
        if (wv == 0) {
            if (l < kTile / 16 && (i0 >> 4) + l < ngroups) s_grp[l] = grp[(i0 >> 4) + l];
            wave_sync();
            dec_places(in, s_grp, cnt, s_w, s_off, l);
        }
        __syncthreads();
        uint32_t d0[kPerWave], d1[kPerWave];
#pragma unroll
        for (int k = 0; k < kPerWave; ++k) {
            const int q = wv + k * kTileWaves;
            d0[k] = d1[k] = 0;
            if (q < cnt) dec_fetch(in, s_off[q], s_w[q], l, d0[k], d1[k]);
        }
#pragma unroll
        for (int k = 0; k < kPerWave; ++k) {
            const int q = wv + k * kTileWaves;
            if (q >= cnt) break;
            const bool raw = s_w[q] == 32;
            if (!raw) {
                // inclusive sums over lanes of the same class (stride 4), the
                // second half after the first
#pragma unroll
                for (int dist = 4; dist < 64; dist <<= 1) {
                    const uint32_t a = __shfl_up(d0[k], dist, 64), b = __shfl_up(d1[k], dist, 64);
                    if (l >= dist) {
                        d0[k] += a;
                        d1[k] += b;
                    }
                }
                d1[k] += __shfl(d0[k], 60 + (l & 3), 64);
            }
            if (l >= 60) s_c[q].v[l - 60] = d1[k];
            if (l == 60) s_c[q].r = raw ? 1u : 0u;
        }
        __syncthreads();
        if (wv == 0) {
            const Carry end = dec_compose(s_c, cnt, s_run, l);
            wave_sync();
            if (l == 0) s_run = end;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPerWave; ++k) {
            const int q = wv + k * kTileWaves;
            if (q >= cnt) break;
            const uint32_t c = s_w[q] == 32 ? 0u : s_c[q].v[l & 3];
            out[128 * (i0 + q) + l] = c + d0[k];
            out[128 * (i0 + q) + l + 64] = c + d1[k];
        }
        __syncthreads();  // s_c, s_w and s_off are rewritten by the next tile
    }
}

// ---- short queues in one workgroup ----
// At most one tile of miniblocks: one launch, no position tables.  The decode
// works on a copy of the stream in LDS.
constexpr int64_t kSmallValues = kTile * 128;
// the longest stream of that many values (g5_s4_max_words)
constexpr int64_t kSmallWords = 4 + 4 * (kTile / 16) + kTile * 128 + 160;

struct EncSmall {
    uint8_t bytes[kTailBytes];
    uint8_t w[kTile];
    int64_t pos[kTile];
    uint32_t d[kTileWaves][128];
    int64_t packed, nw;  // the miniblocks' words, the stream's
};

// n <= kSmallValues; returns the stream's length to every thread
__device__ __forceinline__ int64_t enc_small(const uint32_t *in, int64_t n, uint32_t *__restrict__ out,
                                             EncSmall &s)
{
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int cnt = (int)(n / 128);
    if (cnt == 0) {  // a tail alone
        if (wv == 0) {
            const int64_t nw = enc_tail_wave(in, n, 0, 0, 0, out, s.bytes, l);
            if (l == 0) s.nw = nw;
        }
        __syncthreads();
        return s.nw;
    }
    Mini m[kPerWave] = {};
#pragma unroll
    for (int k = 0; k < kPerWave; ++k)
        if (wv + k * kTileWaves < cnt) m[k] = load_mini(in, wv + k * kTileWaves, l);
#pragma unroll
    for (int k = 0; k < kPerWave; ++k) {
        const uint32_t w = mini_width(m[k]);  // 0 past the last miniblock
        if (l == 0) s.w[wv + k * kTileWaves] = (uint8_t)w;
    }
    __syncthreads();
    if (wv == 0) {
        const uint32_t words = enc_positions(s.w, 0, s.pos, l);
        wave_sync();
        enc_headers(0, cnt, s.w, s.pos, out, l);
        if (l == 0) s.packed = words;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPerWave; ++k) {
        const int q = wv + k * kTileWaves;
        if (q < cnt) enc_pack(m[k], s.w[q], out + 8 + 4 * (q >> 4) + s.pos[q], s.d[wv], l);
    }
    if (wv == kTileWaves - 1) {  // the wave with the fewest miniblocks
        const int64_t nw = enc_tail_wave(in, n, (int64_t)cnt * 128, cnt, s.packed, out, s.bytes, l);
        if (l == 0) s.nw = nw;
    }
    __syncthreads();
    return s.nw;
}

__global__ __launch_bounds__(kTileThreads) void k_enc_small(const uint32_t *__restrict__ in, int64_t n,
                                                            uint32_t *__restrict__ out, int64_t *__restrict__ nw_out,
                                                            int64_t *__restrict__ host)
{
    __shared__ EncSmall s;
    const int64_t nw = enc_small(in, n, out, s);
    if (threadIdx.x == 0) {
        *nw_out = nw;
        if (host) *host = nw;
    }
}

struct DecSmall {
    uint32_t words[kSmallWords];
    int64_t grp[kTile / 16], off[kTile];
    uint8_t w[kTile];
    Carry c[kTile];
    int64_t err, tailpos;
};

// A stream of nwords <= kSmallWords words.  More miniblocks than a tile (the
// words do not tell): nothing is written, and the record says so (kMetaBig).
__device__ __forceinline__ void dec_small(const uint32_t *in, int64_t nwords, int64_t cap, uint32_t *out,
                                          int64_t n_expect, int64_t *__restrict__ flag, int64_t *__restrict__ meta,
                                          int64_t *__restrict__ host, DecSmall &s)
{
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    for (int64_t k = threadIdx.x; k < nwords; k += kTileThreads) s.words[k] = in[k];
    __syncthreads();
    const int64_t L = s.words[0];
    int64_t err = 0;
    if (s.words[1] != kCookie || s.words[2] != kCookie || s.words[3] != kCookie) err = 1;
    if (L % 128 != 0 || L > cap) err = 2;
    if (!err && L > kSmallValues) {
        if (threadIdx.x == 0) {
            meta[kMetaBig] = 1;
            if (host) {
                host[kMetaErr] = 0;
                host[kMetaBig] = 1;
            }
        }
        return;
    }
    const int cnt = err ? 0 : (int)(L / 128);
    if (threadIdx.x == 0) {
        int64_t p = 4;
        for (int g = 0; 16 * g < cnt && !err; ++g) {
            s.grp[g] = p;
            p = after_group(s.words, nwords, p, min(16, cnt - 16 * g));
            if (p < 0) err = err_of((int32_t)p);
        }
        s.err = err;
        s.tailpos = p;
    }
    __syncthreads();
    err = s.err;
    if (!err && cnt) {
        if (wv == 0) dec_places(s.words, s.grp, cnt, s.w, s.off, l);
        __syncthreads();
        uint32_t d0[kPerWave], d1[kPerWave];
#pragma unroll
        for (int k = 0; k < kPerWave; ++k) {
            const int q = wv + k * kTileWaves;
            d0[k] = d1[k] = 0;
            if (q >= cnt) break;
            dec_fetch(s.words, s.off[q], s.w[q], l, d0[k], d1[k]);
            const bool raw = s.w[q] == 32;
            if (!raw) {
#pragma unroll
                for (int dist = 4; dist < 64; dist <<= 1) {
                    const uint32_t a = __shfl_up(d0[k], dist, 64), b = __shfl_up(d1[k], dist, 64);
                    if (l >= dist) {
                        d0[k] += a;
                        d1[k] += b;
                    }
                }
                d1[k] += __shfl(d0[k], 60 + (l & 3), 64);
            }
            if (l >= 60) s.c[q].v[l - 60] = d1[k];
            if (l == 60) s.c[q].r = raw ? 1u : 0u;
        }
        __syncthreads();
        if (wv == 0) (void)dec_compose(s.c, cnt, Carry{0, {0, 0, 0, 0}}, l);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPerWave; ++k) {
            const int q = wv + k * kTileWaves;
            if (q >= cnt) break;
            const uint32_t c = s.w[q] == 32 ? 0u : s.c[q].v[l & 3];
            out[128 * q + l] = c + d0[k];
            out[128 * q + l + 64] = c + d1[k];
        }
    }
    if (wv == kTileWaves - 1)
        dec_finish((const uint8_t *)s.words, nwords, err, L, s.tailpos, cap, out, n_expect, flag, meta, host, l);
}

__global__ __launch_bounds__(kTileThreads) void k_dec_small(const uint32_t *__restrict__ in, int64_t nwords,
                                                            int64_t cap, uint32_t *__restrict__ out,
                                                            int64_t *__restrict__ meta, int64_t *__restrict__ host)
{
    __shared__ DecSmall s;
    dec_small(in, nwords, cap, out, -1, nullptr, meta, host, s);
}

// encode, then decode from the words the encode wrote to memory, as a
// receiver would
__global__ __launch_bounds__(kTileThreads) void k_rt_small(const uint32_t *in, int64_t n, uint32_t *words,
                                                           int64_t *__restrict__ nw_out, uint32_t *out,
                                                           int64_t *__restrict__ meta, int64_t *__restrict__ flag,
                                                           int64_t *__restrict__ host)
{
    __shared__ EncSmall se;
    __shared__ DecSmall sd;
    const int64_t nw = enc_small(in, n, words, se);
    if (threadIdx.x == 0) *nw_out = nw;
    // enc_small's last barrier lets the workgroup's other waves read the words
    dec_small(words, nw, n, out, n, flag, meta, host, sd);
}

// the tables that bring `groups` groups down to kTopWalk for one thread
int hop_tables(int64_t groups)
{
    int t = 1;
    while (t < kMaxTables && (groups >> (kHopLog * t)) > kTopWalk) ++t;
    return t;
}

}  // namespace

namespace g5 {

size_t S4Codec::bind(uint8_t *base, int64_t n)
{
    const int64_t nblk = n / 128 + 2;
    const int64_t ngrp = nblk / 16 + 2;
    const int64_t ncand = (int64_t)g5_s4_max_words((size_t)n) / 4 + 2;
    const int nhop = hop_tables(ngrp);
    size_t off = 0;
    // pieces start 256 B apart from each other
    auto take = [&](size_t bytes) -> uint8_t * {
        uint8_t *p = base ? base + off : nullptr;
        off += (bytes + 255) / 256 * 256;
        return p;
    };
    uint8_t *width = take((size_t)nblk);
    uint8_t *total = take((size_t)(kMaxTiles + 1) * 8);
    uint8_t *rec = take((size_t)(kMaxTiles + 1) * sizeof(Carry));
    uint8_t *grp = take((size_t)ngrp * 8);
    uint8_t *anchor = take((size_t)(ngrp / (1 << kHopLog) + 2) * 4);
    uint8_t *hop[kMaxTables] = {};
    for (int t = 0; t < nhop; ++t) hop[t] = take((size_t)ncand * 4);
    uint8_t *meta = take(16 * 8);
    uint8_t *nw = take(2 * 8);
    if (base) {
        d_base = base;
        d_width = width;
        d_total = (int64_t *)total;
        d_rec = rec;
        d_grp = (int64_t *)grp;
        d_anchor = (int32_t *)anchor;
        static_assert(kMaxTables == sizeof(d_hop) / sizeof(d_hop[0]), "hop tables");
        for (int t = 0; t < kMaxTables; ++t) d_hop[t] = (int32_t *)hop[t];
        d_meta = (int64_t *)meta;
        d_nw = (int64_t *)nw;
        ncand_cap = ncand;
        hop_cap = nhop;
        cap = n;
    }
    return off;
}

int S4Codec::reserve(int64_t n)
{
    if (n <= cap && d_meta) return G5_OK;
    release();
    uint8_t *base = nullptr;
    hipError_t e = hipMalloc(&base, bind(nullptr, n));
    if (e == hipSuccess) e = hipHostMalloc(&h_meta, 16 * 8, hipHostMallocDefault);
    if (e != hipSuccess) {
        if (base) (void)hipFree(base);
        h_meta = nullptr;
        return fail_hip(e, "S4Codec::reserve", __FILE__, __LINE__);
    }
    bind(base, n);
    owned = true;
    return G5_OK;
}

void S4Codec::release()
{
    if (owned) {
        if (d_base) (void)hipFree(d_base);
        if (h_meta) (void)hipHostFree(h_meta);
        h_meta = nullptr;
    }
    owned = false;
    d_base = nullptr;
    d_width = nullptr;
    d_rec = nullptr;
    d_total = d_grp = d_meta = nullptr;
    d_anchor = nullptr;
    for (int32_t *&h : d_hop) h = nullptr;
    d_nw = nullptr;
    ncand_cap = 0;
    hop_cap = 0;
    cap = 0;
}

// the encode kernels; the stream's word count goes to d_nw[0] and, when
// given, pinned host memory
int S4Codec::encode_launch(const uint32_t *d_in, int64_t n, uint32_t *d_out, int64_t *host, hipStream_t s)
{
    if (n <= kSmallValues) {
        hipLaunchKernelGGL(k_enc_small, 1, kTileThreads, 0, s, d_in, n, d_out, d_nw, host);
        G5_HIP(hipGetLastError());
        return G5_OK;
    }
    const int64_t nblk = n / 128, per = per_group(nblk);
    const unsigned grid = (unsigned)((nblk + per - 1) / per);
    hipLaunchKernelGGL(k_enc_sizes, grid, kTileThreads, 0, s, d_in, nblk, per, d_width, d_total);
    hipLaunchKernelGGL(k_enc_write, grid + 1, kTileThreads, 0, s, d_in, n, nblk, per, (const uint8_t *)d_width,
                       (const int64_t *)d_total, d_out, d_nw, host);
    G5_HIP(hipGetLastError());
    return G5_OK;
}

int S4Codec::encode(const uint32_t *d_in, int64_t n, uint32_t *d_out, size_t cap_words, size_t *nwords,
                    hipStream_t s)
{
    G5_REQUIRE(n >= 0 && cap_words >= g5_s4_max_words((size_t)n), G5_E_OVERFLOW,
               "s4 encode: output capacity %zu below the bound for %lld values", cap_words, (long long)n);
    int rc = reserve(n);
    if (rc) return rc;
    if (acct) G5_HIP(acct->start());
    rc = encode_launch(d_in, n, d_out, h_meta, s);
    if (rc) return rc;
    if (acct) G5_HIP(acct->stop());
    G5_HIP(hipStreamSynchronize(s));
    *nwords = (size_t)h_meta[0];
    if (acct) G5_HIP(acct->commit(G5_UNIT_ENCODE, 4.0 * (double)n + 4.0 * (double)*nwords, 1));
    return G5_OK;
}

// The decode kernels of a stream whose word count is *nwp on the device (or
// nwv, when nwp is null) and at most words_bound: the values to d_out, the
// record to d_meta and, when given, pinned host memory.
int S4Codec::decode_launch(const uint32_t *d_in, const int64_t *nwp, int64_t nwv, int64_t words_bound,
                           int64_t cap_values, uint32_t *d_out, int64_t n_expect, int64_t *d_flag, int64_t *host,
                           hipStream_t s)
{
    const int64_t ncand = (words_bound - 4) / 4 + 1;  // bound on the 4-word group starts
    // bounds on the stream's miniblocks: the capacity's, and 16 per start
    const int64_t nblk = std::min(cap_values / 128, 16 * ncand);
    const int64_t ngroups = (nblk + 15) / 16;
    // a stream longer than one of cap_values values can be has its groups in
    // the words one can have; what is beyond is the tail
    const int64_t nuse = std::min(ncand, ncand_cap);
    HopTables hops{};
    hops.n = std::min(hop_tables(ngroups), hop_cap);
    const unsigned grid = (unsigned)grid_for(nuse, 256, 16384);
    for (int t = 0; t < hops.n; ++t) {
        if (t == 0)
            hipLaunchKernelGGL(k_dec_hop, grid, 256, 0, s, d_in, nwp, nwv, nuse, d_hop[0]);
        else
            hipLaunchKernelGGL(k_dec_hop8, grid, 256, 0, s, (const int32_t *)d_hop[t - 1], nwp, nwv, nuse, d_hop[t]);
        hops.t[t] = d_hop[t];
    }
    hipLaunchKernelGGL(k_dec_anchors, 1, 256, 0, s, d_in, cap_values, nwp, nwv, nuse, hops, d_anchor, d_meta);
    const int64_t per = per_group(nblk);
    const unsigned tiles = (unsigned)((nblk + per - 1) / per);
    if (tiles)
        hipLaunchKernelGGL(k_dec_sums, tiles, kTileThreads, 0, s, d_in, nwp, nwv, per, (const int32_t *)d_anchor,
                           d_grp, (Carry *)d_rec, d_meta);
    hipLaunchKernelGGL(k_dec_values, tiles + 1, kTileThreads, 0, s, d_in, nwp, nwv, per, (const int64_t *)d_grp,
                       (const Carry *)d_rec, cap_values, d_out, n_expect, d_flag, d_meta, host);
    G5_HIP(hipGetLastError());
    return G5_OK;
}

int S4Codec::decode(const uint32_t *d_in, size_t nwords, uint32_t *d_out, size_t cap_values, size_t *n,
                    hipStream_t s)
{
    G5_REQUIRE(nwords >= 4, G5_E_STREAM, "s4 decode: stream of %zu words has no header", nwords);
    int rc = reserve((int64_t)cap_values);
    if (rc) return rc;
    if (acct) G5_HIP(acct->start());
    bool small = (int64_t)nwords <= kSmallWords;
    if (small) {
        hipLaunchKernelGGL(k_dec_small, 1, kTileThreads, 0, s, d_in, (int64_t)nwords, (int64_t)cap_values, d_out,
                           d_meta, h_meta);
        G5_HIP(hipGetLastError());
        if (acct) G5_HIP(acct->stop());
        G5_HIP(hipStreamSynchronize(s));
        if (h_meta[kMetaBig]) {  // few words, many miniblocks
            small = false;
            if (acct) {
                G5_HIP(acct->commit(G5_UNIT_DECODE, 0, 0));
                G5_HIP(acct->start());
            }
        }
    }
    if (!small) {
        rc = decode_launch(d_in, nullptr, (int64_t)nwords, (int64_t)nwords, (int64_t)cap_values, d_out, -1, nullptr,
                           h_meta, s);
        if (rc) return rc;
        if (acct) G5_HIP(acct->stop());
        G5_HIP(hipStreamSynchronize(s));
    }
    const int64_t err = h_meta[kMetaErr];
    if (err && acct) G5_HIP(acct->commit(G5_UNIT_DECODE, 0, 0));
    G5_REQUIRE(err == 0 || err == 5, G5_E_STREAM, "s4 decode: malformed stream (code %lld)", (long long)err);
    G5_REQUIRE(err == 0, G5_E_OVERFLOW, "s4 decode: output capacity %zu exceeded", cap_values);
    *n = (size_t)(h_meta[kMetaL] + h_meta[kMetaTail]);
    if (acct) G5_HIP(acct->commit(G5_UNIT_DECODE, 4.0 * (double)nwords + 4.0 * (double)*n, 1));
    return G5_OK;
}

int S4Codec::roundtrip(const uint32_t *d_in, int64_t n, uint32_t *d_words_out, size_t cap_words, uint32_t *d_out,
                       int64_t *d_flag, hipStream_t s)
{
    G5_REQUIRE(n >= 0 && cap_words >= g5_s4_max_words((size_t)n), G5_E_OVERFLOW,
               "s4 round trip: word capacity %zu below the bound for %lld values", cap_words, (long long)n);
    int rc = reserve(n);
    if (rc) return rc;
    // the record goes home when it is asked for (a borrowed layout has no pinned memory)
    int64_t *host = owned && !d_flag ? h_meta : nullptr;
    if (n <= kSmallValues) {
        hipLaunchKernelGGL(k_rt_small, 1, kTileThreads, 0, s, d_in, n, d_words_out, d_nw, d_out, d_meta, d_flag,
                           host);
        G5_HIP(hipGetLastError());
        return G5_OK;
    }
    rc = encode_launch(d_in, n, d_words_out, nullptr, s);
    if (rc) return rc;
    // the stream's length stays on the device; sizes the host needs follow from n
    return decode_launch(d_words_out, d_nw, 0, (int64_t)g5_s4_max_words((size_t)n), n, d_out, n, d_flag, host, s);
}

int S4Codec::roundtrip_result(size_t *nwords, const char *who)
{
    if (owned) G5_HIP(hipStreamSynchronize(nullptr));
    else G5_HIP(hipMemcpy(h_meta, d_meta, 8 * 8, hipMemcpyDeviceToHost));
    G5_REQUIRE(h_meta[kMetaFlag] == 0, G5_E_STREAM, "%s: the decoded stream lost values", who);
    *nwords = (size_t)h_meta[kMetaNw];
    return G5_OK;
}

}  // namespace g5

namespace {
g5::S4Codec &abi_codec()
{
    static thread_local g5::S4Codec c;
    return c;
}
}  // namespace

extern "C" size_t g5_s4_max_words(size_t n)
{
    const size_t L = n / 128 * 128;
    return 4 + 4 * ((L + 2047) / 2048) + L + (5 * (n - L) + 3) / 4;
}

extern "C" int g5_s4_encode(const uint32_t *d_in, size_t n, uint32_t *d_out, size_t out_cap, size_t *nwords)
{
    G5_REQUIRE((d_in || n == 0) && d_out && nwords, G5_E_ARG, "g5_s4_encode: null argument");
    G5_REQUIRE(((uintptr_t)d_out & 15) == 0, G5_E_ARG, "g5_s4_encode: output must be 16-byte aligned");
    g5::ExchangeTimer t(nullptr);
    g5::S4Codec &c = abi_codec();
    c.acct = &t;
    const int rc = c.encode(d_in, (int64_t)n, d_out, out_cap, nwords, nullptr);
    c.acct = nullptr;
    return rc;
}

extern "C" int g5_s4_decode(const uint32_t *d_in, size_t nwords, uint32_t *d_out, size_t out_cap, size_t *n)
{
    G5_REQUIRE(d_in && (d_out || out_cap == 0) && n, G5_E_ARG, "g5_s4_decode: null argument");
    g5::ExchangeTimer t(nullptr);
    g5::S4Codec &c = abi_codec();
    c.acct = &t;
    const int rc = c.decode(d_in, nwords, d_out, out_cap, n, nullptr);
    c.acct = nullptr;
    return rc;
}

extern "C" int g5_s4_roundtrip(const uint32_t *d_in, size_t n, uint32_t *d_words, size_t cap_words, uint32_t *d_out,
                               size_t *nwords)
{
    G5_REQUIRE(d_in && d_words && d_out && nwords, G5_E_ARG, "g5_s4_roundtrip: null argument");
    g5::S4Codec &c = abi_codec();
    int rc = c.reserve((int64_t)n);
    if (rc) return rc;
    // the flag lives in the decoder's record, which the decode writes
    rc = c.roundtrip(d_in, (int64_t)n, d_words, cap_words, d_out, nullptr, nullptr);
    if (rc) return rc;
    return c.roundtrip_result(nwords, "g5_s4_roundtrip");
}

// int4_planes.hip -- the grouped-INT4 GEMM (matmul_int4_grouped(_ordered),
// tv/quantization/int4.tkv:195-239) of prefill batches on the INT8 matrix
// units, exactly.
//
//   y[m, n] = fl32(sum_k a[m, k] * ((nibble - 8) * scale[n, k / gs]) + bias[n])
//
// with the sums in f64.  On v_mfma_f64_16x16x4_f64 that is bound by the f64
// matrix rate (78.6 TFLOP/s, 1/64 of the INT8 rate).  Here every activation
// becomes a fixed-point integer of up to 8 base-256 digits, and each digit
// plane is multiplied by the 4-bit codes with v_mfma_i32_32x32x32_i8:
//
//   unit   64 rows x 128 k of A.  E = (exponent of the unit's largest |a|) - 5;
//          a = 2^(E - 56) X with X a 62-bit integer: exact for every element
//          down to 2^-38 of the unit's maximum (f32 has 24 bits), and
//          X = sum_p d_p 256^(7 - p), -128 <= d_p <= 127, |d_0| <= 64.
//          Trailing planes that are zero in the whole unit are neither
//          written nor multiplied: the planes of a unit go in pairs, np of
//          them (Gaussian activations: 3 of the 4).
//   pair   P = 256 S_hi + S_lo, S = sum over <= 128 k of one group of
//          digit * 16 (nibble - 8): exact in INT32 (|S| <= 2^21).
//   fold   acc += P * (scale * 2^w) with one f64 fma per pair and group: the
//          product is rounded once, with the sum.
// So all sums inside a group are exact, and an output sees np roundings per
// group (the f64 MFMA form: one per element and group).  Units that hold an
// infinity, a NaN or an element below 2^-38 of the maximum that is not a
// multiple of 2^(E - 56) are flagged, and so are 64 columns x 128 k of W with a
// scale that is not finite (0 * scale is NaN then, also where every activation
// is zero, and the digits of one product may carry either sign).  The
// workgroups whose rows or columns meet a flag run that chunk of K on the f64
// MFMA instead.
//
// k_int4_planes writes A's digits and W's codes as MFMA fragments (1 KB per
// 32 rows x 32 k, in lane order), so that the GEMM copies them to LDS with
// linear DMA and reads them without address arithmetic or bank conflicts.
#include <algorithm>

#include "tkv_device.h"
#include "tkv_internal.h"

namespace tkv {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int kUnitRows = 64, kUnitK = 128;
constexpr int kMaxPairs = 4;
constexpr int kSlot = 16384;                    // a pair: 2 planes x 64 rows x 128 k
constexpr int kUnitBytes = kMaxPairs * kSlot;
constexpr int kWCodes = 4096;                   // 64 columns x 128 k codes

constexpr int kMaxChunks = 128;                 // K <= 16384
constexpr unsigned kFlag = 8;                   // meta: np | flag | (E + 512) << 8

__device__ __forceinline__ uint32_t perm_b(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}

// Max / or over the wave, returned to every lane, by DPP row shifts and
// broadcasts (as wave_max_nonneg; the whole wave must be active).
template <bool OR>
__device__ __forceinline__ uint32_t wave_fold(uint32_t v) {
#define TKV_FOLD(CTRL, ROWS)                                                                       \
    do {                                                                                           \
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false); \
        v = OR ? (v | o) : max(v, o);                                                              \
    } while (0)
    TKV_FOLD(0x111, 0xf);
    TKV_FOLD(0x112, 0xf);
    TKV_FOLD(0x114, 0xf);
    TKV_FOLD(0x118, 0xf);
    TKV_FOLD(0x142, 0xa);
    TKV_FOLD(0x143, 0xc);
#undef TKV_FOLD
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Byte p of four words as one word: out[p] = a.p | b.p << 8 | c.p << 16 | d.p << 24.
__device__ __forceinline__ void transpose4(uint32_t a, uint32_t b, uint32_t c, uint32_t d,
                                           uint32_t (&out)[4]) {
    const uint32_t t0 = perm_b(b, a, 0x05010400u), t1 = perm_b(b, a, 0x07030602u);
    const uint32_t u0 = perm_b(d, c, 0x05010400u), u1 = perm_b(d, c, 0x07030602u);
    out[0] = perm_b(u0, t0, 0x05040100u);
    out[1] = perm_b(u0, t0, 0x07060302u);
    out[2] = perm_b(u1, t1, 0x05040100u);
    out[3] = perm_b(u1, t1, 0x07060302u);
}

// Blocks [0, units * nk): one unit of A each: its digit planes (pairs
// [0, np)) and meta.  Thread t takes 16 elements: row t / 8, k 16 (t % 8)
// ..; the even ones of each 8 are stored before the odd ones, as the packed
// nibbles unpack.  Rows past M are zeros.
// The remaining blocks retile W: one (64 columns, 128 k) record each, the
// packed bytes of lane (column c, half h) and k-step s at [c][16 s + 8 h ..],
// columns past N code 8 (w = 0) with scale 0, and flag the records that hold a
// scale that is not finite (wflag: one word per record).
__global__ __launch_bounds__(512) void k_int4_planes(
    const float* __restrict__ A, const uint8_t* __restrict__ Wp, const float* __restrict__ scales, int M, int N, int K, int gs,
    int units, int subs, uint8_t* __restrict__ planes, unsigned* __restrict__ meta,
    uint8_t* __restrict__ wt, unsigned* __restrict__ wflag) {
    const int nk = K / kUnitK, t = threadIdx.x;
    const int b = (int)blockIdx.x;
    if (b >= units * nk) {
        const int w = b - units * nk, nb = w / nk, g = w - nb * nk;
        const int half = K / 2, ng = K / gs, blk = nb % 4;
        uint8_t* rec = wt + ((int64_t)(nb / 4) * nk + g) * (4 * kWCodes + subs * 1024);
        int odd = 0;
        if (t < 256) {
            const int lane = t & 63, h = lane >> 5;
            const int col = nb * 64 + (t >> 7) * 32 + (lane & 31);
            uint2 lo = make_uint2(0x88888888u, 0x88888888u), hi = lo;
            if (col < N) {
                const uint8_t* src = Wp + (int64_t)col * half + g * 64 + 32 * ((t >> 6) & 1) + 8 * h;
                lo = *reinterpret_cast<const uint2*>(src);
                hi = *reinterpret_cast<const uint2*>(src + 16);
            }
            reinterpret_cast<uint4*>(rec + blk * kWCodes)[t] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        } else if (t < 256 + 64 * subs) {
            const int sub = (t - 256) >> 6, c = t & 63, col = nb * 64 + c;
            const float sc =
                col < N ? scales[(int64_t)col * ng + (g * kUnitK + sub * (kUnitK / subs)) / gs] : 0.0f;
            reinterpret_cast<float*>(rec + 4 * kWCodes)[(sub * 4 + blk) * 64 + c] = sc;
            odd = (__float_as_uint(sc) & 0x7f800000u) == 0x7f800000u;
        }
        odd = __syncthreads_or(odd);
        if (t == 0) wflag[((int64_t)(nb / 4) * nk + g) * 4 + blk] = odd ? kFlag : 0u;
        return;
    }
    __shared__ uint32_t s_max[8], s_lo[8], s_hi[8], s_bad[8];
    const int u = b / nk, g = b - u * nk;
    const int row = u * kUnitRows + (t >> 3), k0 = g * kUnitK + 16 * (t & 7);
    uint32_t x[16];
    if (row < M) {
        const float* src = A + (int64_t)row * K;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint4 v = *reinterpret_cast<const uint4*>(src + k0 + 4 * e);
            x[4 * e] = v.x;
            x[4 * e + 1] = v.y;
            x[4 * e + 2] = v.z;
            x[4 * e + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 16; e++) x[e] = 0u;
    }
    uint32_t mx = 0;
#pragma unroll
    for (int e = 0; e < 16; e++) mx = max(mx, x[e] & 0x7fffffffu);
    mx = wave_fold<false>(mx);
    if ((t & 63) == 0) s_max[t >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 8; w++) mx = max(mx, s_max[w]);
    const int emax = max((int)(mx >> 23), 1);
    // X = m24 << (ex - emax + 38); digits: byte p of X + 128 (256^0 + .. +
    // 256^6), less 128 below the top byte
    uint32_t alo = 0, ahi = 0;
    bool bad = emax == 255;
    uint64_t d[16];
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const uint32_t v = x[e];
        const int ex = max((int)((v >> 23) & 255u), 1);
        const uint32_t m24 = (v & 0x7fffffu) | ((v & 0x7f800000u) ? 0x800000u : 0u);
        const int sh = ex - emax + 38, rs = min(max(-sh, 0), 31);
        uint64_t X = (uint64_t)(m24 >> rs) << max(sh, 0);
        bad = bad || (m24 & ((1u << rs) - 1u)) != 0u;
        alo |= (uint32_t)X;
        ahi |= (uint32_t)(X >> 32);
        if (v >> 31) X = 0 - X;
        d[e] = (X + 0x0080808080808080ull) ^ 0x0080808080808080ull;
    }
    alo = wave_fold<true>(alo);
    ahi = wave_fold<true>(ahi);
    bad = __any(bad);
    if ((t & 63) == 0) {
        s_lo[t >> 6] = alo;
        s_hi[t >> 6] = ahi;
        s_bad[t >> 6] = bad;
    }
    __syncthreads();
    uint32_t any_bad = 0;
#pragma unroll
    for (int w = 0; w < 8; w++) {
        alo |= s_lo[w];
        ahi |= s_hi[w];
        any_bad |= s_bad[w];
    }
    const int low = alo ? __builtin_ctz(alo) : ahi ? 32 + __builtin_ctz(ahi) : 64;
    const int np = kMaxPairs - low / 16;  // planes 8 - low / 8, in whole pairs
    if (t == 0)
        meta[b] = (unsigned)np | (any_bad ? kFlag : 0u) | (unsigned)(emax - 132 + 512) << 8;
    uint8_t* dst = planes + (int64_t)b * kUnitBytes + (t >> 8) * 4096 + ((t >> 1) & 3) * 1024 +
                   ((t & 1) * 32 + ((t >> 3) & 31)) * 16;
    uint32_t q[2][4][4];  // [word][dword of the run][byte]
#pragma unroll
    for (int w = 0; w < 2; w++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int e = (i >> 1) * 8 + (i & 1);
            transpose4((uint32_t)(d[e] >> (32 * w)), (uint32_t)(d[e + 2] >> (32 * w)),
                       (uint32_t)(d[e + 4] >> (32 * w)), (uint32_t)(d[e + 6] >> (32 * w)), q[w][i]);
        }
#pragma unroll
    for (int pl = 0; pl < 8; pl++)
        if (pl < 2 * np) {
            const int w = pl < 4 ? 1 : 0, by = 3 - (pl & 3);
            *reinterpret_cast<uint4*>(dst + (pl >> 1) * kSlot + (pl & 1) * 8192) =
                make_uint4(q[w][0][by], q[w][1][by], q[w][2][by], q[w][3][by]);
        }
}

__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A workgroup of 4 waves owns 32 rows (half a unit) x 256 columns, wave w the
// columns 64 w .. + 63.  kR ring slots of 8 KB for A's pairs ([plane][k-step]
// of 1 KB fragments) and one buffer for W's record: 74-77 KB, two workgroups
// per CU.  They meet no common barrier, so one's barriers, DMA issue and fold
// tails run under the other's MFMAs.  The same kernel with 8 waves on 64 x 256
// and one workgroup per CU measured 50.8 us against 42.3 (2048 x 2304 x 768,
// prepass included), 148.7 against 131.8 (8192 x 3072 x 768); 64 x 128 tiles
// 51.7 and 174.5.
constexpr int kTileRows = 32, kTileCols = 256, kR = 7;
constexpr int kHalfSlot = 8192;
// W record of one (column tile, chunk): the codes of its four 64-column
// blocks, then SUBS scales per column.
constexpr int wrec_bytes(int subs) { return 4 * kWCodes + subs * kTileCols * 4; }
constexpr int lds_bytes(int subs) { return kR * kHalfSlot + wrec_bytes(subs) + 4 * (kMaxChunks + 1); }
static_assert(kTileRows * kTileCols * 8 <= kR * kHalfSlot + wrec_bytes(1), "f64 tile within the ring");

// What a lane loads for 32 k of the f64 form: 8 k (lane quad q takes 8 q .. + 7)
// of 2 rows of A and of 4 columns of W with their scales.
struct F64Raw {
    float4 a[2][2];
    uint32_t w[4];
    float sc[4];
};

// y (or, SPLIT, the f64 partials of K chunks [z chunks, (z + 1) chunks)) of one
// 32 x 256 tile per workgroup.  SUBS = 128 / gs (1 for gs >= 128) folds per
// chunk.  Bound by the VALU and the matrix unit together: per wave and pair 16
// MFMAs of 32 cycles and 96 fold operations of ~4.7 (shift-add, i32 -> f64,
// f64 fma for each of 32 outputs), two waves per SIMD.
template <int SUBS, bool SPLIT>
__global__ __launch_bounds__(256, 2) void k_matmul_int4_planes(
    const uint8_t* __restrict__ planes, const unsigned* __restrict__ meta,
    const uint8_t* __restrict__ wt, const unsigned* __restrict__ wflag,
    const float* __restrict__ A, const uint8_t* __restrict__ Wp, const float* __restrict__ scales,
    const float* __restrict__ bias, float* __restrict__ Y, int M, int N, int K, int gs,
    int tiles_m, int tiles_n, int chunks, double* __restrict__ part) {
    constexpr int kWRec = wrec_bytes(SUBS), kOffW = kR * kHalfSlot;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    unsigned* s_chunk = reinterpret_cast<unsigned*>(smem + kOffW + kWRec);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nk = K / kUnitK;
    // contiguous tile ranges per XCD; a tile's K splits run next to each other
    const int total = (int)gridDim.x, per = total / 8, rem = total % 8;
    const int xcd = (int)blockIdx.x % 8, jx = (int)blockIdx.x / 8;
    const int v = xcd < rem ? xcd * (per + 1) + jx : rem * (per + 1) + (xcd - rem) * per + jx;
    const int splits = SPLIT ? total / (tiles_m * tiles_n) : 1;
    const int tile = v / splits, z = v - tile * splits;
    const int mt = tile / tiles_n, nt = tile - mt * tiles_n;
    const int g0 = SPLIT ? z * chunks : 0, g1 = SPLIT ? min(nk, g0 + chunks) : nk;
    const int ng = g1 - g0;
    const int unit = mt / 2;
    // the chunks of this tile that have any digits, as chunk | np << 12 |
    // (E + 512) << 16, built by wave 0; their count at the end
    // and, from the list's end, the flagged chunks
    int nch = 0, nbad = 0;
    if (wave == 0) {
        for (int base = 0; base < ng; base += 64) {
            const int g = base + lane;
            unsigned m = 0u, w = 0u;
            if (g < ng) {
                m = meta[(int64_t)unit * nk + g0 + g];
                const uint4 f = reinterpret_cast<const uint4*>(wflag)[(int64_t)nt * nk + g0 + g];
                w = f.x | f.y | f.z | f.w;
            }
            const bool bad = ((m | w) & kFlag) != 0u, has = !bad && (m & 7u) != 0u;
            const uint64_t live = __ballot(has), bads = __ballot(bad), below = (1ull << lane) - 1ull;
            if (has)
                s_chunk[nch + __popcll(live & below)] =
                    (unsigned)g | (m & 7u) << 12 | (m >> 8) << 16;
            if (bad) s_chunk[kMaxChunks - 1 - nbad - __popcll(bads & below)] = (unsigned)g;
            nch += __popcll(live);
            nbad += __popcll(bads);
        }
        if (lane == 0) s_chunk[kMaxChunks] = (unsigned)(nch | nbad << 16);
    }
    __syncthreads();
    nch = __builtin_amdgcn_readfirstlane((int)s_chunk[kMaxChunks]);
    nbad = nch >> 16;
    nch &= 0xffff;
    const int64_t ntc = (int64_t)tiles_n * kTileCols;  // columns of the split partials
    double* __restrict__ mine = SPLIT ? part + (int64_t)z * tiles_m * kTileRows * ntc : nullptr;
    auto store = [&](int row, int col, double a, double b) {
        if (SPLIT)
            mine[(int64_t)row * ntc + col] = a;
        else if (row < M && col < N)
            __builtin_nontemporal_store((float)(a + b), Y + (int64_t)row * N + col);
    };
    double acc[2][16];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[j][r] = 0.0;

    // The chunk list in registers, lane l holding entries l and 64 + l: an
    // entry is one readlane.
    const unsigned list0 = s_chunk[lane], list1 = s_chunk[64 + lane];
    auto chunk_at = [&](int i) {
        return (unsigned)__builtin_amdgcn_readlane((int)(i < 64 ? list0 : list1), i & 63);
    };
    const uint8_t* const wsrc = wt + ((int64_t)nt * nk + g0) * kWRec;
    const uint8_t* const asrc = planes + ((int64_t)unit * nk + g0) * kUnitBytes + (mt & 1) * 4096;
    const uint32_t aoff = (uint32_t)(wave * 1024 + lane * 16);
    // The A stream: the next pair to copy (fsrc) and its ring position (fat).
    const uint8_t* fsrc = asrc;
    int fat = 0;
    auto issue_pair = [&]() {
        uint8_t* dst = smem + fat * kHalfSlot + wave * 1024;
#pragma unroll
        for (int d = 0; d < 2; d++)  // planes of the pair; the wave's k-step
            __builtin_amdgcn_global_load_lds((const void*)(fsrc + d * 8192 + aoff),
                                             (lds_ptr)(dst + d * 4096), 16, 0, 0);
        fsrc += kSlot;
        fat = fat == kR - 1 ? 0 : fat + 1;
    };
    auto seek = [&](unsigned e) { fsrc = asrc + (e & 0xfffu) * (uint32_t)kUnitBytes; };
    // entry e's W record: KBs wave, wave + 4, ..
    auto issue_w = [&](unsigned e) {
        const uint8_t* src = wsrc + (e & 0xfffu) * (uint32_t)kWRec;
        uint8_t* dst = smem + kOffW + wave * 1024;
#pragma unroll
        for (int d = 0; d < (kWRec / 1024 + 3) / 4; d++)
            if (4 * (d + 1) <= kWRec / 1024 || wave + 4 * d < kWRec / 1024)
                __builtin_amdgcn_global_load_lds((const void*)(src + d * 4096 + aoff),
                                                 (lds_ptr)(dst + d * 4096), 16, 0, 0);
    };
    v4i ah[4], al[4], wf[2][4];
    v16i hi[2], lo[2];  // S_hi, S_lo of the block in flight and the one being folded
    double wlast = 0.0;
    const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    hi[1] = lo[1] = zero;
    auto frags = [&](int ring, int plane, v4i (&f)[4]) {
        const uint8_t* p = smem + ring * kHalfSlot + plane * 4096 + lane * 16;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) f[ks] = *reinterpret_cast<const v4i*>(p + ks * 1024);
    };
    // Chunk by chunk: at its start all its slots and its W record have landed
    // (they were issued a chunk ahead, and nothing else is in flight), one
    // barrier publishes them and frees the last chunk's; the waves then run
    // its slots without meeting again.
    unsigned en = nch > 0 ? chunk_at(0) : 0u;
    int ring = 0, ahead = 0;  // ring position of this chunk's first slot; slots issued of the next
    if (nch > 0) {
        issue_w(en);
        seek(en);
        ahead = (int)(en >> 12) & 7;
        for (int q = 0; q < ahead; q++) issue_pair();
    }
    for (int c = 0; c < nch; c++) {
        const unsigned e = en;
        const int np = (int)(e >> 12) & 7, E = (int)(e >> 16) - 512;
        if (ahead < np) {  // the ring was too full for all of them
            lds_barrier();
            for (; ahead < np; ahead++) issue_pair();
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        lds_barrier();
        // no DMA is in flight here: the compiler's wait for them in front of
        // these reads costs nothing
        float sc[2][SUBS];
        uint4 wr[4];  // [column block][k-step pair]
        const uint8_t* wb = smem + kOffW;
#pragma unroll
        for (int i = 0; i < 4; i++) wr[i] = reinterpret_cast<const uint4*>(wb + wave * kWCodes)[i * 64 + lane];
#pragma unroll
        for (int s = 0; s < SUBS; s++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                sc[j][s] = reinterpret_cast<const float*>(
                    wb + 4 * kWCodes)[s * kTileCols + wave * 64 + j * 32 + (lane & 31)];
        frags(ring, 0, ah);
        __builtin_amdgcn_sched_barrier(0);
        ahead = 0;
        if (c + 1 < nch) {
            en = chunk_at(c + 1);
            ahead = min((int)(en >> 12) & 7, kR - np);
            lds_barrier();  // every wave has read this chunk's record
            issue_w(en);
            seek(en);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const uint4 r = wr[2 * j + ks / 2];
                const uint32_t x0 = ks & 1 ? r.z : r.x, x1 = ks & 1 ? r.w : r.y;
                wf[j][ks][0] = (int)(((x0 << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
                wf[j][ks][1] = (int)((x0 & 0xF0F0F0F0u) ^ 0x80808080u);
                wf[j][ks][2] = (int)(((x1 << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
                wf[j][ks][3] = (int)((x1 & 0xF0F0F0F0u) ^ 0x80808080u);
            }
        // weight of P = 256 S_hi + S_lo (S counts 16 (nibble - 8)) in units of
        // the scale
        double pwt = __builtin_ldexp(1.0, E - 12);
        for (int q = 0; q < np; q++) {
            // the next chunk's pairs are copied one with each of this one's: a
            // burst of them would hold up every wave's issue
            if (q < ahead) issue_pair();
            const int cur = ring;
            ring = ring == kR - 1 ? 0 : ring + 1;
            constexpr int KS = 4 / SUBS;
#pragma unroll
            for (int s = 0; s < SUBS; s++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    // Block (s, j) multiplies while the block before it (j ^ 1)
                    // folds, in three steps per output (combine, convert, fma)
                    // that run one MFMA apart: a dependent f64 operation issued
                    // next to its operand would wait out the latency.
                    constexpr int T = 2 * KS, V = 16 / T;  // MFMAs; outputs folded per MFMA
                    int ci[T][V];
                    double cd[T][V];
#pragma unroll
                    for (int t = 0; t < T + 2; t++) {
                        __builtin_amdgcn_sched_barrier(0);
                        if (t < KS)
                            hi[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                                ah[s * KS + t], wf[j][s * KS + t], t ? hi[j] : zero, 0, 0, 0);
                        else if (t < T)
                            lo[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                                al[s * KS + t - KS], wf[j][s * KS + t - KS], t > KS ? lo[j] : zero, 0,
                                0, 0);
                        if (s == 0 && j == 0 && t == 0) frags(cur, 1, al);
                        // the next pair's (past the chunk's last: not used)
                        if (s == SUBS - 1 && j == 1 && t == KS) frags(ring, 0, ah);
#pragma unroll
                        for (int w = 0; w < V; w++) {
                            if (t >= 2)
                                acc[j ^ 1][(t - 2) * V + w] =
                                    __builtin_fma(cd[t - 2][w], wlast, acc[j ^ 1][(t - 2) * V + w]);
                            if (t >= 1 && t <= T) cd[t - 1][w] = (double)ci[t - 1][w];
                            if (t < T) ci[t][w] = (hi[j ^ 1][t * V + w] << 8) + lo[j ^ 1][t * V + w];
                        }
                    }
                    wlast = (double)sc[j][s] * pwt;
                }
            pwt *= 0x1p-16;
            __builtin_amdgcn_sched_barrier(0);
        }
        for (int q = np; q < ahead; q++) issue_pair();
    }
#pragma unroll
    for (int r = 0; r < 16; r++)
        acc[1][r] = __builtin_fma((double)((hi[1][r] << 8) + lo[1][r]), wlast, acc[1][r]);
    // The flagged chunks: the wave's 32 x 64 outputs on the f64 MFMA, each 32 k
    // loaded while the 32 before multiply; rows past M and columns past N read the
    // last one.  Then through LDS to the layout of acc.  Bound by the f64 matrix
    // rate of the tile's own CU, 7 us a chunk.  No flag / one element flagged / every
    // unit flagged, against the f64 GEMM for any values: 2048 x 2304 x 768 39.8 /
    // 38.9 / 174 us against 140, 300 x 2304 x 768 19.5 / 29.1 / 67 against 36 (90
    // tiles), 2048 x 768 x 3072 53 / 62 / 242 against 196, 8192 x 3072 x 768 135 /
    // 133 / 672 against 654.  (With the tile's whole K on the f64 MFMA: one element
    // 84, 82, 298 and 157 us.)
    if (nbad > 0) {
        const int l16 = lane & 15, quad = lane >> 4, ngrp = K / gs;
        const int col0 = nt * kTileCols + wave * 64;
        const float* arow[2];
        const uint8_t* wcol[4];
        const float* scol[4];
#pragma unroll
        for (int i = 0; i < 2; i++)
            arow[i] = A + (int64_t)min(mt * kTileRows + 16 * i + l16, M - 1) * K;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t col = min(col0 + 16 * j + l16, N - 1);
            wcol[j] = Wp + col * (K / 2);
            scol[j] = scales + col * ngrp;
        }
        auto load = [&](int step, F64Raw& r) {
            const int g = (int)(chunk_at(kMaxChunks - 1 - step / 4) & 0xfffu);
            const int k0 = (g0 + g) * kUnitK + 32 * (step % 4), kk = k0 + 8 * quad;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                r.a[i][0] = *reinterpret_cast<const float4*>(arow[i] + kk);
                r.a[i][1] = *reinterpret_cast<const float4*>(arow[i] + kk + 4);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                r.w[j] = *reinterpret_cast<const uint32_t*>(wcol[j] + kk / 2);
                r.sc[j] = scol[j][k0 / gs];
            }
        };
        f64x4 fa[2][4];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) fa[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
        F64Raw next;
        load(0, next);
        for (int step = 0; step < 4 * nbad; step++) {
            const F64Raw r = next;
            if (step + 1 < 4 * nbad) load(step + 1, next);
            const float* av[2] = {reinterpret_cast<const float*>(r.a[0]),
                                  reinterpret_cast<const float*>(r.a[1])};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                double b[4];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    b[j] = (double)((int)((r.w[j] >> (4 * e)) & 15) - 8) * (double)r.sc[j];
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        fa[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)av[i][e], b[j],
                                                                       fa[i][j], 0, 0, 0);
            }
        }
        __syncthreads();  // every wave is past its last read of the ring
        double* s_f = reinterpret_cast<double*>(smem) + wave * (kTileRows * 64);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    s_f[(16 * i + quad + 4 * e) * 64 + 16 * j + l16] = fa[i][j][e];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                acc[j][r] += s_f[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * 64 + j * 32 + (lane & 31)];
    }
    // D layout: lane l, register r holds row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int col = nt * kTileCols + wave * 64 + j * 32 + (lane & 31);
        const double bb = bias && col < N ? (double)bias[col] : 0.0;
#pragma unroll
        for (int r = 0; r < 16; r++)
            store(mt * kTileRows + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3), col,
                  acc[j][r], bb);
    }
}

// Row panel of one pass: its planes fit kPlanesBytes.
constexpr int64_t kPlanesBytes = (int64_t)256 << 20;

struct PlanesArgs {
    const uint8_t* planes;
    const unsigned* meta;
    const uint8_t* wt;
    const unsigned* wflag;
    const float* a;
    const uint8_t* wp;
    const float *scales, *bias;
    float* y;
    int m, n, k, gs, tiles_m, tiles_n, chunks, splits;
    double* part;
};

template <int SUBS, bool SPLIT>
void run_planes(Ctx* c, const PlanesArgs& g) {
    hipLaunchKernelGGL((k_matmul_int4_planes<SUBS, SPLIT>),
                       dim3((unsigned)(g.tiles_m * g.tiles_n * g.splits)), dim3(256),
                       lds_bytes(SUBS), c->stream, g.planes, g.meta, g.wt, g.wflag, g.a, g.wp,
                       g.scales, g.bias, g.y, g.m, g.n, g.k, g.gs, g.tiles_m, g.tiles_n, g.chunks, g.part);
}

template <int SUBS>
void run_planes_subs(Ctx* c, const PlanesArgs& g) {
    if (g.splits > 1)
        run_planes<SUBS, true>(c, g);
    else
        run_planes<SUBS, false>(c, g);
}

// K splits (f64 partial tiles, k_int4_split_sum) for `tiles` tiles of nk
// chunks: rounds of workgroups (a CU with two takes 1.5 times as long as with
// one) times chunks at 1.45 us, plus 3 us for the sum's launch, its traffic
// at 5 TB/s and 0.15 us per split.  Over forced counts on five (N, K) pairs,
// M = 33 .. 2048, the pick is within 4% of the best on average (768 x 3072:
// M = 64 46.1 us unsplit, 21.0 in 8; M = 768 52.9 and 35.4 in 3).
int64_t planes_splits(int64_t tiles, int64_t nk, int64_t ncu, int64_t mt, int64_t nt) {
    double best = 1e300;
    int64_t pick = 1;
    for (int64_t s = 1; s <= std::min<int64_t>(nk, 24); s++) {
        const int64_t chunks = ceil_div(nk, s), w = ceil_div(tiles * s, ncu);
        if (ceil_div(nk, chunks) != s || s * mt * nt * 8 > kPlanesBytes) continue;
        const double est = (w == 1 ? 1.0 : 0.75 * (double)w) * (double)chunks * 1.45 +
                           (s > 1 ? 3.0 + 0.15 * (double)s + (double)(s * mt * nt) * 16.0 / 5e6 : 0.0);
        if (est < best) best = est, pick = s;
    }
    return pick;
}

}  // namespace

int launch_matmul_int4_planes(Ctx* c, const float* a, const uint8_t* wp, const float* scales,
                              const float* bias, const int64_t* perm, float* y, int64_t m,
                              int64_t n, int64_t k, int64_t gs) {
    const bool subs_ok = gs == 32 || gs == 64 || (gs >= 128 && gs % 128 == 0);
    const int64_t nk = k / kUnitK;
    if (m < 1 || n < 1 || k < kUnitK || k % kUnitK != 0 || nk > kMaxChunks || !subs_ok ||
        !aligned(a, 16) || !aligned(wp, 8) || m >= (1 << 24) || n >= (1 << 24))
        return TKV_HIP_UNSUPPORTED;
    const int64_t panel = std::max<int64_t>(kPlanesBytes / (kUnitBytes * nk), 1);
    const int64_t units_all = ceil_div(m, (int64_t)kUnitRows);
    const int64_t units_max = std::min(units_all, panel);
    const int subs = gs >= 128 ? 1 : (int)(128 / gs);
    const int64_t tiles_n = ceil_div(n, (int64_t)kTileCols);
    const int64_t mt = units_max * kUnitRows, nt = tiles_n * kTileCols;
    const int64_t splits = planes_splits(2 * units_max * tiles_n, nk, c->num_cus, mt, nt);
    const size_t planes_need = (size_t)(units_max * nk) * (kUnitBytes + 4);
    const size_t wt_need = (size_t)(tiles_n * nk) * (wrec_bytes(subs) + 16);
    const size_t part_need = splits > 1 ? (size_t)(splits * mt * nt) * 8 : 0;
    // inside a capture nothing can grow: the f64 kernels may need no workspace
    const size_t perm_need = perm ? (size_t)(std::min(m, mt) * k) * 4 : 0;
    if (c->capturing && (c->ws_bytes[15] < perm_need || c->ws_bytes[13] < planes_need || c->ws_bytes[14] < wt_need ||
                         c->ws_bytes[12] < part_need))
        return TKV_HIP_UNSUPPORTED;
    void *planes, *wt, *part = nullptr, *permuted = nullptr;
    if (perm) TKV_RC_TRY(ctx_workspace(c, 15, perm_need, &permuted));
    TKV_RC_TRY(ctx_workspace(c, 13, planes_need, &planes));
    TKV_RC_TRY(ctx_workspace(c, 14, wt_need, &wt));
    if (splits > 1) TKV_RC_TRY(ctx_workspace(c, 12, part_need, &part));
    unsigned* meta = reinterpret_cast<unsigned*>(static_cast<uint8_t*>(planes) +
                                                 (size_t)(units_max * nk) * kUnitBytes);
    unsigned* wflag = reinterpret_cast<unsigned*>(static_cast<uint8_t*>(wt) +
                                                  (size_t)(tiles_n * nk) * wrec_bytes(subs));
    for (int64_t u0 = 0; u0 < units_all; u0 += panel) {
        const int64_t units = std::min(panel, units_all - u0), row0 = u0 * kUnitRows;
        PlanesArgs g;
        g.planes = static_cast<const uint8_t*>(planes);
        g.meta = meta;
        g.wt = static_cast<const uint8_t*>(wt);
        g.wflag = wflag;
        g.a = a + row0 * k;
        g.wp = wp;
        g.scales = scales;
        g.bias = bias;
        g.y = y + row0 * n;
        g.m = (int)std::min(m - row0, units * kUnitRows);
        g.n = (int)n;
        g.k = (int)k;
        g.gs = (int)gs;
        g.tiles_m = (int)(2 * units);
        g.tiles_n = (int)tiles_n;
        g.chunks = (int)ceil_div(nk, splits);
        g.splits = (int)splits;
        g.part = static_cast<double*>(part);
        const unsigned pgrid = (unsigned)(units * nk + (u0 == 0 ? tiles_n * 4 * nk : 0));
        if (perm) {  // act-order: the panel's columns gathered first, row by row through LDS
            float* ap = static_cast<float*>(permuted);
            TKV_RC_TRY(launch_permute_cols(c, g.a, g.m, k, perm, false, ap));
            g.a = ap;
        }
        hipLaunchKernelGGL(k_int4_planes, dim3(pgrid), dim3(512), 0, c->stream, g.a, wp, scales, g.m,
                           (int)n, (int)k, (int)gs, (int)units, subs, static_cast<uint8_t*>(planes),
                           meta, static_cast<uint8_t*>(wt), wflag);
        TKV_LAUNCH_CHECK();
        if (subs == 4)
            run_planes_subs<4>(c, g);
        else if (subs == 2)
            run_planes_subs<2>(c, g);
        else
            run_planes_subs<1>(c, g);
        TKV_LAUNCH_CHECK();
        if (splits > 1)
            TKV_RC_TRY(launch_int4_split_sum(c, g.part, g.splits, units * kUnitRows,
                                             tiles_n * kTileCols, bias, g.y, g.m, (int)n));
    }
    return TKV_HIP_OK;
}

}  // namespace tkv

/*
 * hd_cnn.hip -- the flow surrogate's network on gfx950: 3x3 convolutions as
 * implicit GEMMs on the BF16 MFMA (v_mfma_f32_16x16x32_bf16, FP32
 * accumulation), their data and weight gradients, masked-MSE loss, Adam, and
 * the packing between a hydist context's FP64 state and the network's
 * images (include/hydist_cnn.h).
 *
 * MFMA operand layout (16x16x32, wave64): lane l holds A[m = l%16][k =
 * 8(l/16) .. 8(l/16)+7], B[k = 8(l/16) .. +7][n = l%16], and D[m = 4(l/16) +
 * r][n = l%16] for r = 0..3 (checked by hd_cnn_mfma_check against a host
 * product).
 *
 * Convolution (forward and data gradient): A is the weights, B the pixels, so
 * a lane's results are neighbouring channels of one pixel and leave in 16-byte
 * stores.  A wave keeps the weights of its 32 output channels (all taps) in
 * registers and walks down a strip of 16 columns: the fragments of an input
 * row are loaded once, straight from memory in the operand's layout, and
 * serve the three output rows they touch, each summed over the taps in their
 * order.  Weight gradient: K = pixels; image rows pass through LDS once and
 * both operands are read from there transposed.
 */
#include "hd_internal.h"
#include "../../include/hydist_cnn.h"

#include <cmath>
#include <cstring>
#include <utility>
#include <string>
#include <vector>

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

/* hd_api.hip: device view and stream of a context (same library) */
const HdDev* hd_ctx_device_view(hd_ctx* c, hipStream_t* stream, int* state);

namespace {

constexpr int kCinPad = 32;   /* input channels after padding */
constexpr int kWidth = 64;    /* hidden channels */
constexpr int kOutPad = 32;   /* output channels after padding */
constexpr int kNarrow = 8;    /* stored channels of input images and output gradients (the rest are zero) */
constexpr int kOut4 = 4;      /* stored channels of the network's output */

enum { EPI_RELU = 0, EPI_RESRELU = 1, EPI_LINEAR = 2, EPI_BWD_SET = 3, EPI_BWD_ADD = 4 };

__device__ __forceinline__ f32x4 mfma(const bf16x8& a, const bf16x8& b, const f32x4& c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

/* base[row elements + lane's byte offset]: the row (wave-uniform, kept from
 * being turned into a pointer per lane and per use) in scalar registers */
template <typename T, typename E>
__device__ __forceinline__ T ld_row(const E* base, size_t row, unsigned off)
{
    return *(const T*)((const char*)(base + row) + off);
}
template <typename T, typename E>
__device__ __forceinline__ void st_row(E* base, size_t row, unsigned off, T v)
{
    *(T*)((char*)(base + row) + off) = v;
}
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

/* A stretch of `bytes` bytes of a row as a buffer: loads past either end of
 * it return zeros and stores there are dropped (an offset below 0 is far past
 * the end), and none of a stretch of 0 bytes is touched.  A stretch is what a
 * workgroup's columns need of the row and no more, so that offsets are small
 * however wide the image is.  So every step of a walk over
 * rows has the same memory operations, which is what lets the compiler count
 * those in flight instead of waiting for all of them.  An access that is to
 * touch nothing at all takes kNowhere: past every stretch (66 columns of 256
 * bytes at most), aligned to 16 bytes, and far enough from 2^32 that none of
 * its words wraps round to the row's start. */
constexpr unsigned kNowhere = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_buffer(const void* base, size_t at, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)base + at), 0, (int)bytes, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T buf_ld16(__amdgpu_buffer_rsrc_t r, unsigned off)
{
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
template <typename T>
__device__ __forceinline__ void buf_st16(__amdgpu_buffer_rsrc_t r, unsigned off, T v)
{
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, (int)off, 0, 0);
}
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

/* The work of one convolution launch, in items of a strip of rows: item k
 * covers rows [r0, r0 + R) of 16 * (strips per workgroup) columns.  Dense: k
 * counts columns of items first, then row blocks, then images.  With a tile
 * list (tl != nullptr) the items are the 4 x 64 tiles tl[0 .. *tn). */
struct ConvItems {
    int H, W, R, rows, cols, total;
    const int *tl, *tn;
};

/* Y = conv3x3(X) (+ bias) with epilogue EPI; images [nimg][H][W][C].
 *
 * Bound: the matrix cores and the traffic of the images about evenly (64
 * channels in and out: 74 kflop and 256 to 776 bytes a pixel), if the loads
 * are far enough ahead: a row of a strip is 0.5 us of MFMAs and a load takes
 * up to 2 us.  So a workgroup's rows travel three ahead in registers and wait
 * in an LDS ring of four, one barrier a row; weights cost nothing (144
 * registers, half of the output channels a wave, two waves per SIMD).  A
 * row's fragments serve the three output rows it touches, 36 MFMAs for six
 * LDS reads; pixels are 144 bytes apart there, free of bank conflicts.
 * Staging each tap's weights in LDS instead, for 4 x 64 tiles, needed an LDS
 * read of half its time for every MFMA: 224 us per 64 -> 64 layer at 983 x
 * 1051, against 80 now (dZ and dA of the data gradient: 242 + 158 for the
 * ReLU pass, against 151, 5.3 TB/s).
 *
 * Workgroups stay for as many items as there are; a wave's three
 * accumulators are the output rows above, at and below the input row at
 * hand.  gate: a bit per channel and pixel, whether the layer's ReLU passed
 * (written forward; read backward for the layer below: dZ is
 * bf16(dA) where it did).  The layer adds its input to its output (RESRELU)
 * from the ring. */
template <int EPI>
__global__ void __launch_bounds__(256, 2)
k_conv(const bf16* __restrict__ X, const bf16* __restrict__ Wt, const float* __restrict__ bias, ConvItems it,
       bf16* __restrict__ Y, unsigned char* __restrict__ gate, float* __restrict__ Yf, int store_f)
{
    constexpr bool NARROW = EPI == EPI_RELU || EPI == EPI_BWD_SET; /* stored input channels: 8 of 32, else 64 */
    constexpr int KC = NARROW ? 1 : 2;                             /* 32-channel chunks of a tap */
    constexpr int NB = EPI == EPI_LINEAR ? 1 : 2;                  /* 16-channel blocks of a wave's output */
    constexpr int NH = NB;                                         /* waves that share a strip */
    constexpr int CS = NARROW ? kNarrow : kWidth, CP = 32 * KC, CO = EPI == EPI_LINEAR ? kOutPad : kWidth;
    constexpr int SW = 4 / NH;                                     /* strips per workgroup */
    constexpr int PX = 16 * SW + 2;                                /* columns of a row in LDS */
    constexpr int PS = NARROW ? 8 : 72;                            /* channels between them there */
    /* a row in 16-byte pieces: NL per thread, and for 64 channels the last
     * two columns as a word each of 64 threads */
    constexpr int NL = NARROW ? 1 : SW / 2;
    __shared__ __attribute__((aligned(16))) bf16 ring[4][PX * PS];
    const int wv = uniform(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int half = wv % NH, strip = wv / NH;
    const int n = l & 15, g = l >> 4;
    /* lane group g's results are channels cb .. cb + 4 NB - 1 */
    const int cb = NB == 2 ? 32 * half + 8 * g : 4 * g;
    bf16x8 wf[9][KC][NB];
    {
        const int co = NB == 2 ? 32 * half + 8 * (n >> 2) + (n & 3) : n;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap)
#pragma unroll
            for (int kc = 0; kc < KC; ++kc)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    wf[tap][kc][nb] = *(const bf16x8*)(Wt + ((size_t)tap * CO + co + 4 * nb) * CP + kc * 32 + 8 * g);
    }
    float bv[4 * NB];
    if (EPI == EPI_RELU || EPI == EPI_RESRELU || EPI == EPI_LINEAR) {
#pragma unroll
        for (int q = 0; q < 4 * NB; ++q) bv[q] = bias[cb + q];
    }
    __builtin_amdgcn_s_waitcnt(0x0f70); /* weights and bias are here: no wait for them in the loop */
    const bf16x8 zero8 = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    const int H = it.H, W = it.W;
    constexpr int PER = 64 / (16 * SW); /* items per tile of the list */
    const int total = it.tl ? it.tn[0] * PER : it.total;
    /* the lane's fragments of a row: column 16 strip + n + dx, channels 8 g .. */
    const int fo = (16 * strip + n) * PS + (NARROW ? 0 : 8 * g);
    for (int k = blockIdx.x; k < total; k += gridDim.x) {
        int w0, r0, r1;
        size_t img = 0;
        if (it.tl) {
            const int tilesW = (W + 63) >> 6, t = it.tl[k / PER];
            w0 = (t % tilesW) * 64 + (k % PER) * 16 * SW;
            r0 = (t / tilesW) * 4;
            r1 = r0 + 4;
        } else {
            w0 = (k % it.cols) * 16 * SW;
            const int t = k / it.cols;
            r0 = (t % it.rows) * it.R;
            r1 = r0 + it.R;
            img = (size_t)(t / it.rows) * H * W;
        }
        w0 = uniform(w0);
        r0 = uniform(r0);
        r1 = uniform(r1 < H ? r1 : H);
        /* the columns that the item reads, those of the image from c0 on, and
         * that it writes */
        const int c0 = w0 > 0 ? w0 - 1 : 0;
        const unsigned wr = W - c0 < PX ? W - c0 : PX, ww = W - w0 < 16 * SW ? W - w0 : 16 * SW;
        const size_t imgx = img + c0, imgy = img + w0;
        /* the thread's pieces of a row: byte offsets from column c0, columns
         * outside the image past the row's ends */
        struct Piece {
            bf16x8 q[NL];
            unsigned last;
        };
        unsigned vo[NL], vl = 0;
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const int e = threadIdx.x + 256 * q, c = w0 - 1 - c0 + e / (CS / 8);
            vo[q] = 2u * (unsigned)(c * CS + e % (CS / 8) * 8);
        }
        if (!NARROW) vl = 2u * (unsigned)((w0 - 1 - c0 + PX - 2 + (l >> 5)) * CS) + 4u * (l & 31);
        /* byte offset of row y of the item's image from its column at, E
         * bytes a pixel; rows off the image have no bytes */
        auto row_at = [&](size_t at, int y, int E) -> size_t {
            return (at + (size_t)uniform((y < 0 ? 0 : (y < H ? y : H - 1)) * W)) * E;
        };
        auto load = [&](int i, Piece& r) {
            const auto b = row_buffer(X, row_at(imgx, i, 2 * CS), i >= 0 && i < H && i <= r1 ? 2u * CS * wr : 0u);
#pragma unroll
            for (int q = 0; q < NL; ++q) r.q[q] = buf_ld16<bf16x8>(b, vo[q]);
            if (!NARROW) r.last = __builtin_amdgcn_raw_buffer_load_b32(b, (int)vl, 0, 0);
        };
        auto store = [&](int i, const Piece& r) {
            bf16* to = ring[i & 3];
#pragma unroll
            for (int q = 0; q < NL; ++q) {
                const int e = threadIdx.x + 256 * q;
                if (!NARROW || e < PX) *(bf16x8*)(to + e / (CS / 8) * PS + e % (CS / 8) * 8) = r.q[q];
            }
            if (!NARROW && wv == 0) *(unsigned*)(to + (PX - 2 + (l >> 5)) * PS + 2 * (l & 31)) = r.last;
        };
        const int col = 16 * strip + n;                  /* of the item */
        const unsigned oe = (unsigned)col * kWidth + cb; /* the lane's results in its row of 64 channels */
        /* old dA and the gate of an output row, loaded a row ahead */
        struct Old {
            f32x4 a, b;
            unsigned gate;
        };
        auto load_old = [&](int y, Old& o) {
            if (EPI != EPI_BWD_SET && EPI != EPI_BWD_ADD) return;
            const unsigned w = y >= r0 && y < r1 ? ww : 0u;
            if (EPI == EPI_BWD_ADD) {
                const auto b = row_buffer(Yf, row_at(imgy, y, 4 * kWidth), 4 * kWidth * w);
                o.a = buf_ld16<f32x4>(b, 4 * oe);
                o.b = buf_ld16<f32x4>(b, 4 * oe + 16);
            }
            o.gate = __builtin_amdgcn_raw_buffer_load_b8(row_buffer(gate, row_at(imgy, y, 8), 8 * w), (int)(oe >> 3), 0, 0);
        };
        /* the results of output row y, or with w = 0 the same stores to nowhere */
        auto put = [&](int y, unsigned w, bf16x8 yv, unsigned bits, const f32x4& d0, const f32x4& d1) {
            if (EPI == EPI_LINEAR) {
                buf_st16(row_buffer(Yf, row_at(imgy, y, 4 * kOut4), 4 * kOut4 * w), g == 0 ? 16u * col : kNowhere, d0);
                return;
            }
            if (EPI == EPI_BWD_SET || EPI == EPI_BWD_ADD) {
                const auto b = row_buffer(Yf, row_at(imgy, y, 4 * kWidth), store_f ? 4 * kWidth * w : 0u);
                buf_st16(b, 4 * oe, d0);
                buf_st16(b, 4 * oe + 16, d1);
            } else {
                __builtin_amdgcn_raw_buffer_store_b8((unsigned char)bits, row_buffer(gate, row_at(imgy, y, 8), 8 * w),
                                                     (int)(oe >> 3), 0, 0);
            }
            buf_st16(row_buffer(Y, row_at(imgy, y, 2 * kWidth), 2 * kWidth * w), 2 * oe, yv);
        };
        /* input row i: its products for the output rows i - 1 (below it in
         * the order of the taps: their last three), i and i + 1, then the
         * epilogue of row i - 1 */
        auto step = [&](int i, f32x4(&above)[NB], f32x4(&at)[NB], f32x4(&below)[NB], const Old& o) {
            const int y = i - 1;
            const bool done = y >= r0;
            bf16x8 f[3][KC];
#pragma unroll
            for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                for (int kc = 0; kc < KC; ++kc) {
                    f[dx][kc] = *(const bf16x8*)(ring[i & 3] + fo + dx * PS + 32 * kc);
                    if (NARROW && g != 0) f[dx][kc] = zero8;
                }
            auto taps = [&](int t0, f32x4(&acc)[NB]) {
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                    for (int kc = 0; kc < KC; ++kc)
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma(wf[t0 + dx][kc][nb], f[dx][kc], acc[nb]);
            };
            if (done) taps(6, above);
            if (i >= r0 && i < r1) taps(3, at);
            if (i + 1 < r1) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) below[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
                taps(0, below);
            }
            const unsigned w = done ? ww : 0u;
            if (EPI == EPI_LINEAR) {
                f32x4 v;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = above[0][r] + bv[r];
                put(y, w, zero8, 0, v, v);
                return;
            }
            bf16x8 yv;
            if (EPI == EPI_RELU || EPI == EPI_RESRELU) {
                unsigned bits = 0;
                bf16x8 rs = zero8;
                if (EPI == EPI_RESRELU) rs = *(const bf16x8*)(ring[y & 3] + (16 * strip + n + 1) * PS + cb);
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float v = fmaxf(above[NB == 2 ? q >> 2 : 0][q & 3] + bv[q % (4 * NB)], 0.f);
                    yv[q] = (bf16)(EPI == EPI_RESRELU ? (float)rs[q] + v : v);
                    /* the rounded value is positive (the smallest bf16 is 2^-133) */
                    bits |= v > 0x1p-134f ? 1u << q : 0u;
                }
                put(y, w, yv, bits, above[0], above[NB - 1]);
            } else {
                f32x4 d0 = above[0], d1 = above[NB - 1];
                if (EPI == EPI_BWD_ADD) { d0 = o.a + d0; d1 = o.b + d1; }
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    yv[q] = (o.gate >> q) & 1 ? (bf16)(q < 4 ? d0[q & 3] : d1[q & 3]) : (bf16)0.f;
                put(y, w, yv, 0, d0, d1);
            }
        };
        f32x4 a0[NB], a1[NB], a2[NB];
        Piece p0, p1, p2;
        Old o0, o1, o2;
        int i = r0 - 1;
        /* the loads of the first rows with a step's other operations between
         * them (on no bytes), so that the loop is entered with the same
         * operations in flight that it leaves */
        auto idle = [&](Old& o) {
            load_old(-1, o);
            put(0, 0u, zero8, 0, f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f});
        };
        load(i, p0);
        __builtin_amdgcn_sched_barrier(0);
        load(i + 1, p1);
        __builtin_amdgcn_sched_barrier(0);
        idle(o1);
        __builtin_amdgcn_sched_barrier(0);
        load(i + 2, p2);
        __builtin_amdgcn_sched_barrier(0);
        idle(o2);
        __syncthreads(); /* the item before has read its last rows */
        store(i, p0);
        __builtin_amdgcn_sched_barrier(0);
        load(i + 3, p0);
        __builtin_amdgcn_sched_barrier(0);
        idle(o0);
        __syncthreads();
        /* three steps a round: accumulators, pieces and old values change
         * roles without moving.  Step i: row i + 1 to LDS, row i + 4 on its way */
        auto round = [&](f32x4(&above)[NB], f32x4(&at)[NB], f32x4(&below)[NB], Piece& pc, const Old& o, Old& on) {
            store(i + 1, pc);
            load(i + 4, pc);
            if (EPI != EPI_BWD_ADD) __builtin_amdgcn_sched_barrier(0);
            load_old(i, on);
            step(i, above, at, below, o);
            __syncthreads();
        };
#pragma unroll 1
        for (;;) {
            round(a0, a1, a2, p1, o0, o1);
            if (++i > r1) break;
            round(a1, a2, a0, p2, o1, o2);
            if (++i > r1) break;
            round(a2, a0, a1, p0, o2, o0);
            if (++i > r1) break;
        }
    }
}

/* 16 channels x 8 pixels of an LDS image row as an MFMA operand (lane l:
 * channel l % 16, pixels 8 (l / 16) ..): two transposing reads.  p: the
 * lane's address of the first, pixel 8 (l / 16) + (l % 16) / 4, channel
 * 4 (l % 4); S: channels between pixels. */
template <int S>
__device__ __forceinline__ bf16x8 ld_tr(const bf16* p)
{
    typedef __attribute__((address_space(3))) s16x4* lp;
    union {
        s16x4 h[2];
        bf16x8 v;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)p);
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(p + 4 * S));
    return u.v;
}

/* dW[tap][co][ci] += sum over pixels p of dZ[p][co] * X[p + off(tap)][ci],
 * db[co] += sum of dZ[p][co].  MB, NBI: 16-channel blocks of dZ and of X (1
 * where 8 channels are stored).
 *
 * Bound: the matrix cores, then LDS.  Each half of a workgroup walks down 64
 * columns: each row of dZ and of X comes to LDS once (the X rows in a ring of
 * four, loaded two rows ahead, one barrier a row) and is read from there
 * transposed.  A wave takes 16 input channels, all output channels and
 * all taps: 13 operands for 36 MFMAs, 0.7 of the LDS rate.  Pixels are 160
 * bytes apart, so that the four rows of a transposing read lie in different
 * banks.  The bias gradient is one more product, with ones.  Sums stay in
 * registers until the workgroup has no rows left; then the halves' meet in
 * LDS, since the additions to the shared gradient are 0.09 us for every
 * workgroup, whatever its work.  64 -> 64 layer, two images of 983 x 1051:
 * 232 us with a workgroup per four waves and rows one ahead, 192 now; half
 * the LDS reads (32 columns, rows of dZ kept in registers) made no
 * difference. */
template <int MB, int NBI>
__global__ void __launch_bounds__(512, 2) k_wgrad(const bf16* __restrict__ X, const bf16* __restrict__ dZ,
                                                  ConvItems it, float* __restrict__ dw, float* __restrict__ db)
{
    constexpr int SZ = MB == 4 ? 80 : 16, SX = NBI == 4 ? 80 : 16;
    constexpr int CZ = MB == 4 ? 64 : kNarrow, CX = NBI == 4 ? 64 : kNarrow; /* stored channels */
    constexpr int COP = MB == 4 ? kWidth : kOutPad, CIP = NBI == 4 ? kWidth : kCinPad;
    constexpr int QZ = 64 * CZ / 8, QX = 66 * CX / 8;                        /* 16-byte pieces of a row */
    constexpr int NZ = (QZ + 255) / 256, NX = (QX + 255) / 256;
    constexpr int MW = NBI == 4 ? MB : 1;                                    /* dZ blocks of a wave */
    constexpr int NA = 9 * MW + 1;                                           /* sums of a lane, by four */
    struct Half {
        bf16 z[2][64 * SZ], x[4][66 * SX];
    };
    union Lds {
        Half half[2];
        f32x4 sum[NA][256];
    };
    __shared__ __attribute__((aligned(16))) Lds lds;
    const int half = uniform(threadIdx.x >> 8), tid = threadIdx.x & 255;
    const int wv = uniform(tid >> 6), l = threadIdx.x & 63;
    auto& sZ = lds.half[half].z;
    auto& sX = lds.half[half].x;
    const int H = it.H, W = it.W;
    const bf16x8 zero8 = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    const bf16x8 ones = bf16x8{1, 1, 1, 1, 1, 1, 1, 1};
    if (MB == 1)
        for (int q = tid; q < 128; q += 256) *(bf16x8*)(sZ[q >> 6] + (q & 63) * SZ + 8) = zero8;
    if (NBI == 1)
        for (int q = tid; q < 4 * 66; q += 256) *(bf16x8*)(sX[q / 66] + (q % 66) * SX + 8) = zero8;
    f32x4 acc[9][MW], accb = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int m = 0; m < MW; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int mb0 = NBI == 4 ? 0 : wv, nb0 = NBI == 4 ? wv : 0; /* the wave's first blocks */
    const int px = 8 * (l >> 4) + ((l & 15) >> 2), ch = 4 * (l & 3);
    for (int k2 = 2 * blockIdx.x; k2 < it.total; k2 += 2 * gridDim.x) {
        /* an item for each half; they share the barriers, so both walk R
         * rows (those past an item's end, or of no item, are zeros) */
        const int k = k2 + half < it.total ? k2 + half : it.total - 1;
        const int w0 = uniform((k % it.cols) * 64), t = k / it.cols;
        const int r0 = uniform((t % it.rows) * it.R);
        const int r1 = uniform(k != k2 + half ? r0 : (r0 + it.R < H ? r0 + it.R : H));
        const size_t img = (size_t)uniform(t / it.rows) * H * W;
        /* the columns of X, from c0 on, and of dZ that the item reads */
        const int c0 = w0 > 0 ? w0 - 1 : 0;
        const unsigned wx = W - c0 < 66 ? W - c0 : 66, wz = W - w0 < 64 ? W - w0 : 64;
        const size_t imgx = img + c0, imgz = img + w0;
        /* row h of dZ and row h + 1 of X, as each thread carries them */
        struct Rows {
            bf16x8 z[NZ], x[NX];
        };
        auto row_at = [&](size_t at, int y, int E) -> size_t {
            return (at + (size_t)uniform((y < 0 ? 0 : (y < H ? y : H - 1)) * W)) * E;
        };
        auto ld_x = [&](int h, bool on, bf16x8(&x)[NX]) {
            const auto b = row_buffer(X, row_at(imgx, h, 2 * CX), on && h >= 0 && h < H ? 2u * CX * wx : 0u);
#pragma unroll
            for (int q = 0; q < NX; ++q) {
                const int e = tid + 256 * q;
                const int c = w0 - 1 - c0 + e / (CX / 8);
                x[q] = buf_ld16<bf16x8>(b, e < QX ? 2u * (unsigned)(c * CX + e % (CX / 8) * 8) : kNowhere);
            }
        };
        auto ld = [&](int h, Rows& r) {
            const auto b = row_buffer(dZ, row_at(imgz, h, 2 * CZ), h < r1 ? 2u * CZ * wz : 0u);
#pragma unroll
            for (int q = 0; q < NZ; ++q) {
                const int e = tid + 256 * q;
                const unsigned at = 2u * (unsigned)(e / (CZ / 8) * CZ + e % (CZ / 8) * 8);
                r.z[q] = buf_ld16<bf16x8>(b, e < QZ ? at : kNowhere);
            }
            ld_x(h + 1, h < r1, r.x);
        };
        auto st_x = [&](int h, const bf16x8(&x)[NX]) {
#pragma unroll
            for (int q = 0; q < NX; ++q) {
                const int e = tid + 256 * q;
                if (e < QX) *(bf16x8*)(sX[h & 3] + e / (CX / 8) * SX + e % (CX / 8) * 8) = x[q];
            }
        };
        auto st = [&](int h, const Rows& r) {
#pragma unroll
            for (int q = 0; q < NZ; ++q) {
                const int e = tid + 256 * q;
                if (e < QZ) *(bf16x8*)(sZ[h & 1] + e / (CZ / 8) * SZ + e % (CZ / 8) * 8) = r.z[q];
            }
            st_x(h + 1, r.x);
        };
        Rows ra, rb;
        {
            bf16x8 x0[NX], x1[NX];
            ld_x(r0 - 1, r0 < r1, x0);
            ld_x(r0, r0 < r1, x1);
            ld(r0, ra);
            ld(r0 + 1, rb);
            __syncthreads(); /* the item before has read its last rows */
            st_x(r0 - 1, x0);
            st_x(r0, x1);
            st(r0, ra);
        }
        __syncthreads();
        /* row h's products; row h + 1 to LDS, loaded two rows of products
         * ago, row h + 2 on its way */
        auto row = [&](int h, Rows& next, Rows& after) {
            ld(h + 2, after);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int kc = 0; kc < 2; ++kc) {
                bf16x8 af[MW];
#pragma unroll
                for (int m = 0; m < MW; ++m)
                    af[m] = ld_tr<SZ>(sZ[h & 1] + (kc * 32 + px) * SZ + (mb0 + m) * 16 + ch);
#pragma unroll
                for (int tap = 0; tap < 9; ++tap) {
                    const bf16x8 bf =
                        ld_tr<SX>(sX[(h - 1 + tap / 3) & 3] + (kc * 32 + px + tap % 3) * SX + nb0 * 16 + ch);
#pragma unroll
                    for (int m = 0; m < MW; ++m) acc[tap][m] = mfma(af[m], bf, acc[tap][m]);
                }
                if (MW == 4) {
#pragma unroll
                    for (int m = 0; m < MW; ++m)
                        if (m == wv) accb = mfma(af[m], ones, accb);
                } else if (NBI == 1 || wv == 0) {
                    accb = mfma(af[0], ones, accb);
                }
            }
            st(h + 1, next);
            __syncthreads();
        };
#pragma unroll 1
        for (int h = r0; h < r0 + it.R; h += 2) {
            row(h, rb, ra);
            if (h + 1 < r0 + it.R) row(h + 1, ra, rb);
        }
    }
    /* the halves' sums meet in LDS */
    if (half == 1) {
#pragma unroll
        for (int tap = 0; tap < 9; ++tap)
#pragma unroll
            for (int m = 0; m < MW; ++m) lds.sum[tap * MW + m][tid] = acc[tap][m];
        lds.sum[NA - 1][tid] = accb;
    }
    __syncthreads();
    if (half == 1) return;
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
        for (int m = 0; m < MW; ++m) acc[tap][m] += lds.sum[tap * MW + m][tid];
    accb += lds.sum[NA - 1][tid];
    const int ci = nb0 * 16 + (l & 15), c4 = 4 * (l >> 4);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
        for (int m = 0; m < MW; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                unsafeAtomicAdd(&dw[((size_t)tap * COP + (mb0 + m) * 16 + c4 + r) * CIP + ci], acc[tap][m][r]);
    if ((l & 15) == 0 && (MB == 4 || wv == 0)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) unsafeAtomicAdd(&db[(MB == 4 ? wv * 16 : 0) + c4 + r], accb[r]);
    }
}

/* prediction = base + out[0..2]; masked squared error and its gradient
 * dOut (bf16, kNarrow channels) = 2 m (pred - tgt) / (3 sum m), the sum of
 * the mask at *nmask.  Bound: HBM (72 bytes a pixel), and the additions to
 * the loss, about 10 ns each one after another: one for 1024 threads and at
 * most 512 of them.  With one for 256 threads, at most 2048: a 983 x 1051
 * image 34.8 us (two take 31 now), two of 251 x 268 8.4 (4.1 now). */
__global__ void __launch_bounds__(1024) k_loss(const float* __restrict__ out, const float* __restrict__ base,
                                              const float* __restrict__ tgt, const float* __restrict__ msk,
                                              long npix, const double* __restrict__ nmask, hd_cnn_scales sc,
                                              float* __restrict__ pred, bf16* __restrict__ dOut,
                                              double* __restrict__ loss)
{
    __shared__ double red[16];
    double s = 0;
    const float dsc[3] = {sc.d_u, sc.d_v, sc.d_z};
    const float nm = (float)nmask[0];
    const float inv_norm = nm > 0 ? 1.f / (3.f * nm) : 0.f;
    for (long p = blockIdx.x * 1024L + threadIdx.x; p < npix; p += gridDim.x * 1024L) {
        const float m = msk[p];
        const f32x4 o = *(const f32x4*)(out + p * kOut4);
        bf16x8 g = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float pr = base[p * 3 + c] + dsc[c] * o[c];
            pred[p * 3 + c] = pr;
            if (m != 0.f) {   /* pixels outside the mask neither add loss nor gradient */
                const float d = (pr - tgt[p * 3 + c]) / dsc[c];   /* increment error in d units */
                s += (double)(m * d * d);
                g[c] = (bf16)(2.f * m * d * inv_norm);
            }
        }
        if (dOut) *(bf16x8*)(dOut + p * kNarrow) = g;
    }
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) s += __shfl_xor(s, k);
    if (lane == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    s = red[lane & 15];
#pragma unroll
    for (int k = 8; k > 0; k >>= 1) s += __shfl_xor(s, k);
    if (lane == 0) atomicAdd(loss, s * (double)inv_norm);
}

/* One layer's parameters on the device. */
struct LayerDev {
    float *w, *dw, *mw, *vw, *b, *db, *mb, *vb;
    bf16 *w16, *wT16;
    int cin, cout;
};

__device__ __forceinline__ float adam_one(float* w, const float* g, float* m, float* v, long i, float lr, float bc1,
                                          float bc2)
{
    const float gi = g[i];
    const float mi = 0.9f * m[i] + 0.1f * gi;
    const float vi = 0.999f * v[i] + 0.001f * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float x = w[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + 1e-8f);
    w[i] = x;
    return x;
}

/* Adam on every layer's weights and biases (grid.y: the layer), with the
 * BF16 copies of the weights as k_wcast writes them: one launch for the
 * network. */
__global__ void __launch_bounds__(256) k_adam(const LayerDev* __restrict__ layers, float lr, float bc1, float bc2)
{
    const LayerDev& y = layers[blockIdx.y];
    const int cin = y.cin, cout = y.cout;
    const long n = 9L * cin * cout;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        const int ci = (int)(i % cin);
        const long q = i / cin;
        const int co = (int)(q % cout), tap = (int)(q / cout);
        const bf16 x = (bf16)adam_one(y.w, y.dw, y.mw, y.vw, i, lr, bc1, bc2);
        y.w16[i] = x;
        y.wT16[((size_t)(8 - tap) * cin + ci) * cout + co] = x;
    }
    if (blockIdx.x == 0 && (int)threadIdx.x < cout) adam_one(y.b, y.db, y.mb, y.vb, threadIdx.x, lr, bc1, bc2);
}

/* w16[tap][co][ci] = bf16(w32), wT16[8 - tap][ci][co] = bf16(w32) */
__global__ void __launch_bounds__(256) k_wcast(const float* __restrict__ w32, int cin, int cout,
                                               bf16* __restrict__ w16, bf16* __restrict__ wT16)
{
    const long n = 9L * cin * cout;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        const int ci = (int)(i % cin);
        const long q = i / cin;
        const int co = (int)(q % cout), tap = (int)(q / cout);
        const bf16 x = (bf16)w32[i];
        w16[i] = x;
        wT16[((size_t)(8 - tap) * cin + ci) * cout + co] = x;
    }
}

/* FP32 host images -> BF16 input and the FP32 base u, v, z */
__global__ void __launch_bounds__(256) k_load_x(const float* __restrict__ x8, long npix, bf16* __restrict__ x0,
                                                float* __restrict__ base)
{
    for (long p = blockIdx.x * 256L + threadIdx.x; p < npix; p += gridDim.x * 256L) {
        for (int c = 0; c < HD_CNN_CIN; ++c) x0[p * kNarrow + c] = (bf16)x8[p * HD_CNN_CIN + c];
        for (int c = 0; c < 3; ++c) base[p * 3 + c] = x8[p * HD_CNN_CIN + c];
    }
}

/* One sample of the store -> image d of the batch, its mask's sum added to
 * *nmask (whole numbers: the order does not matter) */
__global__ void __launch_bounds__(256) k_gather(const bf16* __restrict__ sx, const float* __restrict__ sbase,
                                                const float* __restrict__ stgt, const float* __restrict__ smsk,
                                                long npix, bf16* __restrict__ x0, float* __restrict__ base,
                                                float* __restrict__ tgt, float* __restrict__ msk,
                                                double* __restrict__ nmask)
{
    __shared__ double red[4];
    double s = 0;
    for (long p = blockIdx.x * 256L + threadIdx.x; p < npix; p += gridDim.x * 256L) {
        *(bf16x8*)(x0 + p * kNarrow) = *(const bf16x8*)(sx + p * kNarrow);
        for (int c = 0; c < 3; ++c) {
            base[p * 3 + c] = sbase[p * 3 + c];
            tgt[p * 3 + c] = stgt[p * 3 + c];
        }
        const float m = smsk[p];
        msk[p] = m;
        s += (double)m;
    }
    for (int k = 32; k > 0; k >>= 1) s += __shfl_down(s, k, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(nmask, red[0] + red[1] + red[2] + red[3]);
}

/* A context's state -> sample input (8 BF16 channels), FP32 base, mask */
__global__ void __launch_bounds__(256) k_pack(const HdDev* __restrict__ dv, hd_cnn_scales s, float q, float zb,
                                              bf16* __restrict__ xs, float* __restrict__ base, float* __restrict__ msk)
{
    const HdDevG& d = reinterpret_cast<const HdDevG*>(dv)[0];
    const long npix = (long)(d.N + 3) * (d.M + 3);
    for (long p = blockIdx.x * 256L + threadIdx.x; p < npix; p += gridDim.x * 256L) {
        /* state channels only on wet cells: elsewhere the solver's fields
         * carry values no equation reads (they may even be non-finite) */
        const bool wet = d.khouot[p] == 0;
        const float u = wet ? (float)(d.u[p] / s.s_u) : 0.f;
        const float v = wet ? (float)(d.v[p] / s.s_v) : 0.f;
        const float z = wet ? (float)(d.z[p] / s.s_z) : 0.f;
        const float bed = wet ? (float)(d.dH[p] / s.s_b) : 0.f;
        const float ch[HD_CNN_CIN] = {u, v, z, bed, wet ? 1.f : 0.f, q / s.s_q, zb / s.s_z, (float)(d.h[p] / s.s_h)};
        /* the network sees every channel clipped to [-8, 8]; the residual
         * base keeps the unclipped u, v, z */
        for (int c = 0; c < HD_CNN_CIN; ++c) xs[p * HD_CNN_CIN + c] = (bf16)fminf(fmaxf(ch[c], -8.f), 8.f);
        base[p * 3 + 0] = u;
        base[p * 3 + 1] = v;
        base[p * 3 + 2] = z;
        if (msk) msk[p] = wet ? 1.f : 0.f;
    }
}

/* A context's u, v, z -> normalised FP32 target */
__global__ void __launch_bounds__(256) k_target(const HdDev* __restrict__ dv, hd_cnn_scales s, float* __restrict__ tgt)
{
    const HdDevG& d = reinterpret_cast<const HdDevG*>(dv)[0];
    const long npix = (long)(d.N + 3) * (d.M + 3);
    for (long p = blockIdx.x * 256L + threadIdx.x; p < npix; p += gridDim.x * 256L) {
        const bool wet = d.khouot[p] == 0;
        tgt[p * 3 + 0] = wet ? (float)(d.u[p] / s.s_u) : 0.f;
        tgt[p * 3 + 1] = wet ? (float)(d.v[p] / s.s_v) : 0.f;
        tgt[p * 3 + 2] = wet ? (float)(d.z[p] / s.s_z) : 0.f;
    }
}

/* Network output (normalised increments) -> the context's wet cells, FP64 */
__global__ void __launch_bounds__(256) k_unpack(const HdDev* __restrict__ dv, hd_cnn_scales s,
                                                const float* __restrict__ out)
{
    const HdDevG& d = reinterpret_cast<const HdDevG*>(dv)[0];
    const int N = d.N, M = d.M, W = d.W;
    const long npix = (long)(N + 3) * W;
    for (long p = blockIdx.x * 256L + threadIdx.x; p < npix; p += gridDim.x * 256L) {
        const int i = (int)(p / W), j = (int)(p % W);
        if (i < 1 || i > N || j < 1 || j > M || d.khouot[p] != 0) continue;
        d.u[p] += (double)s.s_u * (double)s.d_u * (double)out[p * kOut4 + 0];
        d.v[p] += (double)s.s_v * (double)s.d_v * (double)out[p * kOut4 + 1];
        d.z[p] += (double)s.s_z * (double)s.d_z * (double)out[p * kOut4 + 2];
    }
}

/* The forward tiles (4 rows x 64 columns of the image) that lie within
 * `rad` cells (Chebyshev distance) of a wet cell of [1,N]x[1,M]: one wave
 * per tile, sixteen to a block, scans the tile grown by rad on every side;
 * the list order is arbitrary (each tile's outputs do not depend on it).
 * *count must be zero on entry. */
__global__ void __launch_bounds__(1024) k_active_tiles(const HdDev* __restrict__ dv, int rad, int* __restrict__ list,
                                                       int* __restrict__ count)
{
    __shared__ int found[16];
    const HdDevG& d = reinterpret_cast<const HdDevG*>(dv)[0];
    const int N = d.N, M = d.M, W = d.W, H = N + 3;
    const int tilesW = (W + 63) >> 6;
    const int wave = wave_in_block(), lane = (int)threadIdx.x & 63;
    const int t = blockIdx.x * 16 + wave, tw = t % tilesW, th = t / tilesW;
    const int i0 = max(th * 4 - rad, 1), i1 = th * 4 < H ? min(th * 4 + 3 + rad, N) : 0; /* no row past the last tile */
    const int j0 = max(tw * 64 - rad, 1), j1 = min(tw * 64 + 63 + rad, M);
    /* three rows of 21 lanes with four columns each: a load of 16 bytes for
     * every three rows up to 84 columns wide; one addition to the count per
     * 16 tiles (one per tile was most of 15 us on a 983 x 1051 grid, 8.5 now) */
    typedef int int4u __attribute__((ext_vector_type(4), aligned(4)));
    const int g = lane / 21, q = lane % 21;
    int any = 0;
    if (g < 3)
        for (int jb = j0; jb <= j1; jb += 84) {
            int j = jb + 4 * q;
            j = j < W - 4 ? j : W - 4;
#pragma unroll 6
            for (int i = i0 + g; i <= i1; i += 3) {
                const int4u k = *(HD_GLOBAL_AS const int4u*)(d.khouot + (long)i * W + j);
#pragma unroll
                for (int e = 0; e < 4; ++e) any |= (k[e] == 0) & (j + e >= j0) & (j + e <= j1);
            }
        }
    const bool mine = __any(any);
    if (lane == 0) found[wave] = mine;
    __syncthreads();
    if (wave != 0) return;
    const bool f = lane < 16 && found[lane & 15];
    const unsigned long long m = __ballot(f);
    int base = 0;
    if (lane == 0 && m) base = atomicAdd(count, __popcll(m));
    base = __builtin_amdgcn_readfirstlane(base);
    if (f) list[base + __popcll(m & ((1ull << lane) - 1))] = blockIdx.x * 16 + lane;
}

__global__ void k_zero_int(int* p) { *p = 0; }

__global__ void k_mfma_check(const bf16* A, const bf16* B, float* D)
{
    const int l = threadIdx.x;
    bf16x8 a, b;
    for (int e = 0; e < 8; ++e) {
        a[e] = A[(l % 16) * 32 + 8 * (l / 16) + e];
        b[e] = B[(8 * (l / 16) + e) * 16 + l % 16];
    }
    f32x4 c = f32x4{0.f, 0.f, 0.f, 0.f};
    c = mfma(a, b, c);
    for (int r = 0; r < 4; ++r) D[(4 * (l / 16) + r) * 16 + l % 16] = c[r];
}

struct Layer {
    int cin = 0, cout = 0;
    float *w32 = nullptr, *b32 = nullptr, *dw = nullptr, *db = nullptr;
    float *mw = nullptr, *vw = nullptr, *mb = nullptr, *vb = nullptr;
    bf16 *w16 = nullptr, *wT16 = nullptr;
    size_t nw() const { return (size_t)9 * cin * cout; }
};

inline int nblk(long n) { long b = (n + 255) / 256; return (int)(b < 4096 ? (b > 0 ? b : 1) : 4096); }

} // namespace

struct hd_cnn {
    int device = 0;
    hipStream_t stream = nullptr;
    int H = 0, W = 0, B = 0, L = 0;
    long P = 0;   /* pixels per image */
    std::vector<Layer> layer;
    hd_cnn_scales sc{1, 1, 1, 1, 1, 1, 1, 1, 1};
    std::vector<void*> allocs;
    bf16* x0 = nullptr;                 /* [B][P][8] */
    float* base = nullptr;              /* [B][P][3] */
    float *tgt = nullptr, *msk = nullptr, *pred = nullptr;
    std::vector<bf16*> act;             /* act[1..L-1]: [B][P][64] */
    std::vector<unsigned char*> gate;   /* gate[0..L-2]: which channels the layer's ReLU passed, [B][P][8] bytes */
    float* out = nullptr;               /* [B][P][4] */
    float* dA = nullptr;                /* [B][P][64] */
    bf16 *dZ = nullptr, *dZ2 = nullptr; /* [B][P][64]: a layer's gradient and the one below's */
    bf16* dOut = nullptr;               /* [B][P][8] */
    float* grads = nullptr;             /* every layer's dw and db */
    size_t ngrads = 0;
    LayerDev* ldev = nullptr;
    double* loss = nullptr;
    int nb = 0;                         /* images in the batch */
    double* nmask = nullptr;            /* sum of the batch's mask */
    int step = 0;
    /* sample store */
    int nsamp = 0;
    bf16* sx = nullptr;                 /* [n][P][8] */
    /* tile-sparse inference (hd_cnn_predict_into_ctx) */
    bool sparse = true;
    int* tlist = nullptr;               /* [tiles of one image] */
    int* tcount = nullptr;              /* [1] */
    const int* tl = nullptr;            /* the list the next forward uses (nullptr: all tiles) */
    float *sbase = nullptr, *stgt = nullptr, *smsk = nullptr;
    std::string err;
};

static std::string g_cnn_err;

static int cfail(hd_cnn* n, int code, const std::string& m)
{
    if (n) n->err = m;
    g_cnn_err = m;
    return code;
}

#define CHK(n, x)                                                                      \
    do {                                                                               \
        hipError_t e_ = (x);                                                           \
        if (e_ != hipSuccess) return cfail((n), HD_EHIP, std::string(#x ": ") + hipGetErrorString(e_)); \
    } while (0)

/* zero-filled device allocation; the fill runs on the network's
 * (non-blocking) stream and has finished when this returns, so it is
 * ordered before everything queued on that stream afterwards */
static int calloc_dev(hd_cnn* n, void** p, size_t bytes)
{
    if (hipMalloc(p, bytes ? bytes : 8) != hipSuccess) return cfail(n, HD_ENOMEM, "hipMalloc (network)");
    n->allocs.push_back(*p);
    if (hipMemsetAsync(*p, 0, bytes ? bytes : 8, n->stream) != hipSuccess ||
        hipStreamSynchronize(n->stream) != hipSuccess)
        return cfail(n, HD_EHIP, "hipMemsetAsync");
    return HD_OK;
}

/* splitmix64 -> uniform [-1, 1) */
static double rnd(uint64_t& s)
{
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
}

static int refresh_layer(hd_cnn* n, int l)
{
    Layer& y = n->layer[l];
    hipLaunchKernelGGL(k_wcast, dim3(nblk((long)y.nw())), dim3(256), 0, n->stream, y.w32, y.cin, y.cout, y.w16, y.wT16);
    CHK(n, hipGetLastError());
    return HD_OK;
}

/* Rows per item such that the items fill the 512 resident workgroups (two on
 * each CU) in whole rounds, weighing the rows an item reads beyond its own
 * and, in rows' time, what each workgroup adds at its end (k_wgrad). */
static ConvItems conv_items(const hd_cnn* n, int nimg, int width, double add = 0)
{
    ConvItems c{};
    c.H = n->H;
    c.W = n->W;
    c.cols = (n->W + width - 1) / width;
    double best = 0;
    for (int R = 4; R <= 64; ++R) {
        const int rows = (n->H + R - 1) / R;
        const long items = (long)nimg * rows * c.cols;
        const double cost = (double)((items + 511) / 512) * (R + 1.5) + add * (items < 512 ? items : 512);
        if (c.R == 0 || cost < best) {
            best = cost;
            c.R = R;
            c.rows = rows;
            c.total = (int)items;
        }
    }
    return c;
}

template <int EPI>
static void conv(hd_cnn* n, const bf16* X, const Layer& y, bool transposed, int nimg, bf16* Y, unsigned char* gate,
                 float* Yf, bool store_f = true)
{
    ConvItems it = conv_items(n, nimg, EPI == EPI_LINEAR ? 64 : 32);
    int grid = it.total < 512 ? it.total : 512;
    if (n->tl) {
        it.tl = n->tl;
        it.tn = n->tcount;
        grid = 512;
    }
    hipLaunchKernelGGL((k_conv<EPI>), dim3(grid), dim3(256), 0, n->stream, X, transposed ? y.wT16 : y.w16, y.b32, it, Y,
                       gate, Yf, store_f ? 1 : 0);
}

template <int MB, int NBI>
static void wgrad(hd_cnn* n, const bf16* X, const bf16* dZ, const Layer& y, int nimg)
{
    const ConvItems it = conv_items(n, nimg, 64, 0.017);
    hipLaunchKernelGGL((k_wgrad<MB, NBI>), dim3(it.total < 512 ? (it.total + 1) / 2 : 256), dim3(512), 0, n->stream, X,
                       dZ, it, y.dw, y.db);
}

/* The gates are written in every pass: a backward pass takes the activations
 * of the last one, a prediction's too, and the gates have to be that one's. */
static int forward(hd_cnn* n, int nimg)
{
    const int L = n->L;
    conv<EPI_RELU>(n, n->x0, n->layer[0], false, nimg, n->act[1], n->gate[0], nullptr);
    for (int l = 1; l <= L - 2; ++l)
        conv<EPI_RESRELU>(n, n->act[l], n->layer[l], false, nimg, n->act[l + 1], n->gate[l], nullptr);
    conv<EPI_LINEAR>(n, n->act[L - 1], n->layer[L - 1], false, nimg, nullptr, nullptr, n->out);
    CHK(n, hipGetLastError());
    return HD_OK;
}

/* the loss of the last forward (and dOut), left at n->loss */
static int loss_and_grad(hd_cnn* n, int nimg, bool grad)
{
    long npix = (long)nimg * n->P;
    CHK(n, hipMemsetAsync(n->loss, 0, sizeof(double), n->stream));
    const long blocks = (npix + 1023) / 1024;
    hipLaunchKernelGGL(k_loss, dim3((unsigned)(blocks < 512 ? blocks : 512)), dim3(1024), 0, n->stream, n->out, n->base,
                       n->tgt, n->msk, npix, n->nmask, n->sc, n->pred, grad ? n->dOut : nullptr, n->loss);
    CHK(n, hipGetLastError());
    return HD_OK;
}

/* waits for the stream, the loss in *loss */
static int finish(hd_cnn* n, double* loss)
{
    if (loss) CHK(n, hipMemcpyAsync(loss, n->loss, sizeof(double), hipMemcpyDeviceToHost, n->stream));
    CHK(n, hipStreamSynchronize(n->stream));
    return HD_OK;
}

static int backward(hd_cnn* n, int nimg)
{
    const int L = n->L;
    CHK(n, hipMemsetAsync(n->grads, 0, n->ngrads * 4, n->stream));
    wgrad<1, 4>(n, n->act[L - 1], n->dOut, n->layer[L - 1], nimg);
    conv<EPI_BWD_SET>(n, n->dOut, n->layer[L - 1], true, nimg, n->dZ, n->gate[L - 2], n->dA);
    bf16 *z = n->dZ, *zn = n->dZ2;
    for (int l = L - 2; l >= 1; --l) {
        wgrad<4, 4>(n, n->act[l], z, n->layer[l], nimg);
        /* dA itself is not read below layer 1 */
        conv<EPI_BWD_ADD>(n, z, n->layer[l], true, nimg, zn, n->gate[l - 1], n->dA, l > 1);
        std::swap(z, zn);
    }
    wgrad<4, 1>(n, n->x0, z, n->layer[0], nimg);
    CHK(n, hipGetLastError());
    return HD_OK;
}

static int adam(hd_cnn* n, float lr)
{
    n->step += 1;
    float bc1 = 1.f - std::pow(0.9f, (float)n->step), bc2 = 1.f - std::pow(0.999f, (float)n->step);
    hipLaunchKernelGGL(k_adam, dim3(36, n->L), dim3(256), 0, n->stream, n->ldev, lr, bc1, bc2);
    CHK(n, hipGetLastError());
    return HD_OK;
}

extern "C" {

const char* hd_cnn_last_error(const hd_cnn* n) { return n ? n->err.c_str() : g_cnn_err.c_str(); }

int hd_cnn_create(int device, int H, int W, int batch, int layers, uint64_t seed, hd_cnn** out)
{
    if (!out || H < 1 || W < 1 || batch < 1 || layers < 3) return cfail(nullptr, HD_EINVAL, "hd_cnn_create: bad arguments");
    if (hipSetDevice(device) != hipSuccess) return cfail(nullptr, HD_EHIP, "hipSetDevice");
    hd_cnn* n = new hd_cnn();
    n->device = device;
    n->H = H; n->W = W; n->B = batch; n->L = layers;
    n->P = (long)H * W;
    if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess) {
        delete n;
        return cfail(nullptr, HD_EHIP, "hipStreamCreate");
    }
    int rc;
    const size_t PB = (size_t)n->P * batch;
    n->layer.resize(layers);
    for (int l = 0; l < layers; ++l) {
        Layer& y = n->layer[l];
        y.cin = l == 0 ? kCinPad : kWidth;
        y.cout = l == layers - 1 ? kOutPad : kWidth;
        n->ngrads += y.nw() + y.cout;
    }
    if ((rc = calloc_dev(n, (void**)&n->grads, n->ngrads * 4)) ||
        (rc = calloc_dev(n, (void**)&n->ldev, layers * sizeof(LayerDev)))) {
        hd_cnn_destroy(n);
        return rc;
    }
    float* grad = n->grads;
    std::vector<LayerDev> ld(layers);
    uint64_t s = seed;
    for (int l = 0; l < layers; ++l) {
        Layer& y = n->layer[l];
        size_t nw = y.nw();
        y.dw = grad;
        y.db = grad + nw;
        grad += nw + y.cout;
        void** f32[] = {(void**)&y.w32, (void**)&y.mw, (void**)&y.vw};
        for (auto p : f32)
            if ((rc = calloc_dev(n, p, nw * 4))) { hd_cnn_destroy(n); return rc; }
        void** fb[] = {(void**)&y.b32, (void**)&y.mb, (void**)&y.vb};
        for (auto p : fb)
            if ((rc = calloc_dev(n, p, (size_t)y.cout * 4))) { hd_cnn_destroy(n); return rc; }
        if ((rc = calloc_dev(n, (void**)&y.w16, nw * 2)) || (rc = calloc_dev(n, (void**)&y.wT16, nw * 2))) {
            hd_cnn_destroy(n);
            return rc;
        }
        /* He-uniform over the real fan-in; padded input channels and padded
         * outputs stay zero; the last layer starts small (near-identity
         * residual prediction) */
        int cin_real = l == 0 ? HD_CNN_CIN : kWidth;
        int cout_real = l == layers - 1 ? HD_CNN_COUT : kWidth;
        double a = std::sqrt(6.0 / (9.0 * cin_real)) * (l == layers - 1 ? 0.1 : (l == 0 ? 1.0 : 0.5));
        std::vector<float> w(nw, 0.f);
        for (int tap = 0; tap < 9; ++tap)
            for (int co = 0; co < cout_real; ++co)
                for (int ci = 0; ci < cin_real; ++ci) w[((size_t)tap * y.cout + co) * y.cin + ci] = (float)(a * rnd(s));
        if (hipMemcpy(y.w32, w.data(), nw * 4, hipMemcpyHostToDevice) != hipSuccess) {
            hd_cnn_destroy(n);
            return cfail(nullptr, HD_EHIP, "hipMemcpy weights");
        }
        if ((rc = refresh_layer(n, l))) { hd_cnn_destroy(n); return rc; }
        ld[l] = LayerDev{y.w32, y.dw, y.mw, y.vw, y.b32, y.db, y.mb, y.vb, y.w16, y.wT16, y.cin, y.cout};
    }
    if (hipMemcpy(n->ldev, ld.data(), layers * sizeof(LayerDev), hipMemcpyHostToDevice) != hipSuccess) {
        hd_cnn_destroy(n);
        return cfail(nullptr, HD_EHIP, "hipMemcpy layer table");
    }
    n->act.assign(layers, nullptr);
    n->gate.assign(layers, nullptr);
    for (int l = 1; l <= layers - 1; ++l)
        if ((rc = calloc_dev(n, (void**)&n->act[l], PB * kWidth * 2))) { hd_cnn_destroy(n); return rc; }
    for (int l = 0; l <= layers - 2; ++l)
        if ((rc = calloc_dev(n, (void**)&n->gate[l], PB * (kWidth / 8)))) { hd_cnn_destroy(n); return rc; }
    if ((rc = calloc_dev(n, (void**)&n->x0, PB * kNarrow * 2)) || (rc = calloc_dev(n, (void**)&n->base, PB * 3 * 4)) ||
        (rc = calloc_dev(n, (void**)&n->tgt, PB * 3 * 4)) || (rc = calloc_dev(n, (void**)&n->msk, PB * 4)) ||
        (rc = calloc_dev(n, (void**)&n->pred, PB * 3 * 4)) || (rc = calloc_dev(n, (void**)&n->out, PB * kOut4 * 4)) ||
        (rc = calloc_dev(n, (void**)&n->dA, PB * kWidth * 4)) || (rc = calloc_dev(n, (void**)&n->dZ, PB * kWidth * 2)) ||
        (rc = calloc_dev(n, (void**)&n->dZ2, PB * kWidth * 2)) || (rc = calloc_dev(n, (void**)&n->dOut, PB * kNarrow * 2)) ||
        (rc = calloc_dev(n, (void**)&n->nmask, 8)) ||
        (rc = calloc_dev(n, (void**)&n->loss, 8)) ||
        (rc = calloc_dev(n, (void**)&n->tlist, (size_t)((W + 63) / 64) * ((H + 3) / 4) * 4)) ||
        (rc = calloc_dev(n, (void**)&n->tcount, 4))) {
        hd_cnn_destroy(n);
        return rc;
    }
    if (hipStreamSynchronize(n->stream) != hipSuccess) { hd_cnn_destroy(n); return cfail(nullptr, HD_EHIP, "sync"); }
    *out = n;
    return HD_OK;
}

int hd_cnn_destroy(hd_cnn* n)
{
    if (!n) return HD_OK;
    hipSetDevice(n->device);
    if (n->stream) hipStreamSynchronize(n->stream);
    for (void* p : n->allocs) hipFree(p);
    if (n->stream) hipStreamDestroy(n->stream);
    delete n;
    return HD_OK;
}

int hd_cnn_set_scales(hd_cnn* n, const hd_cnn_scales* s)
{
    if (!n || !s || !(s->d_u > 0) || !(s->d_v > 0) || !(s->d_z > 0)) return HD_EINVAL;
    n->sc = *s;
    return HD_OK;
}

int hd_cnn_set_sparse(hd_cnn* n, int on)
{
    if (!n) return HD_EINVAL;
    n->sparse = on != 0;
    return HD_OK;
}

int hd_cnn_layer_dims(const hd_cnn* n, int l, int* cin, int* cout)
{
    if (!n || l < 0 || l >= n->L) return HD_EINVAL;
    if (cin) *cin = n->layer[l].cin;
    if (cout) *cout = n->layer[l].cout;
    return HD_OK;
}

int hd_cnn_get_layer(hd_cnn* n, int l, float* host_w, float* host_b)
{
    if (!n || l < 0 || l >= n->L) return HD_EINVAL;
    const Layer& y = n->layer[l];
    CHK(n, hipStreamSynchronize(n->stream));
    if (host_w) CHK(n, hipMemcpy(host_w, y.w32, y.nw() * 4, hipMemcpyDeviceToHost));
    if (host_b) CHK(n, hipMemcpy(host_b, y.b32, (size_t)y.cout * 4, hipMemcpyDeviceToHost));
    return HD_OK;
}

int hd_cnn_set_layer(hd_cnn* n, int l, const float* host_w, const float* host_b)
{
    if (!n || l < 0 || l >= n->L) return HD_EINVAL;
    Layer& y = n->layer[l];
    CHK(n, hipStreamSynchronize(n->stream));
    if (host_w) CHK(n, hipMemcpy(y.w32, host_w, y.nw() * 4, hipMemcpyHostToDevice));
    if (host_b) CHK(n, hipMemcpy(y.b32, host_b, (size_t)y.cout * 4, hipMemcpyHostToDevice));
    CHK(n, hipMemsetAsync(y.mw, 0, y.nw() * 4, n->stream));
    CHK(n, hipMemsetAsync(y.vw, 0, y.nw() * 4, n->stream));
    CHK(n, hipMemsetAsync(y.mb, 0, (size_t)y.cout * 4, n->stream));
    CHK(n, hipMemsetAsync(y.vb, 0, (size_t)y.cout * 4, n->stream));
    int rc = refresh_layer(n, l);
    if (rc) return rc;
    CHK(n, hipStreamSynchronize(n->stream));
    return HD_OK;
}

int hd_cnn_get_grad(hd_cnn* n, int l, float* host_dw, float* host_db)
{
    if (!n || l < 0 || l >= n->L) return HD_EINVAL;
    const Layer& y = n->layer[l];
    CHK(n, hipStreamSynchronize(n->stream));
    if (host_dw && host_db == host_dw + y.nw() && y.db == y.dw + y.nw()) { /* adjacent on both sides: one copy */
        CHK(n, hipMemcpy(host_dw, y.dw, (y.nw() + y.cout) * 4, hipMemcpyDeviceToHost));
        return HD_OK;
    }
    if (host_dw) CHK(n, hipMemcpy(host_dw, y.dw, y.nw() * 4, hipMemcpyDeviceToHost));
    if (host_db) CHK(n, hipMemcpy(host_db, y.db, (size_t)y.cout * 4, hipMemcpyDeviceToHost));
    return HD_OK;
}

int hd_cnn_load_batch(hd_cnn* n, int b, const float* host_x, const float* host_y, const float* host_m)
{
    if (!n || b < 1 || b > n->B || !host_x) return cfail(n, HD_EINVAL, "hd_cnn_load_batch: bad arguments");
    long npix = (long)b * n->P;
    float* tmp = nullptr;
    CHK(n, hipMalloc((void**)&tmp, (size_t)npix * HD_CNN_CIN * 4));
    hipError_t e = hipMemcpy(tmp, host_x, (size_t)npix * HD_CNN_CIN * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_load_x, dim3(nblk(npix)), dim3(256), 0, n->stream, tmp, npix, n->x0, n->base);
        e = hipStreamSynchronize(n->stream);
    }
    hipFree(tmp);
    if (e != hipSuccess) return cfail(n, HD_EHIP, hipGetErrorString(e));
    if (host_y) CHK(n, hipMemcpy(n->tgt, host_y, (size_t)npix * 3 * 4, hipMemcpyHostToDevice));
    double ms = 0;
    if (host_m) {
        CHK(n, hipMemcpy(n->msk, host_m, (size_t)npix * 4, hipMemcpyHostToDevice));
        for (long p = 0; p < npix; ++p) ms += host_m[p];
    }
    CHK(n, hipMemcpy(n->nmask, &ms, sizeof(double), hipMemcpyHostToDevice));
    n->nb = b;
    return HD_OK;
}

int hd_cnn_forward(hd_cnn* n, float* host_out)
{
    if (!n || n->nb < 1) return cfail(n, HD_ESTATE, "hd_cnn_forward: no batch loaded");
    int rc = forward(n, n->nb);
    if (rc) return rc;
    if ((rc = loss_and_grad(n, n->nb, false))) return rc;
    if (host_out) {
        CHK(n, hipStreamSynchronize(n->stream));
        CHK(n, hipMemcpy(host_out, n->pred, (size_t)n->nb * n->P * 3 * 4, hipMemcpyDeviceToHost));
    }
    return HD_OK;
}

int hd_cnn_backward(hd_cnn* n, double* loss)
{
    if (!n || n->nb < 1) return cfail(n, HD_ESTATE, "hd_cnn_backward: no batch loaded");
    int rc = loss_and_grad(n, n->nb, true);
    if (!rc) rc = backward(n, n->nb);
    if (!rc) rc = finish(n, loss);
    return rc;
}

int hd_cnn_adam(hd_cnn* n, float lr)
{
    if (!n) return HD_EINVAL;
    int rc = adam(n, lr);
    if (!rc) rc = finish(n, nullptr);
    return rc;
}

/* one wait for the whole step */
int hd_cnn_train_step(hd_cnn* n, float lr, double* loss)
{
    if (!n || n->nb < 1) return cfail(n, HD_ESTATE, "hd_cnn_forward: no batch loaded");
    int rc = forward(n, n->nb);
    if (!rc) rc = loss_and_grad(n, n->nb, true);
    if (!rc) rc = backward(n, n->nb);
    if (!rc) rc = adam(n, lr);
    if (!rc) rc = finish(n, loss);
    return rc;
}

int hd_cnn_data_alloc(hd_cnn* n, int count)
{
    if (!n || count < 1 || n->nsamp) return cfail(n, HD_EINVAL, "hd_cnn_data_alloc: bad arguments");
    size_t np = (size_t)n->P * count;
    int rc;
    if ((rc = calloc_dev(n, (void**)&n->sx, np * HD_CNN_CIN * 2)) || (rc = calloc_dev(n, (void**)&n->sbase, np * 3 * 4)) ||
        (rc = calloc_dev(n, (void**)&n->stgt, np * 3 * 4)) || (rc = calloc_dev(n, (void**)&n->smsk, np * 4)))
        return rc;
    n->nsamp = count;
    return HD_OK;
}

int hd_cnn_capture(hd_cnn* n, int idx, int role, hd_ctx* c, float q, float zb)
{
    if (!n || !c || idx < 0 || idx >= n->nsamp || (role != 0 && role != 1))
        return cfail(n, HD_EINVAL, "hd_cnn_capture: bad arguments");
    hipStream_t cs;
    int st;
    const HdDev* dv = hd_ctx_device_view(c, &cs, &st);
    HdDev hd;
    CHK(n, hipMemcpy(&hd, dv, sizeof(HdDev), hipMemcpyDeviceToHost));
    if ((long)(hd.N + 3) * (hd.M + 3) != n->P || hd.N + 3 != n->H) return cfail(n, HD_ESHAPE, "grid mismatch");
    CHK(n, hipStreamSynchronize(cs));
    size_t o = (size_t)idx * n->P;
    if (role == 0)
        hipLaunchKernelGGL(k_pack, dim3(nblk(n->P)), dim3(256), 0, n->stream, dv, n->sc, q, zb, n->sx + o * HD_CNN_CIN,
                           n->sbase + o * 3, n->smsk + o);
    else
        hipLaunchKernelGGL(k_target, dim3(nblk(n->P)), dim3(256), 0, n->stream, dv, n->sc, n->stgt + o * 3);
    CHK(n, hipGetLastError());
    CHK(n, hipStreamSynchronize(n->stream));
    return HD_OK;
}

static int gather(hd_cnn* n, const int* idx, int b)
{
    if (!idx || b < 1 || b > n->B) return cfail(n, HD_EINVAL, "sample list");
    for (int k = 0; k < b; ++k)
        if (idx[k] < 0 || idx[k] >= n->nsamp) return cfail(n, HD_EINVAL, "sample index out of range");
    CHK(n, hipMemsetAsync(n->nmask, 0, sizeof(double), n->stream));
    for (int k = 0; k < b; ++k) {
        const size_t o = (size_t)idx[k] * n->P, d = (size_t)k * n->P;
        hipLaunchKernelGGL(k_gather, dim3(nblk(n->P) < 1024 ? nblk(n->P) : 1024), dim3(256), 0, n->stream,
                           n->sx + o * kNarrow, n->sbase + o * 3, n->stgt + o * 3, n->smsk + o, n->P,
                           n->x0 + d * kNarrow, n->base + d * 3, n->tgt + d * 3, n->msk + d, n->nmask);
    }
    CHK(n, hipGetLastError());
    n->nb = b;
    return HD_OK;
}

int hd_cnn_train_samples(hd_cnn* n, const int* host_idx, int b, float lr, double* loss)
{
    if (!n) return HD_EINVAL;
    int rc = gather(n, host_idx, b);
    if (!rc) rc = hd_cnn_train_step(n, lr, loss);
    return rc;
}

int hd_cnn_eval_samples(hd_cnn* n, const int* host_idx, int b, double* loss)
{
    if (!n) return HD_EINVAL;
    int rc = gather(n, host_idx, b);
    if (!rc) rc = forward(n, b);
    if (!rc) rc = loss_and_grad(n, b, false);
    if (!rc) rc = finish(n, loss);
    return rc;
}

int hd_cnn_predict_into_ctx(hd_cnn* n, hd_ctx* c, float q, float zb)
{
    if (!n || !c) return HD_EINVAL;
    hipStream_t cs;
    int st;
    const HdDev* dv = hd_ctx_device_view(c, &cs, &st);
    HdDev hd;
    CHK(n, hipMemcpy(&hd, dv, sizeof(HdDev), hipMemcpyDeviceToHost));
    if ((long)(hd.N + 3) * (hd.M + 3) != n->P || hd.N + 3 != n->H) return cfail(n, HD_ESHAPE, "grid mismatch");
    if (st != 0) return cfail(n, HD_ESTATE, "context between half-steps");
    CHK(n, hipStreamSynchronize(cs));
    hipLaunchKernelGGL(k_pack, dim3(nblk(n->P)), dim3(256), 0, n->stream, dv, n->sc, q, zb, n->x0, n->base, nullptr);
    if (n->sparse) {
        /* Only the tiles within L - 1 cells of a wet cell: the first layer
         * reads the whole input image, and a layer's value at a cell is the
         * dense one wherever its 3x3 neighbours' values were, so with every
         * cell within L - 1 of a wet cell computed the network's output at
         * the wet cells is that of the dense pass, bit for bit. */
        int tiles = ((n->W + 63) / 64) * ((n->H + 3) / 4);
        hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, n->stream, n->tcount);
        hipLaunchKernelGGL(k_active_tiles, dim3((tiles + 15) / 16), dim3(1024), 0, n->stream, dv, n->L - 1, n->tlist, n->tcount);
        n->tl = n->tlist;
    }
    int rc = forward(n, 1);
    n->tl = nullptr;
    if (rc) return rc;
    hipLaunchKernelGGL(k_unpack, dim3(nblk(n->P)), dim3(256), 0, n->stream, dv, n->sc, n->out);
    CHK(n, hipGetLastError());
    CHK(n, hipStreamSynchronize(n->stream));
    return hd_flow_refresh(c);
}

int hd_cnn_mfma_check(int device, const float* host_a, const float* host_b, float* host_d)
{
    if (!host_a || !host_b || !host_d) return HD_EINVAL;
    if (hipSetDevice(device) != hipSuccess) return cfail(nullptr, HD_EHIP, "hipSetDevice");
    std::vector<bf16> a(16 * 32), b(32 * 16);
    for (int i = 0; i < 16 * 32; ++i) a[i] = (bf16)host_a[i];
    for (int i = 0; i < 32 * 16; ++i) b[i] = (bf16)host_b[i];
    bf16 *da = nullptr, *db = nullptr;
    float* dd = nullptr;
    int rc = HD_OK;
    if (hipMalloc((void**)&da, a.size() * 2) != hipSuccess || hipMalloc((void**)&db, b.size() * 2) != hipSuccess ||
        hipMalloc((void**)&dd, 256 * 4) != hipSuccess)
        rc = cfail(nullptr, HD_ENOMEM, "hipMalloc");
    if (!rc && (hipMemcpy(da, a.data(), a.size() * 2, hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(db, b.data(), b.size() * 2, hipMemcpyHostToDevice) != hipSuccess))
        rc = cfail(nullptr, HD_EHIP, "hipMemcpy");
    if (!rc) {
        hipLaunchKernelGGL(k_mfma_check, dim3(1), dim3(64), 0, 0, da, db, dd);
        if (hipDeviceSynchronize() != hipSuccess || hipMemcpy(host_d, dd, 256 * 4, hipMemcpyDeviceToHost) != hipSuccess)
            rc = cfail(nullptr, HD_EHIP, "mfma check");
    }
    if (da) hipFree(da);
    if (db) hipFree(db);
    if (dd) hipFree(dd);
    return rc;
}

} // extern "C"

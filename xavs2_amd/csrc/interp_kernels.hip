// Reference-plane producer for gfx950: border expansion of a plane
// (plane_expand_border, source/common/frame.c:470-507) and the 15 interpolated
// luma planes of a reference picture (interpolate_lcu_row over every LCU row,
// source/common/mc.c:593-785).
//
// Over the whole frame, the row-window algorithm of the reference computes
// every plane on x in [-4, W+4), y in [-4, H+4) from the border-expanded
// full-pel plane and then replicates that area outward, i.e.
//     plane_k(x, y) = interp_k(clamp(x, -4, W+3), clamp(y, -4, H+3)).
// One kernel computes the [-4, W+4) x [-4, H+4) area tile by tile (full-pel
// tile and its horizontal sums staged in LDS) and, in workgroups of its own,
// the 76-pixel frame around it.  The border kernel serves expand_border.  The horizontal sums of 8-bit
// pictures lie in [-4845, 22440], so the reference's int16 temporaries
// (mct_t, mc.c:466-496) hold them without wrapping and int32 is equivalent.
#include <algorithm>

#include "xme_internal.h"

namespace {

// INTPL_FILTERS, source/common/mc.c:73-78
__constant__ int8_t c_taps[4][8] = { { 0, 0, 0, 64, 0, 0, 0, 0 },
                                     { -1, 4, -10, 57, 19, -7, 3, -1 },
                                     { -1, 4, -11, 40, 40, -11, 4, -1 },
                                     { -1, 3, -7, 19, 57, -10, 4, -1 } };

struct Planes16 {
    uint8_t *p[16];
};

typedef short short2v __attribute__((ext_vector_type(2)));

constexpr int TX = 64;                // output columns per tile
constexpr int TY = 16;                // output rows per tile
constexpr int LX = TX / 4;            // threads of a tile's row
constexpr int NT = LX * TY;           // threads of a workgroup
constexpr int SPW = (TX + 8) / 4;     // staged dwords per row

__device__ __forceinline__ uint32_t clip_pel(int v) { return (uint32_t)(v < 0 ? 0 : (v > 255 ? 255 : v)); }

// Four clipped pixels (each 0..255 in an int) packed into one dword, byte i
// from p[i], with v_perm_b32.  Written as shifts and ors, the clips and the
// packing compile to v_ashr_pk_u8_i32; a build of the diagonal planes in that
// form gave wrong pixels (the cause was not isolated), so every plane packs
// this way.
__device__ __forceinline__ uint32_t pack_pels(uint32_t p0, uint32_t p1, uint32_t p2, uint32_t p3)
{
    return __builtin_amdgcn_perm(__builtin_amdgcn_perm(p3, p2, 0x0C0C0400u), __builtin_amdgcn_perm(p1, p0, 0x0C0C0400u),
                                 0x05040100u);
}

// Taps of a phase packed as two dwords of signed bytes (taps 0-3, 4-7).
__device__ __forceinline__ void packed_taps(int d, int &lo, int &hi)
{
    lo = (int)((uint32_t)(uint8_t)c_taps[d][0] | ((uint32_t)(uint8_t)c_taps[d][1] << 8) |
               ((uint32_t)(uint8_t)c_taps[d][2] << 16) | ((uint32_t)(uint8_t)c_taps[d][3] << 24));
    hi = (int)((uint32_t)(uint8_t)c_taps[d][4] | ((uint32_t)(uint8_t)c_taps[d][5] << 8) |
               ((uint32_t)(uint8_t)c_taps[d][6] << 16) | ((uint32_t)(uint8_t)c_taps[d][7] << 24));
}

// 8-tap filter of 8 pixels held as two dwords of (pixel - 128) signed bytes:
// sum C_k * p_k = sum C_k * (p_k - 128) + 128 * 64, with v_dot4_i32_i8.
__device__ __forceinline__ int fir8(int tlo, int thi, uint32_t p0, uint32_t p1, int base = 8192)
{
    return __builtin_amdgcn_sdot4(thi, (int)p1, __builtin_amdgcn_sdot4(tlo, (int)p0, base, false), false);
}

// A dword of a plane on its way to memory: the planes of a picture are not read
// again before all are written, and stored past the caches they leave at the
// rate of the memory (four 2160p references in turn: 61.9 -> 49.8 us each; one
// over and over, kept by the last-level cache, 51.4 -> 53.3).
__device__ __forceinline__ void stream_out(uint8_t *p, uint32_t v)
{
    __builtin_nontemporal_store(v, reinterpret_cast<uint32_t *>(p));
}

// Column j (bytes j of four row dwords) gathered into one dword, rows in order.
__device__ __forceinline__ void transpose4(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3, uint32_t (&col)[4])
{
    const uint32_t t01l = __builtin_amdgcn_perm(a1, a0, 0x05010400u);
    const uint32_t t01h = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
    const uint32_t t23l = __builtin_amdgcn_perm(a3, a2, 0x05010400u);
    const uint32_t t23h = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
    col[0] = __builtin_amdgcn_perm(t23l, t01l, 0x05040100u);
    col[1] = __builtin_amdgcn_perm(t23l, t01l, 0x07060302u);
    col[2] = __builtin_amdgcn_perm(t23h, t01h, 0x05040100u);
    col[3] = __builtin_amdgcn_perm(t23h, t01h, 0x07060302u);
}

// What one launch of the interpolation covers: the core columns x in
// [-4, W+4) of rows [ys, ye), the strips left and right of those rows, and the
// bands above -4 and below H+4 where asked for.
struct InterpGeom {
    int64_t stride;
    int W, H, frac;
    int xs, ys, ye;            // tiles of the core start at column xs <= -4, row ys
    int xb;                    // tiles of the bands start at column xb <= -PAD
    int gx, gxb;               // tiles of a row, in the core and in the bands
    int n_band, n_top;         // workgroups of both bands, and of the upper one
    int n_strip, n_tiles;      // workgroups of the strips, tiles of the core
};

constexpr int BORDER = XME_PAD - 4;      // rows of a band, columns of a strip
constexpr int BAND_ROWS = BORDER / 4;    // rows that a workgroup of a band fills

// The pixels a workgroup of the border needs, from the full-pel plane: column
// (xx + i), i in [0, N), of row yy of plane k.  Every plane is the 2-D filter
// with the taps of its two phases; phase 0 is the tap 64, with which the sums
// of a 1-D plane come out 64 times as large: (64 h + 2048) >> 12 is
// (h + 32) >> 6.  The rows and columns read lie within 7 of the core.
template <int N>
__device__ __forceinline__ void edge_pels(const uint8_t *__restrict__ P, int64_t stride, int xx, int yy, int k,
                                          uint32_t (&px)[N])
{
    int hl, hh;
    packed_taps(k & 3, hl, hh);
    int h[8][N];
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const uint8_t *row = P + (int64_t)(yy - 3 + r) * stride + xx - 4;   // xx % 4 == 0
        uint32_t d[3];
#pragma unroll
        for (int i = 0; i < 3; i++)
            d[i] = reinterpret_cast<const uint32_t *>(row)[i] ^ 0x80808080u;
#pragma unroll
        for (int i = 0; i < N; i++) {
            // bytes i + 1 .. i + 8
            const uint32_t lo = i == 3 ? d[1] : __builtin_amdgcn_alignbyte(d[1], d[0], (uint32_t)(i + 1));
            const uint32_t hi = i == 3 ? d[2] : __builtin_amdgcn_alignbyte(d[2], d[1], (uint32_t)(i + 1));
            h[r][i] = fir8(hl, hh, lo, hi);
        }
    }
    int t[8];
#pragma unroll
    for (int m = 0; m < 8; m++)
        t[m] = c_taps[k >> 2][m];
#pragma unroll
    for (int i = 0; i < N; i++) {
        int s = 2048;
#pragma unroll
        for (int r = 0; r < 8; r++)
            s += t[r] * h[r][i];
        px[i] = clip_pel(s >> 12);
    }
}

// The plane of index j (0..14) among those to fill: 1..15, or 2, 8 and 10
// where only the half-pel planes are asked for; 0 for none.
__device__ __forceinline__ int plane_index(int frac, int j)
{
    if (frac < 2)
        return j == 0 ? 2 : (j == 1 ? 8 : (j == 2 ? 10 : 0));
    return j < 15 ? j + 1 : 0;
}

// A workgroup of the bands: 64 columns of BAND_ROWS rows of every plane.  A
// thread computes 4 pixels of one plane once, in the core's first or last row
// (clamped to the core's columns), and stores them in each row.
__device__ __forceinline__ void fill_band(const Planes16 &pl, const InterpGeom &g, int b)
{
    const bool top = b < g.n_top;
    const int t = top ? b : b - g.n_top;
    const int k = plane_index(g.frac, (int)threadIdx.x / LX);
    const int x = g.xb + (t % g.gxb) * TX + ((int)threadIdx.x & (LX - 1)) * 4;
    if (k == 0 || x < -XME_PAD || x >= g.W + XME_PAD)
        return;
    uint32_t px[4];
    edge_pels(pl.p[0], g.stride, xme_clip3(-4, g.W, x), top ? -4 : g.H + 3, k, px);
    if (x < -4)
        px[1] = px[2] = px[3] = px[0];
    else if (x > g.W)
        px[0] = px[1] = px[2] = px[3];
    const uint32_t v = pack_pels(px[0], px[1], px[2], px[3]);
    uint8_t *o = pl.p[k] + (int64_t)((top ? -XME_PAD : g.H + 4) + (t / g.gxb) * BAND_ROWS) * g.stride + x;
#pragma unroll
    for (int r = 0; r < BAND_ROWS; r++)
        *reinterpret_cast<uint32_t *>(o + r * g.stride) = v;
}

// A workgroup of the strips: 16 rows of the left (b even) or right strip of a
// third of the planes.  A thread computes the pixel of one row and plane; the
// strips' dwords are then stored by rows.
__device__ __forceinline__ void fill_strip(const Planes16 &pl, const InterpGeom &g, int b, uint32_t *sV)
{
    const int np = g.frac < 2 ? 1 : 5, third = b % 3 * np, t = b / 3;
    const bool left = (t & 1) == 0;
    const int y0 = g.ys + (t >> 1) * TY;
    const int j = (int)threadIdx.x >> 4, y = y0 + ((int)threadIdx.x & 15);
    if (j < np && y < g.ye) {
        uint32_t v;
        if (left) {
            uint32_t px[1];
            edge_pels(pl.p[0], g.stride, -4, y, plane_index(g.frac, third + j), px);
            v = px[0];
        } else {
            uint32_t px[4];
            edge_pels(pl.p[0], g.stride, g.W, y, plane_index(g.frac, third + j), px);
            v = px[3];
        }
        sV[threadIdx.x] = v * 0x01010101u;
    }
    __syncthreads();
    const int n = np * 16 * (BORDER / 4);
    for (int e = threadIdx.x; e < n; e += NT) {
        const int i = e / (BORDER / 4), q = e - i * (BORDER / 4);
        const int yy = y0 + (i & 15);
        if (yy < g.ye)
            *reinterpret_cast<uint32_t *>(pl.p[plane_index(g.frac, third + (i >> 4))] + (int64_t)yy * g.stride +
                                          (left ? -XME_PAD : g.W + 4) + 4 * q) = sV[i];
    }
}

// Interpolated planes on the core columns x in [-4, W+4) of rows [ys, ye)
// (the whole core area is ys = -4, ye = H + 4), in tiles whose columns start
// at xs <= -4 (a 64-byte boundary of the output rows), and the border around
// them.  The staged rows below ye + 4 may not be final yet (an LCU row still
// being reconstructed): they only feed outputs at or below ye, which are not
// stored.  The full-pel tile (with its 3 + 4 pixel filter margins) is staged
// in LDS as signed bytes (pixel - 128); every 8-tap sum is two v_dot4_i32_i8
// with an exact 32-bit result, and the horizontal sums feeding the diagonal
// planes, which fit in int16, are kept in LDS as pairs of rows, the operands
// of the vertical v_dot2_i32_i16.
//
// The writes of 15 planes bound it, close before VALU issue (556 instructions
// per wave of a tile).  The border has workgroups of its
// own in the same launch, since a pass over the stored planes afterwards cost
// 10.6 us and a second launch: with the full-pel border, several pictures in
// turn, 2160p 64.9 -> 42.3 us (copy-rate floor 31), 424x240 10.2 -> 7.6, 720p in
// 12 LCU rows 127 -> 91.
// A strip's workgroup takes a third of the planes: with all of them its 18
// stores per thread are the longest chain of a small launch (424x240 9.1 us).
// Tiles of 128 x 8, 128 x 16, 64 x 8 and 64 x 32 were level or slower.
__global__ void __launch_bounds__(NT) interp_kernel(Planes16 pl, InterpGeom g)
{
    // workgroup b runs on XCD b % 8: each XCD takes a contiguous raster run of
    // tiles, so that the 128-byte lines shared by side-by-side tiles (their
    // staged source rows and the halves of their output rows) meet in one L2.
    // The border's workgroups come first, on all XCDs.
    __shared__ uint32_t sP[TY + 8][SPW];
    __shared__ uint32_t sH[3][TY / 2 + 4][TX];
    const int n_border = (g.n_band + g.n_strip + 7) & ~7;
    if ((int)blockIdx.x < n_border) {
        const int b = (int)(blockIdx.x & 7) * (n_border >> 3) + (int)(blockIdx.x >> 3);
        if (b < g.n_band)
            fill_band(pl, g, b);
        else if (b < g.n_band + g.n_strip)
            fill_strip(pl, g, b - g.n_band, &sP[0][0]);
        return;
    }
    const int bt = (int)blockIdx.x - n_border, per_xcd = ((int)gridDim.x - n_border) >> 3;
    const int tile = (bt & 7) * per_xcd + (bt >> 3);
    if (tile >= g.n_tiles)
        return;
    const int tx_i = tile % g.gx, ty_i = tile / g.gx;
    const int64_t stride = g.stride;
    const int W = g.W, H = g.H, frac = g.frac, ye = g.ye;
    const int x0 = g.xs + tx_i * TX, y0 = g.ys + ty_i * TY;
    const uint8_t *P = pl.p[0];
    const int tid = threadIdx.x;
    // stage: column x0 - 4 + 4q .. +3 of rows y0 - 3 .. y0 + TY + 3 (dword aligned
    // since x0 % 4 == 0 and the plane origin and stride are 4-byte aligned)
    for (int e = tid; e < (TY + 8) * SPW; e += NT) {
        const int r = e / SPW, q = e - r * SPW;
        const int y = xme_clip3(-XME_PAD, H + XME_PAD - 1, y0 - 3 + r);
        const int x = x0 - 4 + 4 * q;
        const uint8_t *row = P + (int64_t)y * stride;
        uint32_t v;
        if (x >= -XME_PAD && x + 3 <= W + XME_PAD - 1)
            v = *reinterpret_cast<const uint32_t *>(row + x);
        else
            v = (uint32_t)row[xme_clip3(-XME_PAD, W + XME_PAD - 1, x)] * 0x01010101u;
        sP[r][q] = v ^ 0x80808080u;
    }
    __syncthreads();
    int tl[4], th[4];
#pragma unroll
    for (int d = 1; d <= 3; d++)
        packed_taps(d, tl[d], th[d]);
    // horizontal sums: output column c uses pixels x0 + c - 3 .. x0 + c + 4,
    // i.e. staged bytes c + 1 .. c + 8; a thread does 4 columns of two rows and
    // keeps the sums of a column's two rows as int16 pairs
    if (tid < (TY / 2 + 4) * LX) {
        const int m = tid / LX, c4 = (tid & (LX - 1)) * 4;
        uint32_t lo[2][4], hi[2][4];
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const uint32_t *d = &sP[2 * m + r][c4 / 4];
            const uint32_t d0 = d[0], d1 = d[1], d2 = d[2];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                // bytes c4 + i + 1 .. c4 + i + 8
                lo[r][i] = i == 3 ? d1 : __builtin_amdgcn_alignbyte(d1, d0, (uint32_t)(i + 1));
                hi[r][i] = i == 3 ? d2 : __builtin_amdgcn_alignbyte(d2, d1, (uint32_t)(i + 1));
            }
        }
#pragma unroll
        for (int dx = 1; dx <= 3; dx++) {
            if (frac < 2 && dx != 2)
                continue;
            uint32_t v[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
                v[i] = __builtin_amdgcn_perm((uint32_t)fir8(tl[dx], th[dx], lo[1][i], hi[1][i]),
                                             (uint32_t)fir8(tl[dx], th[dx], lo[0][i], hi[0][i]), 0x05040100u);
            *reinterpret_cast<uint4 *>(&sH[dx - 1][m][c4]) = make_uint4(v[0], v[1], v[2], v[3]);
        }
    }
    __syncthreads();
    // a thread makes 4 columns of one row; the rows of a wave are all even or
    // all odd, so that the row pairs are taken as they lie or all shifted by one
    const bool odd = (tid >> 6) & 1;
    const int ty = (tid >> 7) * (128 / LX) + (tid & 63) / LX * 2 + (odd ? 1 : 0), c0 = (tid & (LX - 1)) * 4;
    const int y = y0 + ty, x = x0 + c0;
    if (y >= ye || x < -4 || x >= W + 4)
        return;
    const int64_t off = (int64_t)y * stride + x;
    // vertical d, h, n: pixels of rows y - 3 .. y + 4 at columns x .. x + 3,
    // i.e. staged dword (c0 + 4) / 4 of rows ty .. ty + 7, transposed to columns
    {
        uint32_t colA[4], colB[4];
        const int q = (c0 + 4) >> 2;
        transpose4(sP[ty][q], sP[ty + 1][q], sP[ty + 2][q], sP[ty + 3][q], colA);
        transpose4(sP[ty + 4][q], sP[ty + 5][q], sP[ty + 6][q], sP[ty + 7][q], colB);
#pragma unroll
        for (int dy = 1; dy <= 3; dy++) {
            if (frac < 2 && dy != 2)
                continue;
            uint32_t px[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
                px[i] = clip_pel(fir8(tl[dy], th[dy], colA[i], colB[i], 8192 + 32) >> 6);
            stream_out(pl.p[dy << 2] + off, pack_pels(px[0], px[1], px[2], px[3]));
        }
    }
    // horizontal a, b, c are the sums of row ty + 3; diagonal e..r (MC_SHIFT =
    // 12) the vertical 8-tap sums of rows ty .. ty + 7, four v_dot2_i32_i16 on
    // the int16 pairs of the horizontal sums, which lie in [-4845, 22440]; with
    // taps and rounding 16 times as large the pixel is the third byte
    for (int dx = 1; dx <= 3; dx++) {
        if (frac < 2 && dx != 2)
            continue;
        uint32_t hp[5][4];
#pragma unroll
        for (int m = 0; m < 5; m++) {
            const uint4 v = *reinterpret_cast<const uint4 *>(&sH[dx - 1][(ty >> 1) + m][c0]);
            hp[m][0] = v.x;
            hp[m][1] = v.y;
            hp[m][2] = v.z;
            hp[m][3] = v.w;
        }
        if (odd) {
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    hp[m][i] = __builtin_amdgcn_alignbyte(hp[m + 1][i], hp[m][i], 2);
        }
        uint32_t px[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            px[i] = clip_pel((int)(hp[1][i] + (32u << 16)) >> 22);
        stream_out(pl.p[dx] + off, pack_pels(px[0], px[1], px[2], px[3]));
#pragma unroll
        for (int dy = 1; dy <= 3; dy++) {
            if (frac < 2 && dy != 2)
                continue;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                int s = 2048 * 16;
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const short2v taps = { (short)(16 * c_taps[dy][2 * m]), (short)(16 * c_taps[dy][2 * m + 1]) };
                    s = __builtin_amdgcn_sdot2(__builtin_bit_cast(short2v, hp[m][i]), taps, s, false);
                }
                px[i] = (uint32_t)xme_clip3(0, 0xFFFFFF, s);
            }
            // the pixels are bytes 2
            stream_out(pl.p[(dy << 2) + dx] + off,
                       __builtin_amdgcn_perm(__builtin_amdgcn_perm(px[3], px[2], 0x0C0C0602u),
                                             __builtin_amdgcn_perm(px[1], px[0], 0x0C0C0602u), 0x05040100u));
        }
    }
}

// Fill [-pad, W+pad) x [-pad, H+pad) outside the core rectangle [cx0, cx1) x
// [cy0, cy1) with the nearest core value.  The grid covers only the border's
// dwords (core edges and pad are dword aligned), in four regions laid end to
// end: the bands above and below the core (full width; either may be left
// out, as for an LCU row inside the picture), then the strips left and right
// of the core rows.
struct BorderGeom {
    int64_t stride;
    int pad, W, H, cx0, cy0, cx1, cy1;
    int wdw;                   // dwords of a full row
    int ldw, rdw;              // dwords of the left and right strips
    int64_t n_top, n_bot, n_side;
};

__global__ void __launch_bounds__(256) border_kernel(uint8_t *base, BorderGeom g)
{
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int x, y;
    if (t < g.n_top) {
        y = -g.pad + (int)(t / g.wdw);
        x = -g.pad + 4 * (int)(t % g.wdw);
    } else if ((t -= g.n_top) < g.n_bot) {
        y = g.cy1 + (int)(t / g.wdw);
        x = -g.pad + 4 * (int)(t % g.wdw);
    } else if ((t -= g.n_bot) < g.n_side) {
        const int sdw = g.ldw + g.rdw, r = (int)(t / sdw), q = (int)(t % sdw);
        y = g.cy0 + r;
        x = q < g.ldw ? -g.pad + 4 * q : g.cx1 + 4 * (q - g.ldw);
    } else {
        return;
    }
    const int sy = xme_clip3(g.cy0, g.cy1 - 1, y);
    const uint8_t *src = base + (int64_t)sy * g.stride;
    uint32_t v;
    if (x >= g.cx0 && x < g.cx1) {
        v = *reinterpret_cast<const uint32_t *>(src + x);
    } else {
        const int sx = x < g.cx0 ? g.cx0 : g.cx1 - 1;
        v = (uint32_t)src[sx] * 0x01010101u;
    }
    *reinterpret_cast<uint32_t *>(base + (int64_t)y * g.stride + x) = v;
}

// The border of a plane; every edge and the pad are multiples of 4.  top / bottom: fill the band above cy0 / below cy1.
int launch_border(uint8_t *base, int64_t stride, int W, int H, int pad, int cx0, int cy0, int cx1, int cy1,
                  hipStream_t s, bool top = true, bool bottom = true)
{
    BorderGeom g;
    g.stride = stride;
    g.pad = pad;
    g.W = W;
    g.H = H;
    g.cx0 = cx0;
    g.cy0 = cy0;
    g.cx1 = cx1;
    g.cy1 = cy1;
    g.wdw = (W + 2 * pad) >> 2;
    g.ldw = (cx0 + pad) >> 2;
    g.rdw = (W + pad - cx1) >> 2;
    g.n_top = top ? (int64_t)(cy0 + pad) * g.wdw : 0;
    g.n_bot = bottom ? (int64_t)(H + pad - cy1) * g.wdw : 0;
    g.n_side = (int64_t)(cy1 - cy0) * (g.ldw + g.rdw);
    const int64_t n = g.n_top + g.n_bot + g.n_side;
    if (n <= 0)
        return XME_OK;
    hipLaunchKernelGGL(border_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, base, g);
    XME_HIP(hipGetLastError());
    return XME_OK;
}

// Planes 1..15 on the core columns of rows [ys, ye) and their border: the side
// strips of those rows, and the bands above / below when top / bottom.
int interp_rows(const Planes16 &pl, int64_t stride, int w, int h, int frac, int ys, int ye, bool top, bool bottom,
                hipStream_t s)
{
    // tile columns start where the output planes' rows reach a 64-byte
    // boundary, at or up to 60 columns left of the core's first column -4, so
    // that every 64-column row segment is one whole 64-byte line
    InterpGeom g;
    g.stride = stride;
    g.W = w;
    g.H = h;
    g.frac = frac;
    g.xs = -4 - (int)((reinterpret_cast<uintptr_t>(pl.p[2]) - 4) & 63);
    g.ys = ys;
    g.ye = ye;
    g.xb = g.xs - (g.xs + XME_PAD + TX - 1) / TX * TX;
    g.gx = (w + 4 - g.xs + TX - 1) / TX;
    g.gxb = (w + XME_PAD - g.xb + TX - 1) / TX;
    const int gy = (ye - ys + TY - 1) / TY;
    const int band = g.gxb * (BORDER / BAND_ROWS);
    g.n_top = top ? band : 0;
    g.n_band = g.n_top + (bottom ? band : 0);
    g.n_strip = 6 * gy;
    g.n_tiles = g.gx * gy;
    // multiples of 8: the same number per XCD
    const int grid = ((g.n_band + g.n_strip + 7) & ~7) + ((g.n_tiles + 7) & ~7);
    hipLaunchKernelGGL(interp_kernel, dim3(grid), dim3(NT), 0, s, pl, g);
    XME_HIP(hipGetLastError());
    return XME_OK;
}

// The planes a caller passes: 16 device origins, of which frac 1 needs 0, 2,
// 8 and 10 (frame.c:343-350); false (with the error set) when one is missing
// or unaligned.
bool pick_planes(pel_t *const d_planes[16], int frac, const char *who, Planes16 &pl)
{
    for (int k = 0; k < 16; k++) {
        const bool need = k == 0 || frac == 2 || k == 2 || k == 8 || k == 10;
        pl.p[k] = need ? d_planes[k] : nullptr;
        if (need && (!pl.p[k] || (reinterpret_cast<uintptr_t>(pl.p[k]) & 3))) {
            xme_set_error("%s: plane %d missing or not 4-byte aligned", who, k);
            return false;
        }
    }
    return true;
}

} // namespace

extern "C" int xme_expand_border(pel_t *d_plane, intptr_t stride, int w, int h, int pad, void *stream)
{
    if (!d_plane || w < 1 || h < 1 || (w & 3) || (pad & 3) || pad < 0 || stride < w + 2 * pad ||
        (reinterpret_cast<uintptr_t>(d_plane) & 3) || (stride & 3)) {
        xme_set_error("xme_expand_border: need 4-aligned plane, stride, width and pad");
        return XME_ERR_ARG;
    }
    if (pad == 0)
        return XME_OK;
    return launch_border(d_plane, (int64_t)stride, w, h, pad, 0, 0, w, h, (hipStream_t)stream);
}

extern "C" int xme_interpolate_frame(pel_t *const d_planes[16], intptr_t stride, int w, int h, int frac, void *stream)
{
    if (!d_planes || !d_planes[0] || w < 8 || h < 8 || (w & 7) || frac < 0 || frac > 2 || (stride & 3) ||
        stride < w + 2 * XME_PAD) {
        xme_set_error("xme_interpolate_frame: need width multiple of 8, stride >= width + %d, multiple of 4",
                      2 * XME_PAD);
        return XME_ERR_ARG;
    }
    if (frac == 0)
        return XME_OK;
    Planes16 pl;
    if (!pick_planes(d_planes, frac, "xme_interpolate_frame", pl))
        return XME_ERR_ARG;
    return interp_rows(pl, (int64_t)stride, w, h, frac, -4, h + 4, true, true, (hipStream_t)stream);
}

extern "C" int xme_expand_border_lcu_row(pel_t *d_plane, intptr_t stride, int w, int h, int pad, int row_log2,
                                         int lcu_y, void *stream)
{
    if (!d_plane || w < 1 || h < 1 || (w & 3) || (pad & 3) || pad < 0 || stride < w + 2 * pad ||
        (reinterpret_cast<uintptr_t>(d_plane) & 3) || (stride & 3) || row_log2 < 2 || row_log2 > 7) {
        xme_set_error("xme_expand_border_lcu_row: need 4-aligned plane, stride, width and pad, row_log2 2..7");
        return XME_ERR_ARG;
    }
    const int n_rows = (h + (1 << row_log2) - 1) >> row_log2;
    if (lcu_y < 0 || lcu_y >= n_rows) {
        xme_set_error("xme_expand_border_lcu_row: LCU row %d outside 0..%d", lcu_y, n_rows - 1);
        return XME_ERR_ARG;
    }
    // xavs2_frame_expand_border_lcurow (frame.c:537-575), one slice: rows
    // [y0, y1), UP_SHIFT 4 rows up except at the picture's top and bottom
    const bool first = lcu_y == 0, last = lcu_y == n_rows - 1;
    const int y0 = (lcu_y << row_log2) - (first ? 0 : 4);
    const int y1 = std::min(h, ((lcu_y + 1) << row_log2) - (last ? 0 : 4));
    if (pad == 0 || y1 <= y0)
        return XME_OK;
    return launch_border(d_plane, (int64_t)stride, w, h, pad, 0, y0, w, y1, (hipStream_t)stream, first, last);
}

extern "C" int xme_interpolate_lcu_row(pel_t *const d_planes[16], intptr_t stride, int w, int h, int frac,
                                       int lcu_level, int lcu_y, void *stream)
{
    if (!d_planes || !d_planes[0] || w < 8 || h < 8 || (w & 7) || frac < 0 || frac > 2 || (stride & 3) ||
        stride < w + 2 * XME_PAD || lcu_level < 3 || lcu_level > 6) {
        xme_set_error("xme_interpolate_lcu_row: need width multiple of 8, stride >= width + %d, multiple of 4, "
                      "lcu_level 3..6", 2 * XME_PAD);
        return XME_ERR_ARG;
    }
    const int n_rows = (h + (1 << lcu_level) - 1) >> lcu_level;
    if (lcu_y < 0 || lcu_y >= n_rows) {
        xme_set_error("xme_interpolate_lcu_row: LCU row %d outside 0..%d", lcu_y, n_rows - 1);
        return XME_ERR_ARG;
    }
    if (frac == 0)
        return XME_OK;
    Planes16 pl;
    if (!pick_planes(d_planes, frac, "xme_interpolate_lcu_row", pl))
        return XME_ERR_ARG;
    // interpolate_lcu_row (mc.c:748-785), one slice: rows [y0, y1) with
    // PAD_OFFSET 4 and MC_OFFSET 8 (mc.c:95-96)
    const bool first = lcu_y == 0, last = lcu_y == n_rows - 1;
    const int y0 = (lcu_y << lcu_level) - (first ? 4 : 8);
    const int y1 = last ? h + 4 : ((lcu_y + 1) << lcu_level) - 8;
    return interp_rows(pl, (int64_t)stride, w, h, frac, y0, y1, first, last, (hipStream_t)stream);
}

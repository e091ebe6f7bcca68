// Integer-pel full search by successive elimination, for batched plans of
// search ranges up to XME_EL_MAX_R.
//
// The exhaustive search of fs_kernels.hip sums W * H absolute differences for
// every candidate.  By the triangle inequality the SAD of a block is at least
// the sum, over its 4x4 sub-blocks, of |sum of the current pixels - sum of the
// reference pixels| (successive elimination, Li and Salari 1995, with the
// sub-block sums of the multilevel form).  A candidate whose bound plus MV cost
// exceeds a cost already reached cannot be the first strict minimum, so its SAD
// is not needed; every other candidate is costed exactly and the (cost, order)
// minimum is the reference's.  The bound takes W * H / 32 v_sad_u16 instead of
// W * H / 4 lane-operations.
//
//  * A task stages a reference window and the current pixels in LDS as the
//    exhaustive search does, and builds the window's map of 4x4 sums (u16 per
//    position) beside it.
//  * A wave takes an item (a PU and reference, a range of candidate rows) and
//    walks it in bands.  A lane owns 2 adjacent candidate columns x K rows: a
//    dword of the map holds both columns' sums, so two map dwords and one
//    v_perm give a column's packed pair, and K rows share the map rows.
//  * Candidates that pass are listed as tiles of 4 columns x 2 rows (they come
//    in clusters) in the wave's LDS, and full waves of tiles are costed with
//    v_qsad_pk_u16_u8: 2 candidate rows share each window row and current row.
//    When fewer than 33 tiles are left, 2 to 64 lanes share a tile's rows.
//  * Before a band's tiles are listed, the tile with the smallest bound is
//    costed by the whole wave; its cost is the next bound's threshold.
//  * Where the bounds let most of a band pass (noise), the rest of the item is
//    costed in strips, every candidate of it: 4 columns x 8 rows a lane, each
//    window row read once.
//
// Bound: VALU issue (83 % busy at 2160p): an 8x8 PU's band of 2048 candidates
// takes about 150 instructions of bounds, 75 of listing and 0.8 x 240 of exact
// costs (19 % of its tiles pass), where the exhaustive strip takes 900.  One
// workgroup of 16 waves holds the 110 KB window and sums of a 64x64 CTU at R =
// 64; two of 8 waves share a CU where they fit.  Search step, MI355X, smooth
// fields with noise, exhaustive -> this: 2160p, R = 64, 1 reference: 8x8 1450
// -> 825, 16x16 1150 -> 590, 32x32 1100 -> 625, 64x64 1045 -> 735, mixed PUs
// 1345 -> 695 us (4 references 4.90 -> 2.9 ms); with random MVPs (+-10 px)
// 1510 -> 870; 1080p 16x16, R = 32: 92 -> 51; 424x240 mixed, R = 16: 170 -> 52
// us.  On pure noise, where nothing is eliminated, exhaustive -> tiles alone ->
// this (1080p, R = 64): 8x8 417 -> 577 -> 425 us, 16x16 330 -> 410 -> 345, 32x32
// 325 -> 381 -> 348, 64x64 303 -> 406 -> 370 (a wave's one or two items there
// begin with bounds), mixed 560 -> 466 -> 374; R = 32, 8x8 117 -> 177 -> 136;
// 2160p mixed 1330 -> 1660 -> 1341, and with noise of 16 levels over structure
// 1330 -> 1574 -> 1405.
#include "xme_dpp.h"
#include "xme_internal.h"

#include <mutex>
#include <type_traits>

namespace {

// Per-wave LDS: sums of the PU's 4x4 sub-blocks (u16 pairs, rows padded to an
// even count), MV rate terms per candidate column and row, the rows' terms packed
// for the bound, and the tile list.
constexpr int kMaxR2 = 2 * XME_EL_MAX_R;
struct WaveArea {
    uint32_t cs[128];
    uint32_t xt[kMaxR2];
    uint32_t yt[kMaxR2];
    uint32_t yp[kMaxR2];
    uint16_t list[64 + 256];
};
static_assert(sizeof(WaveArea) == XME_EL_WAVE_BYTES, "plan and kernel agree on the LDS of a wave");

// Bound term of a candidate that cannot be chosen: above every cost (the SAD
// of 64 x 64 pixels and the rate of two 29-bit vector differences at the
// largest lambda).  A column's and a row's, with the largest bound between
// them, fit the 27 bits that a tile's key gives them.
constexpr uint32_t kNever = 1u << 21;
static_assert(64 * 64 * 255 + (((uint64_t)(1 << 24) * 2 * 29) >> 16) < kNever, "a threshold never reaches the term");
static_assert(2ull * kNever + 64 * 64 * 255 < 1u << 27, "and the term fits the key");

template <int CTRL>
__device__ __forceinline__ uint32_t row_min_step(uint32_t v)
{
    return min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, CTRL, 0xF, 0xF, false));
}

// Minimum over each row of 16 lanes, in all of them.
__device__ __forceinline__ uint32_t row_min(uint32_t v)
{
    v = row_min_step<0xB1>(v);      // quad_perm [1,0,3,2]
    v = row_min_step<0x4E>(v);      // quad_perm [2,3,0,1]
    v = row_min_step<0x124>(v);     // row_ror:4
    return row_min_step<0x128>(v);  // row_ror:8
}

__device__ __forceinline__ uint32_t wave_min(uint32_t v)
{
    v = row_min(v);
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
    const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32);
    const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return min(min(a, b), min(c, d));
}

// Sum over each row of 16 lanes, in all of them.
__device__ __forceinline__ uint32_t row_sum(uint32_t v)
{
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xF, 0xF, true);
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, true);
}

// LDS written by the wave's lanes is read by others of the same wave (in
// order in hardware; this orders it for the compiler).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Stage the window and the current pixels: a wave per row, four rows in
// flight.  Columns and rows outside the padded picture are clamped to it; only
// illegal candidates (never selected) can read them.
__device__ __forceinline__ void stage(const FsTask &t, const FrameDesc *__restrict__ desc, const DevParams &p,
                                      uint32_t *__restrict__ w32, int pd, uint32_t *__restrict__ c32)
{
    const uint8_t *ref = desc->planes[t.ref][0];
    const int64_t stride = desc->stride[t.ref];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int ylo = -XME_PAD, yhi = p.frame_h + XME_PAD - 1;
    const int ndw = t.ww >> 2;
    for (int q = lane; q < ndw; q += 64) {
        const int x = xme_clip3(-XME_PAD, p.frame_w + XME_PAD - 4, t.wx0 + 4 * q);
        for (int r = wave; r < t.wh; r += 4 * nw) {
            uint32_t v[4];
#pragma unroll
            for (int k = 0; k < 4; k++)
                v[k] = *reinterpret_cast<const uint32_t *>(
                    ref + (int64_t)xme_clip3(ylo, yhi, t.wy0 + min(r + k * nw, t.wh - 1)) * stride + x);
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (r + k * nw < t.wh)
                    w32[(r + k * nw) * pd + q] = v[k];
        }
    }
    const int cdw = t.cw >> 2, total = cdw * t.ch;
    for (int e = threadIdx.x; e < total; e += blockDim.x) {
        const int r = e / cdw, q = e - r * cdw;
        c32[e] = *reinterpret_cast<const uint32_t *>(desc->cur + (int64_t)(t.cy0 + r) * desc->i_cur + t.cx0 + 4 * q);
    }
}

// The window's 4x4 sums: a thread takes one dword column over a segment of
// rows, holds the horizontal sums of its four positions as two u16 pairs (4 *
// 4 * 255 < 2^16: the halves never carry) and slides them down.
__device__ __forceinline__ void build_sums(const FsTask &t, const uint32_t *__restrict__ w32, int pd,
                                           uint32_t *__restrict__ s32, int sp)
{
    const int ndw = t.ww >> 2, sh = t.wh - 3;
    const int nseg = max(1, (int)blockDim.x / ndw);
    const int rps = (sh + nseg - 1) / nseg;
    for (int e = threadIdx.x; e < ndw * nseg; e += blockDim.x) {
        const int seg = e / ndw, q = e - seg * ndw;
        const int y0 = seg * rps, y1 = min(sh, y0 + rps);
        if (y0 >= y1)
            continue;
        uint32_t h[4][2];
        auto row = [&](int y, uint32_t (&d)[2]) {
            const uint32_t a = w32[y * pd + q], b = w32[y * pd + q + 1];
            d[0] = __builtin_amdgcn_sad_hi_u8(__builtin_amdgcn_alignbyte(b, a, 1), 0, __builtin_amdgcn_sad_u8(a, 0, 0));
            d[1] = __builtin_amdgcn_sad_hi_u8(__builtin_amdgcn_alignbyte(b, a, 3), 0,
                                              __builtin_amdgcn_sad_u8(__builtin_amdgcn_alignbyte(b, a, 2), 0, 0));
        };
#pragma unroll
        for (int k = 0; k < 3; k++)
            row(y0 + k, h[k]);
        for (int y = y0; y < y1; y += 4) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (y + k < y1) {
                    row(y + k + 3, h[(k + 3) & 3]);
                    s32[(y + k) * sp + 2 * q] = (h[0][0] + h[1][0]) + (h[2][0] + h[3][0]);
                    s32[(y + k) * sp + 2 * q + 1] = (h[0][1] + h[1][1]) + (h[2][1] + h[3][1]);
                }
            }
        }
    }
}

// One chunk of NY x NX sub-blocks of the bound for the lane's 2 columns x K
// rows.  s: the lane's map dword at the chunk's first row (the one that holds
// the lane's first column, in its low half, or in its high half when ODD);
// c32: the chunk's current sums.  Map rows are loaded PF rows ahead.
template <int K, int NX, int NY, bool ODD>
__device__ __forceinline__ void bound_chunk(const uint32_t *__restrict__ s, int sp, const uint32_t *__restrict__ c32,
                                            uint32_t (&acc)[K][2])
{
    constexpr int NP = (NX + 1) / 2, ROWS = K + 4 * (NY - 1), PF = NX <= 2 ? 4 : 2;
    uint32_t e[PF][NX], o[PF][NX];
    // one running row offset: without the barrier every row's address becomes
    // an induction variable of the caller's loop, in a register of its own
    int at = 0;
    auto load = [&](int r) {
        asm volatile("" : "+v"(at));
#pragma unroll
        for (int j = 0; j < NX; j++) {
            e[r % PF][j] = s[at + 2 * j];
            o[r % PF][j] = ODD ? s[at + 2 * j + 1] : e[r % PF][j];
        }
        at += sp;
    };
#pragma unroll
    for (int r = 0; r < PF; r++)
        load(r);
    uint32_t c[NY][NP];
#pragma unroll
    for (int b = 0; b < NY; b++)
#pragma unroll
        for (int j = 0; j < NP; j++)
            c[b][j] = c32[b * NP + j];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        uint32_t lo[NP], hi[NP];
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const uint32_t e0 = e[r % PF][2 * j], o0 = o[r % PF][2 * j];
            if (2 * j + 1 < NX) {
                const uint32_t e1 = e[r % PF][2 * j + 1 < NX ? 2 * j + 1 : 0], o1 = o[r % PF][2 * j + 1 < NX ? 2 * j + 1 : 0];
                lo[j] = __builtin_amdgcn_perm(e1, e0, ODD ? 0x07060302 : 0x05040100);
                hi[j] = __builtin_amdgcn_perm(o1, o0, ODD ? 0x05040100 : 0x07060302);
            } else {
                lo[j] = ODD ? e0 >> 16 : e0 & 0xFFFFu;
                hi[j] = ODD ? o0 & 0xFFFFu : o0 >> 16;
            }
        }
        if (r + PF < ROWS)
            load(r + PF);
#pragma unroll
        for (int j = 0; j < NP; j++) {
#pragma unroll
            for (int b = 0; b < NY; b++) {
                const int k = r - 4 * b;
                if (k >= 0 && k < K) {
                    acc[k][0] = __builtin_amdgcn_sad_u16(lo[j], c[b][j], acc[k][0]);
                    acc[k][1] = __builtin_amdgcn_sad_u16(hi[j], c[b][j], acc[k][1]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// SADs of a tile's 4 columns x 2 rows over `rows` PU rows (4 ND * rows * 255 <
// 2^16) of a strip of 4 ND pixels: a[0] candidate row 0, a[1] row 1, u16 per
// column.  A window row (ND dwords and the one after them, realigned by
// `shift` bytes) meets two current rows; rows are read one ahead, the last
// read passing the tile by a row (inside the task's LDS).  ROWS: the row
// count when it is known (unrolled), else 0.
template <int ND, int ROWS, bool ALIGNED>
__device__ __forceinline__ void tile_strip(const uint32_t *__restrict__ w, int pd, uint32_t shift,
                                           const uint32_t *__restrict__ c, int cpd, int rows, uint64_t (&a)[2])
{
    constexpr int NW = ALIGNED ? ND + 1 : ND + 2;
    uint32_t raw[NW], cw[ND];
    uint64_t cur[ND];
    int wa = 0, ca = 0;
    auto load_w = [&]() {
        if (ROWS > 0)          // one running offset, not an address per row
            asm volatile("" : "+v"(wa));
#pragma unroll
        for (int i = 0; i < NW; i++)
            raw[i] = w[wa + i];
        wa += pd;
    };
    auto load_c = [&]() {
        if (ROWS > 0)
            asm volatile("" : "+v"(ca));
#pragma unroll
        for (int i = 0; i < ND; i++)
            cw[i] = c[ca + i];
        ca += cpd;
    };
    auto operands = [&](uint64_t (&d)[ND]) {
        uint32_t al[ND + 1];
#pragma unroll
        for (int i = 0; i <= ND; i++)
            al[i] = ALIGNED ? raw[i] : __builtin_amdgcn_alignbyte(raw[ALIGNED ? i : i + 1], raw[i], shift);
#pragma unroll
        for (int i = 0; i < ND; i++)
            d[i] = ((uint64_t)al[i + 1] << 32) | al[i];
    };
    load_w();
    load_c();
    operands(cur);
    load_w();
    auto step = [&]() {
        uint64_t nxt[ND];
        uint32_t cc[ND];
        operands(nxt);
#pragma unroll
        for (int i = 0; i < ND; i++)
            cc[i] = cw[i];
        load_w();
        load_c();
#pragma unroll
        for (int i = 0; i < ND; i++) {
            a[0] = __builtin_amdgcn_qsad_pk_u16_u8(cur[i], cc[i], a[0]);
            a[1] = __builtin_amdgcn_qsad_pk_u16_u8(nxt[i], cc[i], a[1]);
        }
#pragma unroll
        for (int i = 0; i < ND; i++)
            cur[i] = nxt[i];
    };
    if constexpr (ROWS > 0) {
#pragma unroll
        for (int y = 0; y < ROWS; y++) {
            step();
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll 2
        for (int y = 0; y < rows; y++)
            step();
    }
}

struct TaskView {
    const uint32_t *w32;       // window
    int pd;                    // its dwords per row
    const uint32_t *c32;       // current pixels
    int cpd;
    const uint32_t *s32;       // 4x4 sums
    int sp;
    int wx0, wy0, cx0, cy0;
};

// Where more than kDenseNum / kDenseDen of a band's tiles pass the bounds, the
// bands after it are searched without them.  With STRIPS (el_strips) every
// candidate of the rest of the item is costed by dense_rows, and so are those
// of the wave's next 3 items, then 15; else the tiles of the next 3 bands are
// all listed.  4 / 5 is quicker on noise of 16 levels over structure (2160p
// mixed PUs, 1 reference 1377 us against 1388) but costs pictures with less (4
// references, noise of 3: 3180 us without strips, 3199 at 9 / 10, 3245 at 4 / 5).
constexpr int kDenseNum = 9, kDenseDen = 10, kDenseRun = 15;

// What a wave keeps between items: what its rate terms were made for, the items
// (or bands) it still searches without bounds after one that eliminated nearly
// nothing, and how many such the last one led to.
struct WaveState {
    bool ok;
    int cx, cy, px, py;
    int dense, run;
};

// An instance's search box: the legal candidate columns, and whether every
// candidate is legal.
struct Box {
    int lox, hix;
    bool all_legal;
};

// One item: the candidate rows [row0, row0 + nrows) of one instance.  ONE: its
// PU is NX x NY sub-blocks; else a multiple of that.
template <int K, int NX, int NY, bool ONE>
struct Item {
    const DevParams &p;
    const TaskView &v;
    const DevPu &pu;
    const DevInst &in;
    WaveArea *__restrict__ wa;
    int lane, bx, by;
    bool all_legal;
    const uint32_t *cpu32;     // the PU's current pixels

    __device__ __forceinline__ int nx() const { return ONE ? NX : pu.w >> 2; }
    __device__ __forceinline__ int h() const { return ONE ? 4 * NY : pu.h; }

    // (cost << 3 | k) of the best of a tile's candidates k (row k / 4, column
    // k % 4) with SADs sad[k]; 0xFFFFFFFF when none is legal
    __device__ __forceinline__ uint32_t tile_key(int trow, int tcol, uint32_t (&sad)[8]) const
    {
        uint32_t key = 0xFFFFFFFFu;
        const uint32_t ty[2] = { wa->yt[trow], wa->yt[trow + 1] };
#pragma unroll
        for (int k = 0; k < 8; k++)
            sad[k] = ((sad[k] + ((wa->xt[tcol + (k & 3)] + ty[k >> 2]) >> 16)) << 3) | (uint32_t)k;
        if (all_legal && (p.R & 1) == 0) {
#pragma unroll
            for (int k = 0; k < 8; k++)
                key = min(key, sad[k]);
        } else {
            const MvWindow mw = xme_mv_window(p, pu.x, pu.y, pu.w, pu.h);
            const int R = p.R;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int j = trow + (k >> 2), i = tcol + (k & 3);
                if (i < 2 * R && j < 2 * R && xme_mv_legal(mw, in.omx + i - R, in.omy + j - R))
                    key = min(key, sad[k]);
            }
        }
        return key;
    }

    static __device__ __forceinline__ void unpack_add(const uint64_t (&a)[2], uint32_t (&sad)[8])
    {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            sad[4 * r + 0] += (uint32_t)a[r] & 0xFFFFu;
            sad[4 * r + 1] += (uint32_t)a[r] >> 16;
            sad[4 * r + 2] += (uint32_t)(a[r] >> 32) & 0xFFFFu;
            sad[4 * r + 3] += (uint32_t)(a[r] >> 48);
        }
    }

    // The smallest cost among the tiles of the smallest bounds, one per row of
    // 16 lanes (PUs of at most 16 dwords) or one for the wave: the lanes share
    // the tile's pixels.  A row of lanes that owns only columns from 2 R on
    // has no tile to offer.
    __device__ __forceinline__ uint32_t probe(uint32_t kmin, int row, int quad) const
    {
        constexpr bool QUARTER = ONE && NX * 4 * NY <= 16;
        const uint32_t best = QUARTER ? row_min(kmin) : wave_min(kmin);
        const int trow0 = row + (((int)(kmin & 31u) - row) & 31);
        uint32_t tile = kmin == best ? (uint32_t)((trow0 << 6) | quad) : 0xFFFFFFFFu;
        tile = QUARTER ? row_min(tile) : wave_min(tile);
        const int trow = (int)(tile >> 6), tcol = (int)(tile & 63u) << 2;
        const uint32_t shift = (uint32_t)bx & 3u;
        const uint32_t *w = v.w32 + (by + trow) * v.pd + ((bx + tcol) >> 2);
        const int n_dw = nx() * h();
        uint64_t a[2] = { 0, 0 };
        for (int d = QUARTER ? lane & 15 : lane; d < n_dw; d += 64) {      // at most 16 dwords a lane: u16 holds them
            const int y = d / nx(), x = d - y * nx();
            const uint32_t cw = cpu32[y * v.cpd + x];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const uint32_t *q = w + (y + r) * v.pd + x;
                const uint32_t q0 = q[0], q1 = q[1], q2 = q[2];
                const uint64_t d = ((uint64_t)__builtin_amdgcn_alignbyte(q2, q1, shift) << 32) |
                                   __builtin_amdgcn_alignbyte(q1, q0, shift);
                a[r] = __builtin_amdgcn_qsad_pk_u16_u8(d, cw, a[r]);
            }
        }
        uint32_t sad[8] = { 0, 0, 0, 0, 0, 0, 0, 0 };
        if constexpr (ONE) {       // at most 256 pixels: the u16 pairs hold the sums
            uint32_t q[4] = { (uint32_t)a[0], (uint32_t)(a[0] >> 32), (uint32_t)a[1], (uint32_t)(a[1] >> 32) };
#pragma unroll
            for (int k = 0; k < 4; k++)
                q[k] = QUARTER ? row_sum(q[k]) : (uint32_t)group_sum((int)q[k], 64);
            a[0] = ((uint64_t)q[1] << 32) | q[0];
            a[1] = ((uint64_t)q[3] << 32) | q[2];
            unpack_add(a, sad);
        } else {
            unpack_add(a, sad);
#pragma unroll
            for (int k = 0; k < 8; k++)
                sad[k] = (uint32_t)group_sum((int)sad[k], 64);
        }
        const uint32_t key = (best >> 5) < kNever ? tile_key(trow, tcol, sad) : 0xFFFFFFFFu;
        return QUARTER ? wave_min(key >> 3) : (uint32_t)__builtin_amdgcn_readlane((int)(key >> 3), 63);
    }

    // Costs the listed tiles [first, first + cnt), 1 << lg lanes a tile, into the lane's best.
    template <bool FULL>
    __device__ __forceinline__ void cost_tiles(int first, int cnt, uint32_t &bc, uint32_t &bo) const
    {
        int lg = 0;
        if constexpr (!FULL) {
            const int gl = cnt > 32 ? 0 : cnt > 16 ? 1 : cnt > 8 ? 2 : cnt > 4 ? 3 : cnt > 2 ? 4 : cnt > 1 ? 5 : 6;
            lg = min(gl, (int)__builtin_ctz((unsigned)h()));
        }
        const int t = lane >> lg, g = lane & ((1 << lg) - 1);
        const int e = wa->list[first + (FULL ? lane : min(t, cnt - 1))];
        const int trow = e >> 6, tcol = (e & 63) << 2;
        const int rows = h() >> lg;
        const uint32_t shift = (uint32_t)bx & 3u;
        const uint32_t *w = v.w32 + (by + trow + (FULL ? 0 : g * rows)) * v.pd + ((bx + tcol) >> 2);
        const uint32_t *c = cpu32 + (FULL ? 0 : g * rows * v.cpd);
        uint32_t sad[8] = { 0, 0, 0, 0, 0, 0, 0, 0 };
        if constexpr (ONE) {
            uint64_t a[2] = { 0, 0 };
            if (shift == 0)
                tile_strip<NX, FULL ? 4 * NY : 0, true>(w, v.pd, shift, c, v.cpd, rows, a);
            else
                tile_strip<NX, FULL ? 4 * NY : 0, false>(w, v.pd, shift, c, v.cpd, rows, a);
            if (lg) {              // at most 256 pixels: the u16 pairs hold the sums
                uint32_t q[4] = { (uint32_t)a[0], (uint32_t)(a[0] >> 32), (uint32_t)a[1], (uint32_t)(a[1] >> 32) };
#pragma unroll
                for (int k = 0; k < 4; k++)
                    q[k] = (uint32_t)group_sum((int)q[k], 1 << lg);
                a[0] = ((uint64_t)q[1] << 32) | q[0];
                a[1] = ((uint64_t)q[3] << 32) | q[2];
            }
            unpack_add(a, sad);
        } else {
            for (int x = 0; x < nx(); x += NX) {
                for (int y = 0; y < rows; y += 16) {      // 16 * 16 * 255 < 2^16
                    uint64_t a[2] = { 0, 0 };
                    const uint32_t *wy = w + y * v.pd + x, *cy = c + y * v.cpd + x;
                    if (shift == 0)
                        tile_strip<NX, 0, true>(wy, v.pd, shift, cy, v.cpd, min(16, rows - y), a);
                    else
                        tile_strip<NX, 0, false>(wy, v.pd, shift, cy, v.cpd, min(16, rows - y), a);
                    unpack_add(a, sad);
                }
            }
            if (lg) {
#pragma unroll
                for (int k = 0; k < 8; k++)
                    sad[k] = (uint32_t)group_sum((int)sad[k], 1 << lg);
            }
        }
        const uint32_t key = tile_key(trow, tcol, sad);
        const uint32_t cost = key >> 3;
        const uint32_t order = XME_ORDER_RASTER + (uint32_t)((trow + (int)((key >> 2) & 1)) * 2 * p.R + tcol + (int)(key & 3));
        bool take = key != 0xFFFFFFFFu && (cost < bc || (cost == bc && order < bo));
        if constexpr (!FULL)
            take = take && t < cnt && g == (1 << lg) - 1;
        if (take) {
            bc = cost;
            bo = order;
        }
    }
};

// The box of an instance, and its rate terms in the wave's LDS.
__device__ __forceinline__ Box rate_terms(const DevParams &p, const DevPu &pu, const DevInst &in,
                                          WaveArea *__restrict__ wa, WaveState &rs)
{
    const int lane = threadIdx.x & 63, R = p.R, R2 = 2 * p.R;
    // The packed range check equals the box test while |MV| < 8192; the bound
    // drops illegal candidates only then (the exact costs check each one).
    const MvWindow mw = xme_mv_window(p, pu.x, pu.y, pu.w, pu.h);
    const bool boxed = mw.min_fpel[0] > -8192 && mw.max_fpel[0] < 8192 && mw.min_fpel[1] > -8192 &&
                       mw.max_fpel[1] < 8192 && in.omx - R > -8192 && in.omx + R < 8192 && in.omy - R > -8192 &&
                       in.omy + R < 8192;
    Box box;
    box.all_legal = boxed && in.omx - R >= mw.min_fpel[0] && in.omx + R - 1 <= mw.max_fpel[0] &&
                    in.omy - R >= mw.min_fpel[1] && in.omy + R - 1 <= mw.max_fpel[1];
    box.lox = boxed ? mw.min_fpel[0] - in.omx + R : 0;
    box.hix = boxed ? min(R2 - 1, mw.max_fpel[0] - in.omx + R) : R2 - 1;
    if (rs.ok && box.all_legal && rs.cx == in.omx && rs.cy == in.omy && rs.px == pu.mvp_x && rs.py == pu.mvp_y)
        return box;
    // ME_COST_IPEL's rate (me.c:187-192) is (lambda * (bits x + bits y)) >> 16;
    // lambda < 2^24 and the bit counts are small, so the sum of the two
    // products is the same (below 2^31)
    const int loy = boxed ? mw.min_fpel[1] - in.omy + R : 0;
    const int hiy = boxed ? min(R2 - 1, mw.max_fpel[1] - in.omy + R) : R2 - 1;
    for (int i = lane; i < min(R2 + 16, kMaxR2); i += 64) {
        const uint32_t ty = __umul24((uint32_t)p.lambda, (uint32_t)xme_mvbits(4 * (in.omy + i - R) - pu.mvp_y));
        const uint32_t tn = __umul24((uint32_t)p.lambda, (uint32_t)xme_mvbits(4 * (in.omy + i + 1 - R) - pu.mvp_y));
        const bool never = i > hiy || i + 1 < loy;      // both rows of the pair
        wa->xt[i] = __umul24((uint32_t)p.lambda, (uint32_t)xme_mvbits(4 * (in.omx + i - R) - pu.mvp_x));
        wa->yt[i] = ty;
        wa->yp[i] = ((never ? kNever : min(ty, tn) >> 16) << 5) | (uint32_t)(i & 31);
    }
    rs.ok = box.all_legal;
    rs.cx = in.omx;
    rs.cy = in.omy;
    rs.px = pu.mvp_x;
    rs.py = pu.mvp_y;
    wave_sync();
    return box;
}

// The bands of an item by elimination, from the middle one outwards, up to the
// first whose bounds eliminate nearly nothing: true when there is one.  Left to
// search are then the candidate rows below end_lo and those from begin_hi on.
template <int K, int NX, int NY, bool ONE, bool STRIPS>
__device__ __forceinline__ bool el_item(const DevParams &p, const TaskView &v, const DevPu &pu, const DevInst &in,
                                       const Box &box, int row0, int nrows, int lc_log2, uint32_t T,
                                       WaveArea *__restrict__ wa, WaveState &rs, uint32_t &bc, uint32_t &bo,
                                       int &end_lo, int &begin_hi)
{
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));      // keeps what follows from the lane inside this item's code
    Item<K, NX, NY, ONE> I{ p, v, pu, in, wa, lane, 0, 0, box.all_legal, nullptr };
    const int R = p.R, R2 = 2 * p.R;
    const int bx = I.bx = pu.x + in.omx - R - v.wx0, by = I.by = pu.y + in.omy - R - v.wy0;
    constexpr int CP = (NX + 1) / 2;           // dwords of a sub-block row of a chunk
    const int chunks_x = ONE ? 1 : (pu.w >> 2) / NX, chunks_y = ONE ? 1 : (pu.h >> 2) / NY;
    const uint32_t *cpu32 = I.cpu32 = v.c32 + (pu.y - v.cy0) * v.cpd + ((pu.x - v.cx0) >> 2);

    // current sums, chunk by chunk
    for (int s = lane; s < chunks_x * chunks_y * NY * CP; s += 64) {
        const int j = s % CP, b = s / CP % NY, ch = s / (CP * NY);
        const int cy = ONE ? 0 : ch / chunks_x, cx = ONE ? 0 : ch - cy * chunks_x;
        const uint32_t *c = cpu32 + 4 * (cy * NY + b) * v.cpd + cx * NX + 2 * j;
        uint32_t s0 = 0, s1 = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            s0 = __builtin_amdgcn_sad_u8(c[k * v.cpd], 0, s0);
            if (2 * j + 1 < NX)
                s1 = __builtin_amdgcn_sad_u8(c[k * v.cpd + 1], 0, s1);
        }
        wa->cs[s] = s0 | (s1 << 16);
    }
    wave_sync();

    const int lc = lane & ((1 << lc_log2) - 1), rg = lane >> lc_log2;
    const int band_rows = (64 >> lc_log2) * K;
    uint32_t lx[2];
#pragma unroll
    for (int d = 0; d < 2; d++) {
        const int i = 2 * lc + d;
        lx[d] = i < box.lox || i > box.hix ? kNever : wa->xt[min(i, R2 - 1)] >> 16;
    }
    const uint32_t *s_lane = v.s32 + by * v.sp + ((bx + min(2 * lc, R2 - 2)) >> 1);

    int n = 0;
    const int n_bands = (nrows + band_rows - 1) / band_rows;
    bool dense = false;
    end_lo = row0;
    begin_hi = row0 + nrows;
    for (int band = 0; band < n_bands; band++) {
        // bands from the centre outwards: short vectors are likelier
        const int bi = (n_bands >> 1) + ((band & 1) ? -((band + 1) >> 1) : band >> 1);
        const int row = max(row0, min(row0 + bi * band_rows + rg * K, row0 + nrows - K));
        uint32_t tk[K / 2];        // per row pair: the smallest bound of its 4 candidates
        uint32_t kmin = 0xFFFFFFFFu;
        const bool bounds = STRIPS || rs.dense == 0;
        if (!bounds) {             // every legal tile is listed
            rs.dense--;
#pragma unroll
            for (int m = 0; m < K / 2; m++)
                tk[m] = (min(lx[0], lx[1]) << 5) + wa->yp[row + 2 * m];
        } else {
            uint32_t acc[K][2];
#pragma unroll
            for (int k = 0; k < K; k++) {
                acc[k][0] = lx[0];
                acc[k][1] = lx[1];
            }
            const uint32_t *s = s_lane + row * v.sp;
            if constexpr (ONE) {
                if (bx & 1)
                    bound_chunk<K, NX, NY, true>(s, v.sp, wa->cs, acc);
                else
                    bound_chunk<K, NX, NY, false>(s, v.sp, wa->cs, acc);
            } else {
                const uint32_t *c = wa->cs;
                for (int cy = 0; cy < chunks_y; cy++) {
                    const uint32_t *sx = s;
                    for (int cx = 0; cx < chunks_x; cx++) {
                        if (bx & 1)
                            bound_chunk<K, NX, NY, true>(sx, v.sp, c, acc);
                        else
                            bound_chunk<K, NX, NY, false>(sx, v.sp, c, acc);
                        sx += 2 * NX;
                        c += NY * CP;
                    }
                    s += 4 * NY * v.sp;
                }
            }
#pragma unroll
            for (int m = 0; m < K / 2; m++) {
                const uint32_t b = min(min(min(acc[2 * m][0], acc[2 * m][1]), acc[2 * m + 1][0]), acc[2 * m + 1][1]);
                tk[m] = (b << 5) + wa->yp[row + 2 * m];
                kmin = min(kmin, tk[m]);
            }
        }
        // small PUs: a probe costs about as much as what it saves after the first band
        if ((!ONE || NX * NY >= 16 || band == 0) && __any((kmin >> 5) < T))
            T = min(T, I.probe(kmin, row, lc >> 1));
        const uint32_t lim = (T << 5) | 31u;
        const int n0 = n;
        const int tile0 = (row << 6) | (lc >> 1);
#pragma unroll
        for (int m = 0; m < K / 2; m++) {
            const uint64_t b = __ballot(tk[m] <= lim);
            const uint64_t pairs = (b | (b >> 1)) & 0x5555555555555555ull;
            if (pairs) {
                const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(pairs >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)pairs, n));
                if (__builtin_amdgcn_inverse_ballot_w64(pairs))
                    wa->list[at] = (uint16_t)(tile0 + 128 * m);
                n += __popcll(pairs);
            }
        }
        // noise: most tiles pass, and costing them one by one takes longer than
        // costing every candidate of this band and of the others
        if (bounds && kDenseDen * (n - n0) > kDenseNum * ((16 * K * R) >> lc_log2)) {
            if constexpr (!STRIPS) {
                rs.dense = 3;
            } else if (nrows >= K) {
                n = n0;
                end_lo = band ? row0 + ((n_bands >> 1) - (band >> 1)) * band_rows : begin_hi;
                begin_hi = band ? min(begin_hi, row0 + ((n_bands >> 1) + ((band + 1) >> 1)) * band_rows) : begin_hi;
                dense = true;
                break;
            }
        }
        wave_sync();
        while (n >= 64) {
            n -= 64;
            I.template cost_tiles<true>(n, 64, bc, bo);
            T = min(T, wave_min(bc));
        }
    }
    if (n > 0)
        I.template cost_tiles<false>(0, n, bc, bo);
    return dense;
}

typedef const __attribute__((address_space(3))) uint32_t *lds_dwords;

// SADs of 4 columns x KD candidate rows over a strip of ND dwords x `rows` PU
// rows (a multiple of 4; 4 ND * rows * 255 < 2^16).  The last KD window rows
// are kept realigned, so each is read once; the next window and PU rows are in
// flight, the last reads passing the strip by a row (inside the task's LDS).
template <int KD, int ND>
__device__ __forceinline__ void dense_strip(lds_dwords w, int pd, uint32_t shift, lds_dwords c, int cpd, int rows,
                                            uint64_t (&a)[KD])
{
    uint64_t ring[KD][ND];
    uint32_t raw[ND + 2], cur[2][ND];
    auto load_c = [&](int j) {
        asm volatile("" : "+v"(c));
#pragma unroll
        for (int i = 0; i < ND; i++)
            cur[j & 1][i] = c[i];
        c += cpd;
    };
    auto load = [&]() {
        asm volatile("" : "+v"(w));        // one running address, not one per row
#pragma unroll
        for (int i = 0; i < ND + 2; i++)
            raw[i] = w[i];
        w += pd;
    };
    auto realign = [&](uint64_t (&d)[ND]) {
        uint32_t al[ND + 1];
#pragma unroll
        for (int i = 0; i <= ND; i++)
            al[i] = __builtin_amdgcn_alignbyte(raw[i + 1], raw[i], shift);
#pragma unroll
        for (int i = 0; i < ND; i++)
            d[i] = ((uint64_t)al[i + 1] << 32) | al[i];
    };
    load();
    load_c(0);
#pragma unroll
    for (int r = 0; r < KD - 1; r++) {
        realign(ring[r]);
        load();
    }
    for (int y = 0; y < rows; y += 8) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (j == 4 && y + 4 >= rows)
                break;
            realign(ring[(j + KD - 1) % KD]);
            load();
            load_c(j + 1);
#pragma unroll
            for (int i = 0; i < ND; i++)
#pragma unroll
                for (int k = 0; k < KD; k++)
                    a[k] = __builtin_amdgcn_qsad_pk_u16_u8(ring[(j + k) % KD][i], cur[j & 1][i], a[k]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Every candidate of rows [lo, hi) of an item, whose rows begin at row0 and are
// at least KD, R >= 2: a lane owns 4 columns x KD rows.  Lanes past the last
// column or row repeat others.  SMALL: PUs of at most 256 pixels, whose SADs
// the u16 sums hold; the others' sides are multiples of 8.
template <int KD, bool SMALL>
__device__ __forceinline__ void dense_rows(const DevParams &p, const TaskView &v, const DevPu &pu, const DevInst &in,
                                           bool all_legal, int row0, int lo, int hi, int lc_log2,
                                           const WaveArea *__restrict__ wa, uint32_t &bc, uint32_t &bo)
{
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int R = p.R, qc_log2 = lc_log2 - 1;
    const int col = min(4 * (lane & ((1 << qc_log2) - 1)), 2 * R - 4), g = lane >> qc_log2;
    const int x0 = pu.x + in.omx - R - v.wx0 + col, by = pu.y + in.omy - R - v.wy0;
    const uint32_t shift = (uint32_t)x0 & 3u;
    const lds_dwords cpu32 = (lds_dwords)(v.c32 + (pu.y - v.cy0) * v.cpd + ((pu.x - v.cx0) >> 2));
    for (int base = lo; base < hi; base += (64 >> qc_log2) * KD) {
        const int row = max(row0, min(base + g * KD, hi - KD));
        const lds_dwords w = (lds_dwords)(v.w32 + (by + row) * v.pd + (x0 >> 2));
        uint32_t sad[KD][4];
        uint64_t a[KD];
        auto unpack = [&]() {
#pragma unroll
            for (int k = 0; k < KD; k++) {
                sad[k][0] += (uint32_t)a[k] & 0xFFFFu;
                sad[k][1] += (uint32_t)a[k] >> 16;
                sad[k][2] += (uint32_t)(a[k] >> 32) & 0xFFFFu;
                sad[k][3] += (uint32_t)(a[k] >> 48);
                a[k] = 0;
            }
        };
#pragma unroll
        for (int k = 0; k < KD; k++) {
            a[k] = 0;
            sad[k][0] = sad[k][1] = sad[k][2] = sad[k][3] = 0;
        }
        if constexpr (SMALL) {
            if (pu.w & 7)
                for (int x = 0; x < pu.w >> 2; x++)
                    dense_strip<KD, 1>(w + x, v.pd, shift, cpu32 + x, v.cpd, pu.h, a);
            else
                for (int x = 0; x < pu.w >> 2; x += 2)
                    dense_strip<KD, 2>(w + x, v.pd, shift, cpu32 + x, v.cpd, pu.h, a);
            unpack();
        } else {
            for (int x = 0; x < pu.w >> 2; x += 2)
                for (int y = 0; y < pu.h; y += 32) {
                    dense_strip<KD, 2>(w + y * v.pd + x, v.pd, shift, cpu32 + y * v.cpd + x, v.cpd, min(32, pu.h - y), a);
                    unpack();
                }
        }
        uint32_t key = 0xFFFFFFFFu;
#pragma unroll
        for (int k = 0; k < KD; k++) {
            const uint32_t ty = wa->yt[row + k];
#pragma unroll
            for (int c = 0; c < 4; c++)
                sad[k][c] = ((sad[k][c] + ((wa->xt[col + c] + ty) >> 16)) << 5) | (uint32_t)(4 * k + c);
        }
        if (all_legal) {
#pragma unroll
            for (int k = 0; k < KD; k++)
                key = min(key, min(min(sad[k][0], sad[k][1]), min(sad[k][2], sad[k][3])));
        } else {
            const MvWindow mw = xme_mv_window(p, pu.x, pu.y, pu.w, pu.h);
#pragma unroll
            for (int k = 0; k < KD; k++)
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (xme_mv_legal(mw, in.omx + col + c - R, in.omy + row + k - R))
                        key = min(key, sad[k][c]);
        }
        const uint32_t cost = key >> 5;
        const uint32_t order =
            XME_ORDER_RASTER + (uint32_t)((row + (int)((key >> 2) & 7)) * 2 * R + col + (int)(key & 3));
        if (key != 0xFFFFFFFFu && (cost < bc || (cost == bc && order < bo))) {
            bc = cost;
            bo = order;
        }
    }
}

// K rows per lane for PUs up to 16 x 16, KM for the larger ones.  STRIPS: see
// kDenseNum; a template parameter, since as a branch in the loop over bands it
// cost every picture 2 %.
template <int K, int KM, bool STRIPS>
__global__ void __launch_bounds__(1024) elim_kernel(DevParams p, const FrameDesc *__restrict__ desc,
                                                    const DevInst *__restrict__ inst,
                                                    const FsTask *__restrict__ tasks, int n_tasks,
                                                    const ElItem *__restrict__ items, uint64_t *__restrict__ best,
                                                    uint32_t *__restrict__ counters, int lc_log2)
{
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ int s_task;
    __shared__ int s_item;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    WaveState rs;
    rs.dense = rs.run = 0;
    for (;;) {
        if (threadIdx.x == 0)
            s_task = (int)atomicAdd(&counters[0], 1u);
        __syncthreads();
        const int task = __builtin_amdgcn_readfirstlane(s_task);
        if (task >= n_tasks)
            break;
        const FsTask t = tasks[task];
        uint32_t *l32 = reinterpret_cast<uint32_t *>(lds);
        TaskView v;
        v.pd = xme_el_pitch(t.ww);
        v.cpd = t.cw >> 2;
        v.sp = xme_el_sum_pitch(t.ww);
        v.wx0 = t.wx0;
        v.wy0 = t.wy0;
        v.cx0 = t.cx0;
        v.cy0 = t.cy0;
        uint32_t *c32 = l32 + v.pd * t.wh;
        uint32_t *s32 = c32 + v.cpd * t.ch;
        uint32_t *a32 = s32 + v.sp * (t.wh - 3);
        a32 += (4 - ((a32 - l32) & 3)) & 3;
        v.w32 = l32;
        v.c32 = c32;
        v.s32 = s32;
        stage(t, desc, p, l32, v.pd, c32);
        if (threadIdx.x == 0)
            s_item = t.item_begin;
        __syncthreads();
        build_sums(t, l32, v.pd, s32, v.sp);
        __syncthreads();
        WaveArea *wa = reinterpret_cast<WaveArea *>(a32) + wave;
        rs.ok = false;
        rs.cx = rs.cy = rs.px = rs.py = 0;
        for (;;) {
            int it = 0;
            if ((threadIdx.x & 63) == 0)
                it = atomicAdd(&s_item, 1);
            it = __builtin_amdgcn_readlane(it, 0);
            if (it >= t.item_end)
                break;
            const ElItem item = items[it];
            // both in flight at once, whole records
            const uint4 q = reinterpret_cast<const uint4 *>(inst)[item.inst];
            const uint64_t key0 = best[item.inst];
            const DevInst in = __builtin_bit_cast(DevInst, q);
            if (in.status)
                continue;
            DevPu pu;
            pu.x = item.x;
            pu.y = item.y;
            pu.w = item.w;
            pu.h = item.h;
            pu.mvp_x = item.mvp_x;
            pu.mvp_y = item.mvp_y;
            const Box box = rate_terms(p, pu, in, wa, rs);
            uint32_t bc = 0xFFFFFFFFu, bo = 0xFFFFFFFFu;
            // rows still to search when it leaves some: before and after its bands
            int from[2] = { item.row0, 0 }, to[2] = { item.row0 + item.nrows, 0 };
            if (STRIPS && rs.dense > 0 && item.nrows >= (pu.w > 16 || pu.h > 16 ? KM : K)) {
                rs.dense--;
            } else {
                bool dense = false;
#define XME_EL(NXX, NYY, ONE)                                                                                  \
    dense = el_item<ONE ? K : KM, NXX, NYY, ONE, STRIPS>(p, v, pu, in, box, item.row0, item.nrows, lc_log2,    \
                                                         (uint32_t)(key0 >> 32), wa, rs, bc, bo, to[0], from[1])
                switch (pu.w * 64 + pu.h) {
                case 8 * 64 + 8: XME_EL(2, 2, true); break;
                case 16 * 64 + 16: XME_EL(4, 4, true); break;
                case 16 * 64 + 8: XME_EL(4, 2, true); break;
                case 8 * 64 + 16: XME_EL(2, 4, true); break;
                case 16 * 64 + 12: XME_EL(4, 3, true); break;
                case 12 * 64 + 16: XME_EL(3, 4, true); break;
                case 16 * 64 + 4: XME_EL(4, 1, true); break;
                case 4 * 64 + 16: XME_EL(1, 4, true); break;
                case 8 * 64 + 4: XME_EL(2, 1, true); break;
                case 4 * 64 + 8: XME_EL(1, 2, true); break;
                case 4 * 64 + 4: XME_EL(1, 1, true); break;
                case 32 * 64 + 8:
                case 32 * 64 + 24: XME_EL(4, 2, false); break;
                case 8 * 64 + 32:
                case 24 * 64 + 32: XME_EL(2, 4, false); break;
                default: XME_EL(4, 4, false); break;       // multiples of 16 on both sides
                }
#undef XME_EL
                to[1] = item.row0 + item.nrows;
                if (STRIPS)
                    rs.dense = rs.run = dense ? min(4 * rs.run + 3, kDenseRun) : 0;
            }
            if constexpr (STRIPS) {
                for (int k = 0; k < 2; k++) {
                    if (from[k] >= to[k])
                        continue;
                    if (pu.w * pu.h > 256)
                        dense_rows<KM / 2, false>(p, v, pu, in, box.all_legal, item.row0, from[k], to[k], lc_log2, wa, bc, bo);
                    else if (KM < K && (pu.w > 16 || pu.h > 16))
                        dense_rows<KM / 2, true>(p, v, pu, in, box.all_legal, item.row0, from[k], to[k], lc_log2, wa, bc, bo);
                    else
                        dense_rows<K / 2, true>(p, v, pu, in, box.all_legal, item.row0, from[k], to[k], lc_log2, wa, bc, bo);
                }
            }
            const uint32_t wc = wave_min(bc);
            const uint32_t wo = wave_min(bc == wc ? bo : 0xFFFFFFFFu);
            const uint64_t kbest = xme_key(wc, wo);
            if ((threadIdx.x & 63) == 0 && wc != 0xFFFFFFFFu && kbest < key0)
                atomicMin(reinterpret_cast<unsigned long long *>(best + item.inst), (unsigned long long)kbest);
        }
        __syncthreads();   // LDS is reused by the next task
    }
    if (threadIdx.x == 0) {
        // the last workgroup out resets the queue for the next launch / replay
        __threadfence();
        const uint32_t done = atomicAdd(&counters[1], 1u);
        if (done == gridDim.x - 1) {
            atomicExch(&counters[0], 0u);
            atomicExch(&counters[1], 0u);
        }
    }
}

// Every raster candidate's cost, -1 where CHECK_MV_RANGE rejects
// (xme_me_run's d_cost_map): a thread per 4 columns of a candidate row,
// straight from the planes.
__global__ void __launch_bounds__(256) cost_map_kernel(DevParams p, const FrameDesc *__restrict__ desc,
                                                       const DevPu *__restrict__ pus, const DevInst *__restrict__ inst)
{
    const int R = p.R, R2 = 2 * p.R, quads = (R2 + 3) >> 2, per = (R2 * quads + 255) >> 8;
    const int id = blockIdx.x / per;
    const DevInst in = inst[id];
    if (in.status)
        return;
    const int e = (blockIdx.x - id * per) * 256 + threadIdx.x;
    const int j = e / quads, i0 = 4 * (e - j * quads);
    if (j >= R2)
        return;
    const DevPu pu = pus[id / p.n_ref];
    const int r = id % p.n_ref;
    const MvWindow mw = xme_mv_window(p, pu.x, pu.y, pu.w, pu.h);
    const int64_t stride = desc->stride[r];
    int32_t *out = desc->cost_map + (int64_t)id * R2 * R2 + (int64_t)j * R2;
    for (int i = i0; i < min(i0 + 4, R2); i++) {
        const int mx = in.omx + i - R, my = in.omy + j - R;
        if (!xme_mv_legal(mw, mx, my)) {
            out[i] = -1;
            continue;
        }
        const uint8_t *rp = desc->planes[r][0] + (int64_t)(pu.y + my) * stride + pu.x + mx;
        const uint8_t *cp = desc->cur + (int64_t)pu.y * desc->i_cur + pu.x;
        const uint32_t sh = (uint32_t)(reinterpret_cast<uintptr_t>(rp) & 3);
        rp -= sh;
        uint32_t sad = 0;
        for (int y = 0; y < pu.h; y++, rp += stride, cp += desc->i_cur)
            for (int x = 0; x < pu.w; x += 4) {
                const uint32_t *q = reinterpret_cast<const uint32_t *>(rp + x);
                sad = __builtin_amdgcn_sad_u8(*reinterpret_cast<const uint32_t *>(cp + x),
                                              __builtin_amdgcn_alignbyte(q[1], q[0], sh), sad);
            }
        out[i] = (int)sad + xme_weighted_cost(p.lambda, xme_mvbits(4 * mx - pu.mvp_x) + xme_mvbits(4 * my - pu.mvp_y));
    }
}

const void *const kKernels[5] = {
    reinterpret_cast<const void *>(&elim_kernel<4, 4, false>),
    reinterpret_cast<const void *>(&elim_kernel<16, 8, false>),
    reinterpret_cast<const void *>(&elim_kernel<16, 8, true>),
    reinterpret_cast<const void *>(&elim_kernel<16, 16, false>),
    reinterpret_cast<const void *>(&elim_kernel<16, 16, true>),
};

// Whether noise is costed in strips rather than as listed tiles: with 16 rows
// per lane (at 4, R < 24, elimination is the quicker one on noise too) and
// where 3/4 of dense_rows' lanes have a candidate of their own, or 9/16 for odd
// R, whose tiles cost more.  1080p noise, mixed PUs, listed and in strips: R =
// 34 220 and 267 us, 48 330 and 333, 52 409 and 366, 49 495 and 403, 64 488 and
// 391.
bool el_strips(int R)
{
    if (R < 24)
        return false;
    const int lc = xme_el_lc_log2(R), band = (64 >> lc) * 16;
    return 64 * R * R > (R & 1 ? 9 : 12) * (2 << lc) * ((2 * R + band - 1) / band * band);
}

} // namespace

// 16 rows per lane share the map rows best; ranges below 24 leave lanes idle
// with them (64 / LC row groups of 16 rows exceed the 2R rows).  Where a frame
// gives a CU few tasks, PUs beyond 16 x 16 take 8 rows: their items are the
// longest, and half as long they leave a shorter tail (1080p mixed PUs, R =
// 32: 168 -> 141 us), at 14-18 % more work (2160p: 696 -> 734 us, 16 rows kept).
int xme_el_rows(int R, bool few_tasks, int w, int h)
{
    return R < 24 ? 4 : few_tasks && (w > 16 || h > 16) ? 8 : 16;
}

// Lanes per candidate row (2 columns each), as a power of two.
int xme_el_lc_log2(int R)
{
    int l = 1;
    while ((1 << l) < R)
        l++;
    return l;
}

int xme_el_prepare(void)
{
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        for (const void *k : kKernels)
            if (err == hipSuccess)
                err = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, xme_fs_max_lds());
    });
    if (err != hipSuccess)
        return xme_hip_fail(err, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
    return XME_OK;
}

const void *xme_el_kernel_ptr(int R, bool few_tasks)
{
    if (xme_el_rows(R, few_tasks, 4, 4) == 4)
        return kKernels[0];
    return kKernels[(xme_el_rows(R, few_tasks, 64, 64) == 8 ? 1 : 3) + (el_strips(R) ? 1 : 0)];
}

int xme_launch_elim(const DevParams &p, const FrameDesc *d_desc, const DevInst *d_inst, const FsTask *d_tasks,
                    int n_tasks, const ElItem *d_items, uint64_t *d_best, uint32_t *d_counters,
                    size_t lds_bytes, int grid, int threads, bool few_tasks, hipStream_t s)
{
    if (n_tasks <= 0)
        return XME_OK;
    int rc = xme_el_prepare();
    if (rc)
        return rc;
    int lc = xme_el_lc_log2(p.R);
    void *args[] = { (void *)&p, (void *)&d_desc, (void *)&d_inst, (void *)&d_tasks, (void *)&n_tasks,
                     (void *)&d_items, (void *)&d_best, (void *)&d_counters, (void *)&lc };
    XME_HIP(hipLaunchKernel(xme_el_kernel_ptr(p.R, few_tasks), dim3(grid), dim3(threads), args, lds_bytes, s));
    return XME_OK;
}

int xme_launch_cost_map(const DevParams &p, const FrameDesc *d_desc, const DevPu *d_pus, const DevInst *d_inst,
                        int n_inst, hipStream_t s)
{
    const int per = (2 * p.R * ((2 * p.R + 3) / 4) + 255) / 256;      // workgroups per instance
    hipLaunchKernelGGL(cost_map_kernel, dim3(per * n_inst), dim3(256), 0, s, p, d_desc, d_pus, d_inst);
    XME_HIP(hipGetLastError());
    return XME_OK;
}

// The projected Euclidean cascade (OmniVoice / Higgs acoustic quantizers) in
// one launch, for codebooks of width 64: per stage project_in, the codebook
// search and the hidden-space update, each in the reference's arithmetic
// (aq_projected.hip, aq_euclid_kernels.hpp), with the frames' hidden
// residuals in LDS throughout.
//
// A block of four waves takes F frames through all stages; two blocks share
// a CU, so that one's exact chains run beside the other's memory waits.
//  * project_in: weights and residual rows are laid out so that a lane's next
//    four elements of its accumulator's chain are 16 bytes: a 64-element
//    chunk as [16 tinyBLAS lanes][4 steps] for F32 weights, a 128-element
//    chunk as [8 int lanes][4 blocks] dwords for Q8_0.  A thread holds 4
//    outputs x F frames (Q8_0: 2 x F) of one lane; every weight is read once
//    per block, kAhead chunks ahead.
//  * search: the fp16 fragments of the F projected frames against the wave's
//    quarter of the codes, the key merge and select_group, the frames shared
//    out over the waves.  Frames the certificate leaves open are scanned
//    exactly by the block at once (N x 64 values cost about a microsecond),
//    so that every stage's input is the reference's.
//  * update: r -= table[code], the project_out rows built at upload.
// What bounds it: project_in's exact chains (F x 64 x H FMAs, one per lane and
// cycle; Q8_0: four operations per 4-element dot), and for few frames the
// weights' way into the CU (256 KB a stage).  The per-stage launches it
// replaces (projection, sweep, select, refine pair, exact scan; 16 frames
// per projection block) took 87 us a stage for 250 frames (now 11) and 177 us
// for 6 000 frames with Q8_0 weights (now 44); more at proj_frames() below.
#include "aq_euclid_kernels.hpp"
#include "aq_projected.hpp"

#include <cstdlib>

namespace {

constexpr int kPcWaves = 4;
constexpr int kPcThreads = kPcWaves * kWave;
constexpr int kPcKS = 2, kPcK = 64;
static_assert(kPcThreads == kScanThreads, "the exact scan's selection takes the whole block");
// Weight chunks in flight per thread; a row is a whole number of times as
// many (a remainder's conditional steps made the compiler copy the ring every
// round, waiting for all of it).
constexpr int kAhead = 4;
// Loops of these kernels, select_group's among them, run through scalar
// conditions (whole waves), not the execution mask: where a kernel spills,
// ROCm 7.2's compiler has put spill stores and reloads behind such a loop's
// exit, where no lane is active.  (All variants but the F32 ones of four
// frames spill, up to 78 registers; tests/test_kernel_code.py holds the count
// and looks at the built code.)
// Widest hidden size: rows are this far apart, so that a frame's offset is an
// immediate (as a run-time stride the addresses of F rows cost the registers
// of the chains).
constexpr int kPcH = 1024;

struct PcArgs {
    CascadeArgs c;           // stage 0's codebook pointers, bounds, counts; idx, dist, top-k
    aq_frames_desc in;
    const float *wx;         // [Q][64][H/64][16][4] F32 project_in
    const int *wqx;          // [Q][64][H/128][8][4] Q8_0 quants, four to a dword
    const float *wd;         // [Q][64][H/32] Q8_0 scales
    const float *bias;       // [Q][64] or null
    const float *table;      // [Q][N][H] project_out rows
    const int32_t *force;    // [M, Q] or null: the update's codes
    float *rout;             // [M, H] or null
    int H;
};

// LDS of a block (bytes): the residual rows, what outlives a phase, and one
// region for the phases (query blocks; fragments and keys; select queues;
// scan).
template <bool Q8C, int F, int TOPL>
struct PcLayout {
    static constexpr int XSTR = kPcK + 4;
    static constexpr int P = 16 * XSTR * 4;                 // projected rows (16: a fragment's columns)
    static constexpr int NRM = kPcKS * 3 * 16 * 4;
    static constexpr int SELB = (static_cast<int>(sizeof(SelLds<Q8C, kPcK, TOPL>)) + 15) / 16 * 16;
    static constexpr int XH = kPcKS * kWave * 16;
    static constexpr int KEYS = kPcWaves * TOPL * kWave * 4;
    static constexpr int SCAN = (static_cast<int>(sizeof(ScanSh)) + 15) / 16 * 16;
    static constexpr int SEARCH = cmax3(XH + KEYS, kPcWaves * SELB, SCAN);
    static constexpr int QROW = kPcH + 4 * (kPcH / 32);   // a frame's query blocks and scales
    static constexpr int bytes(bool q8w) {
        const int q = q8w ? F * QROW : 0;
        return F * kPcH * 4 + P + NRM + (q > SEARCH ? q : SEARCH);
    }
};

// The Q8_0 projection phases and the exact scan are calls of their own:
// inlined, their registers and the search's add up and spill.  project_f32 is
// inlined: as a call it left its kernels of 4 and 8 frames with 4 and 40
// spilled registers, for 0 and 18.  LDS goes to the projections as LDS
// pointers (a generic pointer would make every read a flat one), what is
// uniform back into scalar registers.
typedef __attribute__((address_space(3))) float lds_float;
typedef __attribute__((address_space(3))) int lds_int;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(1))) const char glb_char;
typedef __attribute__((address_space(1))) const float glb_float;
typedef __attribute__((address_space(1))) const f32x4 glb_f32x4;
typedef __attribute__((address_space(1))) const u32x4 glb_u32x4;
__device__ inline glb_char *uniform_ptr(const void *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint64_t lo = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
    const uint64_t hi = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)));
    return reinterpret_cast<glb_char *>(hi << 32 | lo);
}

// x of lane N of the lane's 16-lane row.
template <int N>
__device__ inline float row_bcast16(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + N, 0xF, 0xF, false));
}
// The largest of a row's 16 values (as unsigned bits; non-negative floats).
template <int N>
__device__ inline unsigned row_ror_umax(unsigned v) {
    return max(v, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x120 + N, 0xF, 0xF, false)));
}
__device__ inline unsigned row_umax16(unsigned v) {
    return row_ror_umax<1>(row_ror_umax<2>(row_ror_umax<4>(row_ror_umax<8>(v))));
}
__device__ inline float row_fmax16(float v) {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// Index (floats) in a residual row of quad `qd`: chunk qd / 16 of 64 elements,
// lane t = qd % 16 holding elements t, 16 + t, 32 + t, 48 + t.
__device__ inline int quad_elem(int qd, int i) { return (qd >> 4) * 64 + 16 * i + (qd & 15); }

// F32 project_in in tinyBLAS order: lane t of 16 accumulates k = 16 u + t, then
// _mm512_reduce_add_ps's pairing tree as DPP row rotations 8, 4, 2, 1.
template <int F>
__device__ __forceinline__ void project_f32(const float *wx_in, const float *bias_in, const lds_float *rows,
                                                      int H_in, lds_float *p) {
    constexpr int xstr = kPcK + 4;
    const int tid = threadIdx.x, t = tid & 15, slot = tid >> 4;   // 16 slots of 4 outputs
    glb_char *wx = uniform_ptr(wx_in);
    glb_float *bias = reinterpret_cast<glb_float *>(uniform_ptr(bias_in));
    const int nu = __builtin_amdgcn_readfirstlane(H_in) / 64;
    const unsigned mine = (static_cast<unsigned>(slot) * 4 * nu * 16 + t) * 16;   // bytes
    f32x4 ring[kAhead][4];
    auto load = [&](int u, int d) {
        const int uc = u < nu ? u : nu - 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) ring[d][i] = *reinterpret_cast<glb_f32x4 *>(wx + (i * nu + uc) * 256 + mine);
    };
#pragma unroll
    for (int d = 0; d < kAhead; ++d) {
        load(d, d);
        __builtin_amdgcn_sched_barrier(0);
    }
    float acc[4][F];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int f = 0; f < F; ++f) acc[i][f] = 0.0f;
    // Four frames at a time, 16 independent chains between the steps of one;
    // the next four's rows are read ahead of this four's chains.
    f32x4 r[4];
    auto load_rows = [&](int u, int fb) {
#pragma unroll
        for (int f = 0; f < 4; ++f)
            r[f] = *reinterpret_cast<const lds_f32x4 *>(rows + (fb + f) * kPcH + (u < nu ? u : nu - 1) * 64 + t * 4);
    };
    load_rows(0, 0);
    for (int u0 = 0; u0 < nu; u0 += kAhead) {
#pragma unroll
        for (int d = 0; d < kAhead; ++d) {
#pragma unroll
            for (int fb = 0; fb < F; fb += 4) {
                f32x4 rc[4];
#pragma unroll
                for (int f = 0; f < 4; ++f) rc[f] = r[f];
                load_rows(fb + 4 < F ? u0 + d : u0 + d + 1, fb + 4 < F ? fb + 4 : 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            acc[i][fb + f] = __fmaf_rn(ring[d][i][q], rc[f][q], acc[i][fb + f]);
            }
            load(u0 + d + kAhead, d);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int f = 0; f < F; ++f) {
            float v = row_ror_add<8>(acc[i][f]);
            v = row_ror_add<4>(v);
            v = row_ror_add<2>(v);
            acc[i][f] = row_ror_add<1>(v);
        }
    if (t != 0) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float b = bias ? bias[slot * 4 + i] : 0.0f;
#pragma unroll
        for (int f = 0; f < F; ++f) p[f * xstr + slot * 4 + i] = bias ? __fadd_rn(acc[i][f], b) : acc[i][f];
    }
}

// Q8_0 project_in from the frames' query blocks (xq: dwords [F][H/128][8][4],
// xd [F][H/32]): 8 int lanes per output, lane j holding word q8_lane_word(j)
// of every block, each 4-element dot scaled by d_w d_x and FMA-accumulated,
// then hsum_float_8 by DPP.
template <int F>
__device__ __attribute__((noinline)) void project_q8(const int *wqx_in, const float *wd_in, const float *bias_in,
                                                     const lds_int *xq, const lds_float *xd, int H_in, lds_float *p) {
    constexpr int xstr = kPcK + 4;
    const int tid = threadIdx.x, l = tid & 7, slot = tid >> 3;   // 32 slots of 2 outputs
    glb_char *wqx = uniform_ptr(wqx_in);
    glb_char *wd = uniform_ptr(wd_in);
    glb_float *bias = reinterpret_cast<glb_float *>(uniform_ptr(bias_in));
    const int nc = __builtin_amdgcn_readfirstlane(H_in) / 128;
    const unsigned mine = (static_cast<unsigned>(slot) * 2 * nc * 8 + l) * 16, scales = static_cast<unsigned>(slot) * 2 * nc * 16;
    u32x4 ring[kAhead][2];
    f32x4 sring[kAhead][2];
    auto load = [&](int u, int d) {
        const int uc = u < nc ? u : nc - 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ring[d][i] = *reinterpret_cast<glb_u32x4 *>(wqx + (i * nc + uc) * 128 + mine);
            sring[d][i] = *reinterpret_cast<glb_f32x4 *>(wd + (i * nc + uc) * 16 + scales);
        }
    };
#pragma unroll
    for (int d = 0; d < kAhead; ++d) {
        load(d, d);
        __builtin_amdgcn_sched_barrier(0);
    }
    float acc[2][F];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int f = 0; f < F; ++f) acc[i][f] = 0.0f;
    // in a register of its own: as a constant, every dot costs a move more
    int zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    u32x4 x[4];
    f32x4 xs[4];
    auto load_blocks = [&](int u, int fb) {   // as project_f32's rows
        const int uc = u < nc ? u : nc - 1;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            x[f] = *reinterpret_cast<const lds_u32x4 *>(xq + (fb + f) * (kPcH / 4) + uc * 32 + l * 4);
            xs[f] = *reinterpret_cast<const lds_f32x4 *>(xd + (fb + f) * (kPcH / 32) + uc * 4);
        }
    };
    load_blocks(0, 0);
    for (int u0 = 0; u0 < nc; u0 += kAhead) {
#pragma unroll
        for (int d = 0; d < kAhead; ++d) {
#pragma unroll
            for (int fb = 0; fb < F; fb += 4) {
                u32x4 xc[4];
                f32x4 sc[4];
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    xc[f] = x[f];
                    sc[f] = xs[f];
                }
                load_blocks(fb + 4 < F ? u0 + d : u0 + d + 1, fb + 4 < F ? fb + 4 : 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // the eight dots, then their conversions and scales, then
                    // the chains' steps: in a row, each dot's steps wait for
                    // one another
                    int dot[4][2];
                    float val[4][2], scale[4][2];
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int i = 0; i < 2; ++i)
                            dot[f][i] = __builtin_amdgcn_sdot4(static_cast<int>(ring[d][i][q]), static_cast<int>(xc[f][q]), zero, false);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            scale[f][i] = __fmul_rn(sring[d][i][q], sc[f][q]);
                            val[f][i] = static_cast<float>(dot[f][i]);
                        }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int i = 0; i < 2; ++i) acc[i][fb + f] = __fmaf_rn(scale[f][i], val[f][i], acc[i][fb + f]);
                }
            }
            load(u0 + d + kAhead, d);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int f = 0; f < F; ++f) acc[i][f] = hsum8_dpp(acc[i][f]);
    if (l != 0) return;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float b = bias ? bias[slot * 2 + i] : 0.0f;
#pragma unroll
        for (int f = 0; f < F; ++f) p[f * xstr + slot * 2 + i] = bias ? __fadd_rn(acc[i][f], b) : acc[i][f];
    }
}

// The frames' Q8_0 query blocks (x86 quantize_row_q8_0) from the residual
// rows, in project_q8's layout.  A 16-lane row takes a 64-element chunk (two
// blocks) of every frame; its blocks' scales are computed together, a block
// per lane, and handed back by row broadcasts.
template <int F, int J>
__device__ inline void q8_scales_back(const float d, const float id, float (&dv)[2 * F], float (&iv)[2 * F], int base) {
    if constexpr (J < 16) {
        if (base + J < 2 * F) {
            dv[base + J] = row_bcast16<J>(d);
            iv[base + J] = row_bcast16<J>(id);
        }
        q8_scales_back<F, J + 1>(d, id, dv, iv, base);
    }
}
template <int F>
__device__ __attribute__((noinline)) void quantize_rows(const lds_float *rows, int H_in, lds_int *xq, lds_float *xd) {
    const int tid = threadIdx.x, t = tid & 15, H = __builtin_amdgcn_readfirstlane(H_in);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    for (int q0 = wave * kWave; q0 < H / 4; q0 += kPcThreads) {   // whole waves
        const int qd = q0 + (tid & (kWave - 1));
        f32x4 v[F];
        unsigned am[2 * F];   // |x| as bits: an infinity or NaN ends up above every finite value
        float dv[2 * F], iv[2 * F];
#pragma unroll
        for (int f = 0; f < F; ++f) {
            v[f] = *reinterpret_cast<const lds_f32x4 *>(rows + f * kPcH + qd * 4);
            unsigned u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = __float_as_uint(v[f][i]) & 0x7FFFFFFFu;
            am[2 * f] = row_umax16(max(u[0], u[1]));
            am[2 * f + 1] = row_umax16(max(u[2], u[3]));
        }
        bool odd = false;   // a non-finite block, or one so small that 127 / amax is infinite
#pragma unroll
        for (int b0 = 0; b0 < 2 * F; b0 += 16) {
            unsigned mine = 0;
            float d, id;
#pragma unroll
            for (int j = 0; j < 16 && b0 + j < 2 * F; ++j) mine = t == j ? am[b0 + j] : mine;
            q8_scale(__uint_as_float(mine), d, id);
            odd = odd || mine >= 0x7F800000u || !(id < INFINITY);
            q8_scales_back<F, 0>(d, id, dv, iv, b0);
        }
        const bool plain = !__any(odd);   // wave-uniform
        const int ib0 = (qd >> 4) * 2;    // the chunk's first block
#pragma unroll
        for (int f = 0; f < F; ++f) {
            if (!plain) {   // fmaxf's amax, which passes over a NaN
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    q8_scale(row_fmax16(fmaxf(fabsf(v[f][2 * h]), fabsf(v[f][2 * h + 1]))), dv[2 * f + h], iv[2 * f + h]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int b = 2 * f + i / 2, ib = ib0 + i / 2;
                // plain: |x * id| <= 127 (1 + 2^-23)^2, the rounded value is
                // an integer in [-127, 127]
                unsigned q = static_cast<unsigned>(plain ? static_cast<int>(__builtin_rintf(__fmul_rn(v[f][i], iv[b])))
                                                         : q8_quant(v[f][i], iv[b])) & 0xFFu;
                // four neighbouring lanes' quants into a dword
                q |= static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(q), 0xB1, 0xF, 0xF, false)) << 8;
                q |= static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(q), 0x4E, 0xF, 0xF, false)) << 16;
                // word 4 (i % 2) + t / 4 of block ib goes to the lane that
                // holds it (q8_lane_word is its own inverse)
                const int wl = q8_lane_word(4 * (i & 1) + t / 4);
                if ((t & 3) == 0) xq[f * (kPcH / 4) + (ib / 4) * 32 + wl * 4 + ib % 4] = static_cast<int>(q);
                if (t == 0 && (i & 1) == 0) xd[f * (kPcH / 32) + ib] = dv[b];
            }
        }
    }
}

// The exact scan of one frame (x in LDS) by the block.  A call, not inlined:
// it is rare, and its registers would be the kernel's (some 90 spilled).
template <int RECIPE, bool Q8C>
__device__ __attribute__((noinline)) void scan_open(const float *cbf, const float *bias, const float *e2, const int8_t *q8,
                                                    const float *q8d, int N, int topk, const float *x, int8_t *xq,
                                                    float *xd, ScanSh *shp) {
    ScanSh &sh = *shp;
    StageArgs a{};
    a.cbf = cbf;
    a.bias = bias;
    a.e2 = e2;
    a.q8 = q8;
    a.q8d = q8d;
    a.N = N;
    a.topk = topk;
    a.order = 0;
    __syncthreads();
    if (threadIdx.x == 0) sh.o_x2 = RECIPE == HIGGS ? sum_squares_k<kPcK>(x) : 0.0f;
    if (Q8C && threadIdx.x < kPcKS) quantize_block_q8(x + 32 * threadIdx.x, xq + 32 * threadIdx.x, xd + threadIdx.x);
    __syncthreads();
    scan_frame<RECIPE, Q8C, kPcKS>(a, x, xq, xd, sh);
    __syncthreads();
}

// The search's loops are the narrow cascade's (euclid_narrow_kernel) for one
// group of frames: as shared code they cost its widest tile 10 to 25 spilled
// registers and 13 % at 6 000 frames, so that it keeps its own.  What the
// certificate rests on is shared: pack_slice, insert_key, merge_key.
//
// K-slice ks of 16 frames' fp32 rows (xrow: the lane's frame's row) as fp16
// fragments, with the slice's part of the rounding norms |x~|^2, |x - x~|^2,
// |x|^2 (n3[0], n3[stride], n3[2 stride], written for the lane's frame by its
// first lane).  A Q8_0 codebook scores the query's Q8_0 image.
template <bool Q8>
__device__ inline u32x4 fragment_slice(const float *xrow, int ks, int kq, float *n3, int stride) {
    const float *row = xrow + ks * 32 + kq * 8;
    const f32x4 lo = *reinterpret_cast<const f32x4 *>(row), hi = *reinterpret_cast<const f32x4 *>(row + 4);
    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    if (Q8) q8_image_block(v);
    float sx, sd, sxx;
    const u32x4 packed = pack_slice(v, sx, sd, sxx);
    if (kq == 0) {
        n3[0] = sx;
        n3[stride] = sd;
        n3[2 * stride] = sxx;
    }
    return packed;
}

// One wave's share of a codebook in fragment order: the 16-code blocks wave,
// wave + NW, ..., contracted with the frames' fragments, R fragments ahead.
template <int KS, int TS, int R, int NW>
struct CodeStream {
    using MX = Mx;
    static constexpr int U = R > KS ? R / KS : 1;   // 16-code blocks per unrolled step
    static_assert((U * KS) % R == 0, "the ring's slots are fixed within a step");
    typename MX::V8 ring[R];
    f32x4 hring[U];
    int wave, lane, nb;
    __device__ CodeStream(int N, int wave_, int lane_) : wave(wave_), lane(lane_) {
        const int nblk = N / 16;
        nb = wave < nblk ? (nblk - wave + NW - 1) / NW : 0;
    }
    // block i of this wave (past its last: the last again, whose keys are
    // not inserted)
    __device__ int blk_of(int i) const { return wave + NW * (i < nb ? i : nb - 1); }
    __device__ typename MX::V8 load_a(const uint16_t *cbx, int i, int ks) const {
        return reinterpret_cast<const typename MX::V8 *>(cbx)[(static_cast<int64_t>(blk_of(i)) * KS + ks) * kWave + lane];
    }
    __device__ f32x4 load_h(const float *nhh, int i) const {
        return *reinterpret_cast<const f32x4 *>(nhh + blk_of(i) * 16 + (lane >> 4) * 4);
    }
    // the first R fragments, in the sweep's order (a block's constants, then
    // its fragments), so that the waits at its head hold on entry too
    __device__ void fill(const uint16_t *cbx, const float *nhh) {
        if (nb == 0) return;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            hring[u] = load_h(nhh, u);
#pragma unroll
            for (int p = u * KS; p < (u + 1) * KS && p < R; ++p) {
                __builtin_amdgcn_sched_barrier(0);
                ring[p] = load_a(cbx, p / KS, p % KS);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __device__ void sweep(const uint16_t *cbx, const float *nhh, const typename MX::V8 (&xb)[KS], float (&top)[TS],
                          unsigned vkeep) {
#pragma unroll
        for (int j = 0; j < TS; ++j) top[j] = -INFINITY;
        for (int i0 = 0; i0 < nb; i0 += U) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                f32x4 acc = hring[u];
                hring[u] = load_h(nhh, i0 + u + U);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const int p = u * KS + ks;
                    acc = MX::mfma(ring[p % R], xb[ks], acc);
                    ring[p % R] = load_a(cbx, i0 + (p + R) / KS, (p + R) % KS);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (i0 + u >= nb) continue;   // wave-uniform
                const unsigned local0 = static_cast<unsigned>(wave + NW * (i0 + u)) * 4;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // in a scalar register of its own, so that the key is one
                    // v_and_or_b32
                    unsigned local = local0 + i;
                    asm("" : "+s"(local));
                    insert_key(key_of(acc[i], local, vkeep), top);
                }
            }
        }
    }
};

template <int RECIPE, bool Q8C, bool Q8W, int F, int TOPL>
__global__ __launch_bounds__(kPcThreads, 2) void proj_cascade_kernel(PcArgs pa) {
    using LY = PcLayout<Q8C, F, TOPL>;
    constexpr int XSTR = LY::XSTR;
    constexpr int R = 16;
    static_assert(F % kPcWaves == 0 && F <= 16, "frames of a block");
    constexpr int FPW = F / kPcWaves;
    extern __shared__ __align__(16) unsigned char lds[];
    const int H = pa.H;
    float *rows = reinterpret_cast<float *>(lds);   // [F][kPcH], quads (quad_elem)
    unsigned char *fixed = lds + F * kPcH * 4;
    float *p = reinterpret_cast<float *>(fixed);                  // [16][XSTR]
    float *nrm = reinterpret_cast<float *>(fixed + LY::P);        // [KS][3][16]
    unsigned char *phase = fixed + LY::P + LY::NRM;
    int *xq = reinterpret_cast<int *>(phase);
    float *xd = reinterpret_cast<float *>(phase + F * kPcH);
    u32x4 *xh = reinterpret_cast<u32x4 *>(phase);
    float *keys = reinterpret_cast<float *>(phase + LY::XH);
    ScanSh &sh = *reinterpret_cast<ScanSh *>(phase);
    __shared__ int s_code[16], s_open[16], s_nopen;
    __shared__ int64_t s_base[F];
    __shared__ __align__(16) int8_t s_xq[kPcK];
    __shared__ float s_xd[kPcKS];

    const lds_float *lrows = (const lds_float *)rows;

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int col = lane & 15, kq = lane >> 4;
    const int64_t M = pa.c.a.M;
    const int N = pa.c.a.N, Q = pa.c.a.Q;
    const int64_t m0 = static_cast<int64_t>(blockIdx.x) * F;
    if (m0 >= M) return;   // block-uniform
    const int nf = static_cast<int>(M - m0 < F ? M - m0 : F);

    int lbits = 0;   // bits of the lane-local code index (N/4 codes per lane)
    while ((1 << lbits) < N / 4) ++lbits;
    unsigned vkeep;
    asm volatile("v_mov_b32 %0, %1" : "=v"(vkeep) : "s"(~((1u << lbits) - 1u)));

    // ---- the input rows (rows past M read the block's first frame) ----
    if (tid < F) {
        const int64_t m = m0 + (tid < nf ? tid : 0);
        s_base[tid] = (m / pa.in.clip_len) * pa.in.clip_stride + (m % pa.in.clip_len) * pa.in.frame_stride;
    }
    for (int e0 = 0; e0 < 16 * XSTR; e0 += kPcThreads)
        if (e0 + tid < 16 * XSTR) p[e0 + tid] = 0.0f;
    if (tid == 0) s_nopen = 0;
    __syncthreads();
    // channel-adjacent frames are read frame-fastest, so that a wave's loads
    // stay close together
    const bool frames_adjacent = pa.in.frame_stride == 1 && pa.in.chan_stride != 1;
#pragma unroll 8
    for (int e0 = 0; e0 < F * H; e0 += kPcThreads) {   // H is a multiple of the block's threads
        const int e = e0 + tid;
        const int f = frames_adjacent ? e % F : e / H, h = frames_adjacent ? e / F : e % H;
        const float v = pa.in.x[s_base[f] + static_cast<int64_t>(h) * pa.in.chan_stride];
        rows[f * kPcH + (h >> 6) * 64 + (h & 15) * 4 + ((h >> 4) & 3)] = v;
    }
    // r -= table[code], the forced code where given
    auto update = [&](int s, int tid) {
        for (int q0 = wave * kWave; q0 < H / 4; q0 += kPcThreads) {   // whole waves
            const int qd = q0 + (tid & (kWave - 1));
            float tv[F][4];
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const float *row = pa.table + (static_cast<int64_t>(s) * N + s_code[f]) * H;
#pragma unroll
                for (int i = 0; i < 4; ++i) tv[f][i] = row[quad_elem(qd, i)];
            }
#pragma unroll
            for (int f = 0; f < F; ++f) {
                f32x4 *d = reinterpret_cast<f32x4 *>(rows + f * kPcH + qd * 4);
                f32x4 o = *d;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = __fsub_rn(o[i], tv[f][i]);
                *d = o;
            }
        }
    };

    for (int s = 0; s < Q; ++s) {
        // the thread's index, opaque in every stage: the addresses made from
        // it are not kept in registers across the stages
        int st = tid;
        asm volatile("" : "+v"(st));
        StageArgs a = cascade_stage(pa.c, s, kPcK);
        a.fail_count = &s_nopen;   // the frames this block scans below
        a.fail_list = s_open;
        a.xin = nullptr;
        a.xout = nullptr;
        a.force_idx = nullptr;
        a.order = 0;   // tinyBLAS: at least two frames, a width of 64
        const uint16_t *cbx = pa.c.cbx + static_cast<int64_t>(s) * N * kPcK;
        if (s > 0) update(s - 1, st);
        __syncthreads();
        // ---- project_in ----
        const float *bias = pa.bias ? pa.bias + s * kPcK : nullptr;
        if constexpr (Q8W) {
            quantize_rows<F>(lrows, H, (lds_int *)xq, (lds_float *)xd);
            __syncthreads();
            project_q8<F>(pa.wqx + static_cast<int64_t>(s) * kPcK * (H / 4), pa.wd + static_cast<int64_t>(s) * kPcK * (H / 32),
                          bias, (const lds_int *)xq, (const lds_float *)xd, H, (lds_float *)p);
        } else {
            project_f32<F>(pa.wx + static_cast<int64_t>(s) * kPcK * H, bias, lrows, H, (lds_float *)p);
        }
        CodeStream<kPcKS, TOPL, R, kPcWaves> codes(N, wave, lane);
        codes.fill(cbx, a.nhh);
        __syncthreads();
        // ---- search ----
        if (wave < kPcKS)
            xh[wave * kWave + lane] = fragment_slice<Q8C>(p + col * XSTR, wave, kq, nrm + wave * 3 * 16 + col, 16);
        __syncthreads();
        typename Mx::V8 xb[kPcKS];
#pragma unroll
        for (int ks = 0; ks < kPcKS; ++ks) xb[ks] = __builtin_bit_cast(typename Mx::V8, xh[ks * kWave + lane]);
        float top[TOPL];
        codes.sweep(cbx, a.nhh, xb, top, vkeep);
#pragma unroll
        for (int j = 0; j < TOPL; ++j) keys[(wave * TOPL + j) * kWave + lane] = top[j];
        __syncthreads();
        float mt[TOPL], taul = -INFINITY, n3[3];
#pragma unroll
        for (int j = 0; j < TOPL; ++j) mt[j] = -INFINITY;
#pragma unroll
        for (int w = 0; w < kPcWaves; ++w)
#pragma unroll
            for (int j = 0; j < TOPL; ++j) merge_key(keys[(w * TOPL + j) * kWave + lane], j == TOPL - 1, mt, taul);
#pragma unroll
        for (int q = 0; q < 3; ++q) n3[q] = nrm[q * 16 + col] + nrm[(3 + q) * 16 + col];
        __syncthreads();   // keys and fragments are read: the select queues take their place
        const int f0 = wave * FPW;
        if (f0 < nf) {   // wave-uniform
            SelLds<Q8C, kPcK, TOPL> &sl = *reinterpret_cast<SelLds<Q8C, kPcK, TOPL> *>(phase + wave * LY::SELB);
            const int code = select_group<RECIPE, Q8C, kPcKS, TOPL>(a, m0, mt, taul, n3[0], n3[1], n3[2], sl, false, p,
                                                                    XSTR, false, ((1u << FPW) - 1u) << f0);
            if (kq == 0 && col >= f0 && col < f0 + FPW) s_code[col] = code >= 0 ? code : 0;
        } else if (kq == 0 && col >= f0 && col < f0 + FPW) {
            s_code[col] = 0;
        }
        __syncthreads();
        // ---- the open frames, exactly ----
        const int nopen = s_nopen;
        for (int o = 0; o < nopen; ++o) {
            const int f = static_cast<int>(s_open[o] - m0);
            scan_open<RECIPE, Q8C>(a.cbf, a.bias, a.e2, a.q8, a.q8d, N, a.topk, p + f * XSTR, s_xq, s_xd, &sh);
            if (tid == 0) {
                const int64_t at = (m0 + f) * Q + s;
                a.idx[at] = sh.o_code;
                if (a.dist) a.dist[at] = -sh.o_code_v;
                for (int r = 0; r < a.topk; ++r) {
                    a.topk_idx[at * a.topk + r] = sh.o_sel_n[r];
                    a.topk_dist[at * a.topk + r] = -sh.o_sel_v[r];
                }
                s_code[f] = sh.o_code;
            }
        }
        if (tid == 0 && nopen > 0) {
            atomicAdd(&pa.c.counts[s % 64], nopen);
            atomicAdd(&pa.c.counts[64 + s % 64], nopen);
            s_nopen = 0;
        }
        if (pa.force) {
            __syncthreads();
            if (tid < nf) {
                int u = pa.force[(m0 + tid) * Q + s];
                if (u < 0 || u >= N) {
                    a.flags[AQ_FLAG_BAD_INDEX] = 1;
                    u = 0;
                }
                s_code[tid] = u;
            }
        }
        __syncthreads();
    }
    if (pa.rout) {
        update(Q - 1, tid);
        __syncthreads();
        for (int f = 0; f < nf; ++f)
            for (int q0 = wave * kWave; q0 < H / 4; q0 += kPcThreads) {
                const int qd = q0 + lane;
                const f32x4 v = *reinterpret_cast<const f32x4 *>(rows + f * kPcH + qd * 4);
#pragma unroll
                for (int i = 0; i < 4; ++i) pa.rout[(m0 + f) * H + quad_elem(qd, i)] = v[i];
            }
    }
}

// project_in weights in the kernels' layouts.
__global__ void pc_weights_f32_kernel(const float *__restrict__ w, int64_t n, int H, float *__restrict__ wx) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int64_t row = e / H;
    const int h = static_cast<int>(e % H);
    wx[row * H + (h >> 6) * 64 + (h & 15) * 4 + ((h >> 4) & 3)] = w[e];
}
__global__ void pc_weights_q8_kernel(const int *__restrict__ wq, int64_t n, int H, int *__restrict__ wqx) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;   // a dword of quants
    if (e >= n) return;
    const int64_t row = e / (H / 4);
    const int d = static_cast<int>(e % (H / 4)), ib = d / 8;
    wqx[row * (H / 4) + (ib / 4) * 32 + q8_lane_word(d % 8) * 4 + ib % 4] = wq[e];
}

using PcFn = void (*)(PcArgs);
struct PcKernel {
    PcFn fn;
    int frames, lds;
};
template <int RECIPE, bool Q8C, bool Q8W, int TOPL>
PcKernel pick_frames(int F) {
    switch (F) {
        case 4: return {proj_cascade_kernel<RECIPE, Q8C, Q8W, 4, TOPL>, 4, PcLayout<Q8C, 4, TOPL>::bytes(Q8W)};
        case 8: return {proj_cascade_kernel<RECIPE, Q8C, Q8W, 8, TOPL>, 8, PcLayout<Q8C, 8, TOPL>::bytes(Q8W)};
        default: return {proj_cascade_kernel<RECIPE, Q8C, Q8W, 12, TOPL>, 12, PcLayout<Q8C, 12, TOPL>::bytes(Q8W)};
    }
}
template <int RECIPE, bool Q8C>
PcKernel pick(bool q8w, int topl, int F) {
    if (q8w) return topl == 3 ? pick_frames<RECIPE, Q8C, true, 3>(F) : pick_frames<RECIPE, Q8C, true, 4>(F);
    return topl == 3 ? pick_frames<RECIPE, Q8C, false, 3>(F) : pick_frames<RECIPE, Q8C, false, 4>(F);
}

// Frames per block, by the estimated time of the launch: rounds of two blocks
// per CU, a last round of at most one block per CU at that block's own time.
// The times of both are eight stages' at H = 1 024, N = 1 024, F32 (Q8_0's
// have the same proportions: 130 / 185, 180 / 254, 260 / 345 us), in us:
//   frames        4    8   12 per block   per-stage launches
//      250       89  125  159                  699
//    2 048      132  132  162                  703
//    4 096      241  165  211                  720
//    6 000      333  256  218                  759
// (Q8_0 weights and codebook, 250: 130, 181, 260, per stage 792; 4 096: 349,
// 254, 339, 835; 6 000: 511, 404, 348, 1 415.)
int proj_frames(int64_t M, int cus) {
    if (const char *e = std::getenv("AQ_PROJ_FRAMES")) {   // comparisons and tests: 4, 8 or 12
        const int f = std::atoi(e);
        if (f == 4 || f == 8 || f == 12) return f;
    }
    constexpr struct {
        int frames;
        int64_t alone, pair;
    } kinds[] = {{4, 91, 131}, {8, 125, 165}, {12, 160, 215}};
    int best = 0;
    int64_t best_cost = 0;
    for (const auto &k : kinds) {
        const int64_t blocks = (M + k.frames - 1) / k.frames, rest = blocks % (2 * cus);
        const int64_t cost = blocks / (2 * cus) * k.pair + (rest == 0 ? 0 : (rest <= cus ? k.alone : k.pair));
        if (best == 0 || cost < best_cost) {
            best = k.frames;
            best_cost = cost;
        }
    }
    return best;
}

}  // namespace

bool aq_proj_cascade_shape(const aq_proj_weights *pw, int64_t N) {
    return pw->K == kPcK && pw->H <= kPcH && pw->H % ((pw->q8 ? 128 : 64) * kAhead) == 0 && N % 16 == 0 && N >= 64 &&
           N <= kScanChunk;
}

size_t aq_proj_cascade_bytes(const aq_proj_weights *pw) {
    return static_cast<size_t>(pw->Q * pw->K * pw->H) * (pw->q8 ? 1 : 4);
}

aq_status aq_proj_cascade_weights(aq_ctx *ctx, aq_proj_weights *pw) {
    const int64_t n = static_cast<int64_t>(aq_proj_cascade_bytes(pw)) / 4;   // dwords
    const dim3 grid(static_cast<unsigned>((n + 255) / 256)), block(256);
    if (pw->q8)
        hipLaunchKernelGGL(pc_weights_q8_kernel, grid, block, 0, ctx->stream, reinterpret_cast<const int *>(pw->w_in_q), n,
                           static_cast<int>(pw->H), static_cast<int *>(pw->w_cx));
    else
        hipLaunchKernelGGL(pc_weights_f32_kernel, grid, block, 0, ctx->stream, pw->w_in, n, static_cast<int>(pw->H),
                           static_cast<float *>(pw->w_cx));
    AQ_HIP(ctx, hipGetLastError());
    return AQ_OK;
}

aq_status aq_proj_cascade(aq_ctx *ctx, const aq_proj_weights *pw, const CascadeArgs &c, bool q8c, int recipe, int topl,
                          const aq_frames_desc &in, const int32_t *force, float *rout, bool timed) {
    const int64_t M = c.a.M;
    const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
    const int F = proj_frames(M, cus);
    PcKernel k;
    if (recipe == AQ_EUCLID_OMNIVOICE) k = pick<OMNI, false>(pw->q8, topl, F);
    else if (q8c) k = pick<HIGGS, true>(pw->q8, topl, F);
    else k = pick<HIGGS, false>(pw->q8, topl, F);
    const void *fn = reinterpret_cast<const void *>(k.fn);
    aq_status ls = aq_launch_lds(ctx, fn, static_cast<size_t>(k.lds), "aq_euclid_encode (projected cascade)");
    if (ls != AQ_OK) return ls;
    PcArgs a{};
    a.c = c;
    a.in = in;
    a.wx = pw->q8 ? nullptr : static_cast<const float *>(pw->w_cx);
    a.wqx = pw->q8 ? static_cast<const int *>(pw->w_cx) : nullptr;
    a.wd = pw->w_in_d;
    a.bias = pw->b_in;
    a.table = pw->table;
    a.force = force;
    a.rout = rout;
    a.H = static_cast<int>(pw->H);
    aq_launch_timed(ctx, timed, k.fn, dim3(static_cast<unsigned>((M + k.frames - 1) / k.frames)), dim3(kPcThreads),
                    static_cast<uint32_t>(k.lds), a);
    AQ_HIP(ctx, hipGetLastError());
    return AQ_OK;
}

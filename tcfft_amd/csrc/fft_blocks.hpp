// fft_blocks.hpp -- device building blocks shared by the pass kernels
// (fft_kernels.hip) and the fused convolution kernels (conv.hip): epilogue
// twiddles, the in-wave 4096-point DIT, and the 4096*W-point single-pass
// transform (load, per-line DIT, LDS exchange, radix-W stage, store).
#pragma once
#include "fft_device.hpp"
#include "fft_kernels.hpp"

namespace tcfft {

// Start delay of a first-pass workgroup under schedule s (see StartSched):
// s.delay sleep quanta of 1024 cycles per group index, for the workgroups of
// the first resident wave only.  The loop count is uniform and bounded.
__device__ __forceinline__ void start_delay(const StartSched& s) {
    if (s.delay && blockIdx.x < s.resident) {
        const u32 quanta = ((blockIdx.x >> 3) % s.groups) * s.delay;
        for (u32 i = 0; i < quanta; ++i) __builtin_amdgcn_s_sleep(16);
    }
}

// Epilogue twiddle for the next pass: element at position P (within the
// transform axis, P = global_pos >> shift) gets W_{s*R}^{c*rev(j)} with
// c = P mod s, j = (P / s) mod R and rev the two-digit DIT reversal of the
// next pass (radix ra first, then R/ra).  W_M^m = hi[m >> lo_bits]*lo[m & lo_mask].
// Digit reversal of a row index j (0 <= j < R) of the next pass, whose DIT
// digits are [2^ra, 2^rb, 2^rc] (rc = r - ra - rb, often 0):
// j = j0 + 2^ra*j1 + 2^(ra+rb)*j2 -> j2 + 2^rc*j1 + 2^(rc+rb)*j0.
__device__ __forceinline__ u32 epi_rev_row(const EpiParams& e, u32 j) {
    const u32 rc = e.r_log2 - e.ra_log2 - e.rb_log2;
    const u32 j0 = j & ((1u << e.ra_log2) - 1u);
    const u32 j1 = (j >> e.ra_log2) & ((1u << e.rb_log2) - 1u);
    const u32 j2 = j >> (e.ra_log2 + e.rb_log2);
    return j2 | (j1 << rc) | (j0 << (rc + e.rb_log2));
}

__device__ __forceinline__ cf epi_twiddle(const EpiParams& e, u32 gpos, float sgn) {
    const u32 P = gpos >> e.shift;
    const u32 c = P & ((1u << e.s_log2) - 1u);
    const u32 j = (P >> e.s_log2) & ((1u << e.r_log2) - 1u);
    const u32 rj = epi_rev_row(e, j);
    const u32 m = (c * rj) & e.m_mask;
    const cf a = twiddle(e.hi, m >> e.lo_bits, sgn);
    const cf b = twiddle(e.lo, m & ((1u << e.lo_bits) - 1u), sgn);
    return cmul(a, b);
}

// Strided passes see their output at (block blk, row, column col) of a
// buffer viewed as [blk][R][s]; along the axis that is P = blk*R*sa + row*sa
// + xc with sa = s >> shift and xc = col >> shift, so the next pass's twiddle
// is W_M^{(row*sa + xc)*rev(blk mod R')}: a per-column factor times a
// per-row factor, both powers of one root.  epi_rev gives rev(blk mod R'),
// epi_w gives W_M^m from the two-level table.
__device__ __forceinline__ u32 epi_rev(const EpiParams& e, u32 blk) {
    return epi_rev_row(e, blk & ((1u << e.r_log2) - 1u));
}

__device__ __forceinline__ cf epi_w(const EpiParams& e, u32 m, float sgn) {
    m &= e.m_mask;
    return cmul(twiddle(e.hi, m >> e.lo_bits, sgn), twiddle(e.lo, m & ((1u << e.lo_bits) - 1u), sgn));
}

// ----------------------------------------------------------------------------
// In-wave 4096-point DIT over the digits d0, d1, d2 of a 4096-element chunk.
// In : d[t][j] = tile t (d2), lane (c16 = d1, g), word j (d0 = 4g + j).
// Out: d[t][i] = tile t (k0), lane%16 = k1, (g, i) = k2, after post(t, i, v)
//      is applied to every FP32 result of the last stage.
// Stage-1 twiddle W_256^{k0*d1} is a per-lane constant; the stage-2 twiddle
// W_4096^{(k0+16k1)*d2} is a per-lane recurrence over the tiles.  The
// last stage uses the operand make_op2() (B-form), which may carry a row
// scale; it is built after stage 1 so that it holds no registers before.
// With REC0 the stage-2 inputs of column c = k0 + 16*k1 are also multiplied
// by rec0[i] (k0 = 4g + i, k1 = lane%16): a per-column factor of the caller
// merged into the stage-1 recurrence (rec = rec0 * W_4096^{c*d2}).
// The per-lane twiddles come from the caller (Dit4096Tw), loaded before the
// data: global loads complete in issue order, so a table load issued after
// the data loads would hold stage 0 until the whole chunk has arrived.
struct Dit4096Tw {
    float2 tw1[4], step[4];  // raw table entries: W_256^{k0*d1}, W_4096^{k0+16*k1}
};

__device__ __forceinline__ void dit4096_tw_load(Dit4096Tw& tw, int lane, const float2* __restrict__ w4096) {
    const int c16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        tw.tw1[i] = w4096[((c16 * (4 * g + i)) & 255) * 16];
        tw.step[i] = w4096[16 * c16 + 4 * g + i];
    }
}

template <bool REC0, class MakeOp2, class Post>
__device__ __forceinline__ void dit4096(u32 (&d)[16][4], int sign, const Dit4096Tw& tw, const Dft16Op& op,
                                        MakeOp2 make_op2, const cf (&rec0)[4], Post post) {
    const float sg = sign < 0 ? 1.f : -1.f;
    cf tw1[4], step[4], rec[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        tw1[i] = cf{tw.tw1[i].x, sg * tw.tw1[i].y};
        step[i] = cf{tw.step[i].x, sg * tw.step[i].y};
        rec[i] = REC0 ? rec0[i] : step[i];
    }
    // Stages 0 and 1 only combine points of one tile, so both run tile by
    // tile: tile t needs only its own load, and with the loads issued in tile
    // order (they complete in issue order) its work starts as soon as that
    // load has arrived instead of after the last one.
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        // stage 0: DFT over d0 -> lane%16 = k0, (g,i) = d1
        f32x4 re, im;
        dft16_a(d[t], op, re, im);
#pragma unroll
        for (int i = 0; i < 4; ++i) d[t][i] = pack(cmul(cf{re[i], im[i]}, tw1[i]));
        // stage 1: DFT over d1 -> lane%16 = k1, (g,i) = k0, tile = d2; twiddle W_4096^{c*d2}
        dft16_a(d[t], op, re, im);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            cf v = {re[i], im[i]};
            if (REC0 || t) {
                v = cmul(v, rec[i]);
                if (t < 15) rec[i] = cmul(rec[i], step[i]);
            }
            d[t][i] = pack(v);
        }
    }
    u32 e[16][4];
    transpose_gi_tile(d, e);  // (g,i) = d2, tile = k0
    const Dft16Op op2 = make_op2();
    // stage 2 (B-form): columns k1, points d2 -> (g,i) = k2
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        f32x4 re, im;
        dft16_b(e[t], op2, re, im);
#pragma unroll
        for (int i = 0; i < 4; ++i) d[t][i] = pack(post(t, i, cf{re[i], im[i]}));
    }
}

// ----------------------------------------------------------------------------
// Natural-order input of the row passes, straight into the digit-reversed
// register layout (tile t = line*T + d2, lane (c16 = d1, g), word j: d0 = 4g
// + j) without LDS.  Natural index of a line: m = d2 + T*(d1 + 16*d0), so a
// lane's points with the same d0 are T adjacent words.  T = 2 and 4 load them
// as they stand; T = 8 and 16 load four adjacent words per lane, so that a
// wave instruction covers whole 128-byte lines, and swap lane bit 4 (and 5),
// which then holds d2 bit 2 (and 3), with the register bits of d0.  Measured
// against 16-byte writes and 4-byte reads of 16 KiB of LDS per wave: 1024 x
// 32768 56.1 -> 50.1 us, 2048 x 2000 11.3 -> 9.1, 4096 x 4096 27.2 -> 22.7.
// line_ptr(l): the wave's l-th line (absent lines: any readable line).
template <int T, int NT, class LinePtr>
__device__ __forceinline__ void nat_direct_load(u32 (&d)[NT][4], LinePtr line_ptr, int lane) {
    static_assert(T >= 2 && NT % T == 0, "whole lines of at least 512 points");
    const u32 c16 = (u32)lane & 15u, g = (u32)lane >> 4;
#pragma unroll
    for (int l = 0; l < NT / T; ++l) {
        const u32* const b = line_ptr(l);
        if constexpr (T == 2) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const u32x2 v = ld_at_nt<u32x2>(b + 32 * j, 4u * (2u * c16 + 128u * g));
                d[2 * l][j] = v[0];
                d[2 * l + 1][j] = v[1];
            }
        } else if constexpr (T == 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const u32x4 v = ld_at_nt<u32x4>(b + 64 * j, 4u * (4u * c16 + 256u * g));
#pragma unroll
                for (int i = 0; i < 4; ++i) d[4 * l + i][j] = v[i];
            }
        } else if constexpr (T == 8) {
            u32 v[8][4];
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                const u32x4 q = ld_at_nt<u32x4>(b + 128 * x, 4u * (4u * (g & 1u) + 8u * c16 + 1024u * (g >> 1)));
#pragma unroll
                for (int i = 0; i < 4; ++i) v[x][i] = q[i];
            }
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int i = 0; i < 4; ++i) swap_l4(v[x][i], v[x | 4][i]);
#pragma unroll
            for (int x = 0; x < 8; ++x)
#pragma unroll
                for (int i = 0; i < 4; ++i) d[8 * l + i + 4 * (x >> 2)][x & 3] = v[x][i];
        } else {
            static_assert(T == 16 && NT == 16, "one 4096-point line per wave");
            u32 v[16][4];
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                const u32x4 q = ld_at_nt<u32x4>(b + 256 * x, 4u * (4u * g + 16u * c16));
#pragma unroll
                for (int i = 0; i < 4; ++i) v[x][i] = q[i];
            }
            transpose_gi_tile(v, d);
        }
    }
}

// ----------------------------------------------------------------------------
// k_big<W>: one signal of N = 4096*W (W = 2, 4, 8, 16) per workgroup of W
// waves, in a single HBM round trip.  Radix list [16, 16, 16, W]; position
// p = d0 + 16*d1 + 256*d2 + 4096*w, wave w loads chunk w.
//  phase 1: each wave does the 4096-point DIT of its chunk in registers and
//           multiplies by the final-stage twiddle W_N^{w*c}, c = k0+16k1+256k2:
//           W_N^{256*w*k2} is folded into the stage-2 operand (row scale),
//           W_N^{w*(k0+16k1)} is a per-lane recurrence over the tiles.
//  phase 2: LDS exchange (layout [w][sigma(c)], b128 both ways) and the
//           radix-W stage over w (MFMA for W = 16, VALU for W = 2, 4, 8);
//           output position c + 4096*k3.  Two rounds of 2048 columns for
//           W >= 8 keep the exchange at W*8 KiB of LDS.
// sigma(c) = c ^ ((c >> 4) & 15) << 2 is a bijection that keeps 16-lane
// groups conflict-free both for writers (lane%16 = c bits 4-7) and for
// readers (lane%16 = c bits 2-5); readers own 4 adjacent columns per lane so
// the final global stores are 256-byte runs per 16 lanes.
__device__ __forceinline__ u32 lds_sigma(u32 c) { return c ^ (((c >> 4) & 15u) << 2); }

template <int W, int ROUNDS_ = (W >= 8 ? 2 : 1)>
struct BigCfg {
    static constexpr int ROUNDS = ROUNDS_;
    static constexpr int COLS = 4096 / ROUNDS;  // columns exchanged per round
    static constexpr int LDS_WORDS = W * COLS;
    static constexpr u32 N = 4096u * W;
};

// Twiddle-table values of the per-line phase, loaded before the data (global
// loads complete in issue order, so values loaded after the data would hold
// the first stage until the whole signal has arrived).
//   Phase-1 twiddle W_N^{w*c} = W_Q^{c*e} with root W_Q and exponent e:
//     no epilogue: Q = N, e = w;
//     epilogue (W = 16, next pass of radix R = 2^r at step N over chunks
//     j = sig mod R): the next pass's twiddle W_{NR}^{(c + 4096k)*rev(j)}
//     splits into W_{NR}^{c*rev(j)}, merged here as Q = N*R,
//     e = w*R + rev(j), and W_{NR}^{4096*k*rev(j)}, a row scale of the
//     final-stage operand (output frequency k).
//   rec0: W_Q^{e*(k0 + 16*k1)} (k0 = 4g + i, k1 = lane%16), constant over
//         k2 for c = k0 + 16*k1 + 256*k2, merged into the stage-1 recurrence;
//   s2:   W_Q^{e*256*k2} as a row scale of the stage-2 operand (f = k2);
//   s3:   the final-stage row scale under the epilogue.
struct RawQ {
    float2 h, l;  // W_Q^m = h * l (two-level table entries)
};

struct BigTw {
    Dit4096Tw tw;
    RawQ rec0[4], s2, s3;
};

template <int W, bool EPI>
__device__ __forceinline__ void big_tw_load(BigTw& bt, int lane, int w, u32 sig, const float2* __restrict__ w4096,
                                            const float2* __restrict__ wn_hi, const float2* __restrict__ wn_lo,
                                            u32 wn_lo_bits, const EpiParams& epi) {
    static_assert(!EPI || W == 16, "the epilogue twiddle is folded for W = 16 only");
    const int c16 = lane & 15, g = lane >> 4;
    u32 e_w = (u32)w, rj = 0u;
    if constexpr (EPI) {
        rj = epi_rev(epi, sig);
        e_w = ((u32)w << epi.r_log2) + rj;
    }
    const float2* q_hi = EPI ? epi.hi : wn_hi;
    const float2* q_lo = EPI ? epi.lo : wn_lo;
    const u32 q_bits = EPI ? epi.lo_bits : wn_lo_bits;
    const u32 q_mask = EPI ? epi.m_mask : 4096u * W - 1u;
    auto wq_load = [&](u32 m) -> RawQ {
        m &= q_mask;
        return RawQ{q_hi[m >> q_bits], q_lo[m & ((1u << q_bits) - 1u)]};
    };
    dit4096_tw_load(bt.tw, lane, w4096);
#pragma unroll
    for (int i = 0; i < 4; ++i) bt.rec0[i] = wq_load(e_w * (4u * g + i + 16u * c16));
    bt.s2 = wq_load(256u * e_w * (u32)c16);
    bt.s3 = wq_load(4096u * rj * (u32)c16);
}

// The phase-1 values of a single line with exponent e (twiddle W_Q^{c*e}) from
// the two-level table of W_Q: what big_tw_load gives wave w of chunk j under
// the epilogue for e = w*R + rev(j).
__device__ __forceinline__ void line_tw_load(BigTw& bt, int lane, u32 e, const float2* __restrict__ w4096,
                                             const float2* __restrict__ q_hi, const float2* __restrict__ q_lo,
                                             u32 q_bits, u32 q_mask) {
    const int c16 = lane & 15, g = lane >> 4;
    auto wq_load = [&](u32 m) -> RawQ {
        m &= q_mask;
        return RawQ{q_hi[m >> q_bits], q_lo[m & ((1u << q_bits) - 1u)]};
    };
    dit4096_tw_load(bt.tw, lane, w4096);
#pragma unroll
    for (int i = 0; i < 4; ++i) bt.rec0[i] = wq_load(e * (4u * g + i + 16u * c16));
    bt.s2 = wq_load(256u * e * (u32)c16);
}

template <int SIGN>
__device__ __forceinline__ cf raw_q(const RawQ& r) {
    constexpr float sg = SIGN < 0 ? 1.f : -1.f;
    return cmul(cf{r.h.x, sg * r.h.y}, cf{r.l.x, sg * r.l.y});
}

// Phase 1: the in-wave 4096-point DIT of this wave's line d (the digit-
// reversed chunk 4096*w .. 4096*w + 4095 of the signal, loaded as tile t =
// d2, lane (c16 = d1, g), word j = d0), times W_N^{w*c}; the result is left
// in e with (g,i) = k0, tile = k2, lane%16 = k1, c = k0 + 16*k1 + 256*k2.
// With scale != 1 every result is also multiplied by scale, at no cost: the
// factor rides on the start of the stage-1 recurrence, which multiplies
// every point of the line once (in FP32, before the rounding to fp16).
template <int SIGN>
__device__ __forceinline__ void big_phase1(u32 (&d)[16][4], u32 (&e)[16][4], const BigTw& bt, const Dft16Op& op,
                                           float scale = 1.f) {
    cf rec0[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        rec0[i] = raw_q<SIGN>(bt.rec0[i]);
        rec0[i] = cf{rec0[i].x * scale, rec0[i].y * scale};
    }
    const cf s2 = raw_q<SIGN>(bt.s2);
    auto make_op2 = [&] { return make_dft16_scaled(lane_id(), SIGN, s2); };
    dit4096<true>(d, SIGN, bt.tw, op, make_op2, rec0, [](int, int, cf v) -> cf { return v; });
    transpose_gi_tile(d, e);
}

// Phase 2: LDS exchange of the W lines (layout [w][sigma(c)]) and the
// radix-W stage over w, storing X[c + 4096*k3] at sbase (4 adjacent columns
// per lane).  With SCALE the FP32 results are multiplied by `scale` first.
// The stores are non-temporal, or with CACHED cached, for a pass whose
// output the next pass reads back from the MALL (a template parameter: the
// compiler merges a runtime choice between the two into one cached store).
// Every barrier is a workgroup barrier: all groups of a workgroup run the
// same sequence.
template <int W, int ROUNDS, bool EPI, int SIGN, bool SCALE = false, bool CACHED = false>
__device__ __forceinline__ void big_phase2(u32 (&e)[16][4], int w, u32* lds, u32* __restrict__ sbase,
                                           const BigTw& bt, const Dft16Op& op, bool active, float scale = 1.f) {
    static_assert(!SCALE || W < 16, "output scaling is implemented for the VALU radix-W stage");
    constexpr int sign = SIGN;
    using C = BigCfg<W, ROUNDS>;
    const int lane = lane_id();
    const int c16 = lane & 15, g = lane >> 4;
    // final-stage operand (W = 16): rows k scaled by W_Q^{4096*k*rev(j)} under
    // the epilogue; built after the first exchange barrier (a fresh lane id)
    // so that it does not hold registers during the in-wave DIT
    Dft16Op op3 = op;

#pragma unroll
    for (int r = 0; r < C::ROUNDS; ++r) {
        constexpr int TPR = 16 / C::ROUNDS;  // tiles per round
        if (r) __syncthreads();              // previous round's reads are done
#pragma unroll
        for (int tt = 0; tt < TPR; ++tt) {
            const u32 off = (u32)w * C::COLS + lds_sigma(4u * g + 16u * c16 + 256u * tt);
            store4(lds + off, e[r * TPR + tt]);
        }
        __syncthreads();
        if constexpr (EPI) {
            if (r == 0) op3 = make_dft16_scaled(lane_id(), sign, raw_q<SIGN>(bt.s3));
        }
        if constexpr (W == 16) {
            // reader wave w': columns c = j + 4*c16 + 64h + 128w' (+2048r)
            u32 v[2][4][4];  // [h][i = point (w = 4g+i)][j]
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const u32 off = (u32)(4 * g + i) * C::COLS + lds_sigma(4u * c16 + 64u * h + 128u * w);
                    load4(v[h][i], lds + off);
                }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32 o[4][4];  // [j][i' = k3 word]
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    u32 a[4] = {v[h][0][j], v[h][1][j], v[h][2][j], v[h][3][j]};
                    f32x4 re, im;
                    dft16_b(a, op3, re, im);
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[j][i] = pack(cf{re[i], im[i]});
                }
                const u32 c0 = 2048u * r + 4u * c16 + 64u * h + 128u * w;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    u32 q[4] = {o[0][i], o[1][i], o[2][i], o[3][i]};
                    if (active) {
                        if constexpr (CACHED)
                            store4(sbase + c0 + 4096u * (4u * g + i), q);
                        else
                            store4_nt(sbase + c0 + 4096u * (4u * g + i), q);
                    }
                }
            }
        } else {
            // reader wave w': columns c = j + 4*lane + 256*(q + QN*w') (+2048r)
            constexpr int QN = C::COLS / (256 * W);
#pragma unroll
            for (int q = 0; q < QN; ++q) {
                u32 v[W][4];
#pragma unroll
                for (int s = 0; s < W; ++s)
                    load4(v[s], lds + (u32)s * C::COLS + lds_sigma(4u * lane + 256u * (q + QN * w)));
                u32 o[W][4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (W == 2 && !SCALE) {
                        // radix 2 on the packed words: one packed fp16 add
                        // and subtract, each correctly rounded
                        o[0][j] = hadd2(v[0][j], v[1][j]);
                        o[1][j] = hsub2(v[0][j], v[1][j]);
                    } else {
                        u32 xw[W];
#pragma unroll
                        for (int s = 0; s < W; ++s) xw[s] = v[s][j];
                        cf x[W];
                        small_dft_words<W>(xw, x, sign);
#pragma unroll
                        for (int s = 0; s < W; ++s)
                            o[s][j] = SCALE ? pack(x[s].x * scale, x[s].y * scale) : pack(x[s]);
                    }
                }
                const u32 c0 = 2048u * r + 4u * lane + 256u * (q + QN * w);
#pragma unroll
                for (int s = 0; s < W; ++s)
                    if (active) {
                        if constexpr (CACHED)
                            store4(sbase + c0 + 4096u * s, o[s]);
                        else
                            store4_nt(sbase + c0 + 4096u * s, o[s]);
                    }
            }
        }
    }
}

// big_phase2 for W = 2, 4, 8 that keeps the results in registers instead of
// storing them: o[(r*QN + q)*W + s] holds the four words of positions
// 2048r + 4*lane + 256*(q + QN*w) + 4096*s + (0..3) (the words big_phase2
// stores there).  The caller synchronises before reusing the LDS.
template <int W, int ROUNDS, int SIGN>
__device__ __forceinline__ void big_phase2_regs(u32 (&e)[16][4], int w, u32* lds, u32 (&o)[16][4]) {
    static_assert(W >= 2 && W <= 8, "VALU radix-W stage");
    using C = BigCfg<W, ROUNDS>;
    constexpr int QN = C::COLS / (256 * W);
    static_assert(ROUNDS * QN * W == 16, "one slot per output group");
    const int lane = lane_id();
    const int c16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int r = 0; r < C::ROUNDS; ++r) {
        constexpr int TPR = 16 / C::ROUNDS;
        if (r) __syncthreads();
#pragma unroll
        for (int tt = 0; tt < TPR; ++tt) {
            const u32 off = (u32)w * C::COLS + lds_sigma(4u * g + 16u * c16 + 256u * tt);
            store4(lds + off, e[r * TPR + tt]);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < QN; ++q) {
            u32 v[W][4];
#pragma unroll
            for (int s = 0; s < W; ++s)
                load4(v[s], lds + (u32)s * C::COLS + lds_sigma(4u * lane + 256u * (q + QN * w)));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                u32 xw[W];
#pragma unroll
                for (int s = 0; s < W; ++s) xw[s] = v[s][j];
                cf x[W];
                small_dft_words<W>(xw, x, SIGN);
#pragma unroll
                for (int s = 0; s < W; ++s) o[(r * QN + q) * W + s][j] = pack(x[s]);
            }
        }
    }
}

// Natural-order input of the single-pass kernels: one signal of N = 4096*W
// as W columns (index mod W = d3, the line of wave w) of 4096 rows rho = d2 +
// 16*d1 + 256*d0, loaded with contiguous 16-byte accesses, through LDS once
// (W = 16: in two rounds of 128 KiB) into the register layout of big_body.
// LDS is column-major in quads of four rows, so that a reader takes four
// adjacent d2 with one 16-byte access: 16 reads per lane, where 4-byte reads
// of a row-major image took 64 (128 half-masked ones at W = 16).  The writers
// scatter words (W = 2: pairs of rows), which move the same bytes.
// Quad of (column c, row quad q): bits 0-1 ^= bits 4-5, and, for W >= 4, the
// column's bits (W = 16: c/4) from bit 3 down: the 64 words of a write fall on
// 64 banks (also those of 64 adjacent indices, W = 2 excepted, whose pair of
// columns then shares one address computation), each 16 lanes of a read on 16
// different quads.
template <int W>
__device__ __forceinline__ u32 nat_quad(u32 q, u32 c) {
    return q ^ ((q >> 4) & 3u) ^ (W == 2 ? 0u : W == 4 ? c << 2 : W == 8 ? c << 1 : (c >> 2) << 2);
}
// LDS word of natural index m of a signal of W < 16 columns.
template <int W>
__device__ __forceinline__ u32 nat_big_word(u32 m) {
    const u32 c = m % W, rho = m / W;
    return 4096u * c + 4u * nat_quad<W>(rho >> 2, c) + (rho & 3u);
}

// The line of wave w from there, in the register layout of big_body.
template <int W>
__device__ __forceinline__ void big_nat_read(u32 (&d)[16][4], u32 w, const u32* lds, int lane) {
    const u32 c16 = (u32)lane & 15u, g = (u32)lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            u32 r[4];
            load4(r, lds + 4096u * w + 4u * nat_quad<W>((u32)h + 4u * (c16 + 16u * (4u * g + (u32)j)), w));
#pragma unroll
            for (int i = 0; i < 4; ++i) d[4 * h + i][j] = r[i];
        }
}

// W = 2, 4, 8; the caller synchronises before reusing the LDS.
template <int W>
__device__ __forceinline__ void big_nat_load(u32 (&d)[16][4], const u32* __restrict__ src, u32 w, u32* lds, int lane) {
    static_assert(W == 2 || W == 4 || W == 8, "whole signal in LDS");
    u32 v[16][4];
#pragma unroll
    for (int x = 0; x < 16; ++x) load4_nt(v[x], src + 4096u * w + 256u * x + 4u * (u32)lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 16; ++x) {
        // row of this lane's first word (256/W rows per load)
        const u32 rho = (4096u / W) * w + (256u / W) * x + 4u * (u32)lane / W;
        if constexpr (W == 2) {  // rows rho, rho + 1 of both columns
#pragma unroll
            for (u32 c = 0; c < 2; ++c)
                *reinterpret_cast<u32x2*>(lds + 4096u * c + 4u * nat_quad<W>(rho >> 2, c) + (rho & 3u)) =
                    u32x2{v[x][c], v[x][2 + c]};
        } else {  // four columns of row rho
            const u32 col = W == 8 ? 4u * ((u32)lane & 1u) : 0u;
#pragma unroll
            for (u32 k = 0; k < 4; ++k)
                lds[4096u * (col + k) + 4u * nat_quad<W>(rho >> 2, col + k) + (rho & 3u)] = v[x][k];
        }
    }
    __syncthreads();
    big_nat_read<W>(d, w, lds, lane);
}

// The same in two rounds through W*8 KiB, for W = 16 and for several signals
// per workgroup; row rho at src + rho*row_words (W words of it).  A round
// holds the rows with bit 9 (d0 bit 1) equal to its number, so that which
// loads it writes and which words (j >> 1) it reads is fixed at compile time.
// Every barrier is a workgroup barrier; the caller synchronises before reusing
// the LDS.
template <int W>
__device__ __forceinline__ void big_nat_load2(u32 (&d)[16][4], const u32* __restrict__ src, u32 row_words, u32 w,
                                              u32* lds, int lane) {
    // load x = 8r + xx holds 256/W rows: the low LB row bits are the lane's
    // (and, for W = 2, the word's), then xx, bit 9 = r, then the wave's bits
    constexpr u32 LB = W == 2 ? 7 : W == 4 ? 6 : W == 8 ? 5 : 4;
    const u32 L = (u32)lane, c16 = L & 15u, g = L >> 4;
    auto above = [](u32 k) { return ((k & ((1u << (9 - LB)) - 1u)) << LB) | ((k >> (9 - LB)) << 10); };
    u32 v[16][4];
#pragma unroll
    for (int x = 0; x < 16; ++x) {
        const u32 row = above((u32)(x & 7) | (w << 3)) | ((u32)(x >> 3) << 9);
        const u32x4 q = ld_at_nt<u32x4>(src + (size_t)row * row_words,
                                        W <= 4 ? 16u * L : 4u * (4u * L / W * row_words + (4u * L & (W - 1u))));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[x][i] = q[i];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        if (r) __syncthreads();  // round 0's reads are done
#pragma unroll
        for (int xx = 0; xx < 8; ++xx) {
            // row without bit 9
            const u32 k = (u32)xx | (w << 3), rho = (k << LB) | (4u * L / W);
            if constexpr (W == 2) {
#pragma unroll
                for (u32 c = 0; c < 2; ++c)
                    *reinterpret_cast<u32x2*>(lds + 2048u * c + 4u * nat_quad<W>(rho >> 2, c) + (rho & 3u)) =
                        u32x2{v[8 * r + xx][c], v[8 * r + xx][2 + c]};
            } else {
                const u32 col = 4u * L & (W - 1u);
#pragma unroll
                for (u32 i = 0; i < 4; ++i)
                    lds[2048u * (col + i) + 4u * nat_quad<W>(rho >> 2, col + i) + (rho & 3u)] = v[8 * r + xx][i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                u32 t[4];
                load4(t, lds + 2048u * w + 4u * nat_quad<W>((u32)h + 4u * (c16 + 16u * (2u * g + (u32)jj)), w));
#pragma unroll
                for (int i = 0; i < 4; ++i) d[4 * h + i][2 * r + jj] = t[i];
            }
    }
}

// One signal of N = 4096*W at sbase, processed by the W waves of a group
// (this wave is number w) with lds = the group's W*COLS words of LDS.  sig
// is the signal's index (epilogue only).
template <int W, int ROUNDS, bool EPI, int SIGN, bool CACHED = false>
__device__ __forceinline__ void big_body(u32* __restrict__ sbase, int w, u32* lds, u32 sig,
                                         const float2* __restrict__ w4096, const float2* __restrict__ wn_hi,
                                         const float2* __restrict__ wn_lo, u32 wn_lo_bits, const EpiParams& epi,
                                         bool active = true) {
    const int lane = lane_id();
    const int c16 = lane & 15, g = lane >> 4;
    BigTw bt;
    big_tw_load<W, EPI>(bt, lane, w, sig, w4096, wn_hi, wn_lo, wn_lo_bits, epi);
    __builtin_amdgcn_sched_barrier(0);
    u32 d[16][4];
    {
        const u32* src = sbase + 4096 * w + 16 * c16 + 4 * g;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            load4_nt(d[t], src + 256 * t);
            __builtin_amdgcn_sched_barrier(0);  // keep the tile order of the loads
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    const Dft16Op op = make_dft16(lane, SIGN);
    u32 e[16][4];
    big_phase1<SIGN>(d, e, bt, op);
    big_phase2<W, ROUNDS, EPI, SIGN, false, CACHED>(e, w, lds, sbase, bt, op, active);
}

}  // namespace tcfft

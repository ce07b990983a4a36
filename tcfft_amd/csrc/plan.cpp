// plan.cpp -- plan builder, pass driver and C ABI (include/tcfft.h).
//
// The reference's tcfftCreate fills a fixed size table and a kernel pointer
// table (tcfft_half.cu:1235-1345); tcfftExec launches one first-pass kernel
// then strided passes with a growing step (tcfft_half.cu:1177-1233).  Here
// the plan is computed for any power of two: a first pass over contiguous
// lines of L = min(n, 4096) (one wave per 4096 elements, all in registers),
// then strided passes of radix <= 256 in 8-bit chunks.  Each pass but the
// last multiplies its FP32 results by the twiddle of the pass that follows,
// from FP64-generated tables uploaded at plan creation.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <algorithm>
#include <functional>
#include <map>
#include <new>
#include <vector>

#include "../../include/tcfft.h"
#include "fft_kernels.hpp"
#include "plan_internal.hpp"

using tcfft::EpiParams;

namespace {

constexpr uint32_t kMagic = 0x7cff7a11u;
thread_local int g_last_hip_error = 0;

struct Pass {
    int kind = 0;          // 0: contiguous rows, 1: strided columns, 2: single-pass big lines,
                           // 3: strided columns of radix 256*W in one round trip
    int radix = 0;         // rows: T (line = 256*T); columns: R; big: W (line = 4096*W)
    uint32_t n_tiles = 0;  // rows: 256-element tiles; big: number of lines
    uint32_t s_log2 = 0;   // columns: element step
    uint32_t outer = 0;    // columns: number of [R][s] blocks
    bool has_epi = false;
    EpiParams epi{};
    uint32_t epi_M_log2 = 0;  // table size to bind at upload time
    uint32_t big_M_log2 = 0;  // big: W_L table (L = 4096*W)
    const float2* big_hi = nullptr;
    const float2* big_lo = nullptr;
};

struct Layout {  // host-only result of the plan builder
    int dims = 1;
    int n = 0, nx = 0, ny = 0, batch = 0;
    std::vector<int> rad_x, rad_y;  // 1D: rad_y holds the list
    std::vector<Pass> passes;
};

int ilog2(uint32_t v) {
    int r = 0;
    while ((1u << r) < v) ++r;
    return r;
}
bool is_pow2(long v) { return v > 0 && (v & (v - 1)) == 0; }

// Split `bits` into strided pass radices: one pass of radix 2^9..2^11
// (k_cols_big, 256*W with W = 2, 4, 8) when 9 to 11 bits remain, else
// passes of at most 2^8.
std::vector<int> split_bits(int bits) {
    if (bits >= 9 && bits <= 11) return {1 << bits};
    std::vector<int> out;
    while (bits > 0) {
        int b = bits > 8 ? 8 : bits;
        out.push_back(1 << b);
        bits -= b;
    }
    return out;
}

// DIT radix digits consumed inside one strided pass of radix R:
// [R] (R < 16), [16, R/16] (R <= 256), [16, 16, R/256] (R > 256).
void pass_digits(int R, std::vector<int>& rad) {
    if (R >= 16) {
        rad.push_back(16);
        if (R > 256) {
            rad.push_back(16);
            rad.push_back(R / 256);
        } else if (R > 16) {
            rad.push_back(R / 16);
        }
    } else {
        rad.push_back(R);
    }
}

// A strided pass of radix R: kind 3 (one round trip) above 256.
Pass strided_pass(int R, uint32_t s_log2, uint32_t outer) {
    Pass p;
    p.kind = R > 256 ? 3 : 1;
    p.radix = R;
    p.s_log2 = s_log2;
    p.outer = outer;
    return p;
}

// Epilogue description for a next pass (radix R at axis step s, shift).
void set_epi(Pass& p, uint32_t s_log2_axis, int R_next, uint32_t shift) {
    p.has_epi = true;
    p.epi.shift = shift;
    p.epi.s_log2 = s_log2_axis;
    p.epi.r_log2 = (uint32_t)ilog2((uint32_t)R_next);
    p.epi.ra_log2 = R_next >= 16 ? 4u : p.epi.r_log2;
    p.epi.rb_log2 = R_next > 256 ? 4u : p.epi.r_log2 - p.epi.ra_log2;
    p.epi_M_log2 = s_log2_axis + p.epi.r_log2;
    p.epi.m_mask = (p.epi_M_log2 >= 32) ? 0xffffffffu : ((1u << p.epi_M_log2) - 1u);
    p.epi.lo_bits = p.epi_M_log2 / 2;
}

// Passes for contiguous transforms of length n over `lines` lines.  The first
// pass covers L = min(n, 65536) contiguous elements: one wave per line for
// L <= 4096 (k_rows), one workgroup of L/4096 waves for larger L (k_big,
// a single HBM round trip).
int build_axis_rows(int n, long lines, std::vector<int>& rad, std::vector<Pass>& passes, int first_log2 = 16) {
    const int nb = ilog2((uint32_t)n);
    const int L = n < (1 << first_log2) ? n : (1 << first_log2);
    Pass first;
    rad.push_back(16);
    rad.push_back(16);
    if (L <= 4096) {
        const int T = L / 256;
        first.kind = 0;
        first.radix = T;
        first.n_tiles = (uint32_t)((long)n * lines / 256);
        if (T > 1) rad.push_back(T);
    } else {
        const int W = L / 4096;
        first.kind = 2;
        first.radix = W;
        first.n_tiles = (uint32_t)((long)n * lines / L);
        first.big_M_log2 = (uint32_t)ilog2((uint32_t)L);
        rad.push_back(16);
        rad.push_back(W);
    }
    passes.push_back(first);
    uint32_t s_log2 = (uint32_t)ilog2((uint32_t)L);
    for (int R : split_bits(nb - (int)s_log2)) {
        set_epi(passes.back(), s_log2, R, 0);
        pass_digits(R, rad);
        passes.push_back(strided_pass(R, s_log2, (uint32_t)((long)n * lines / ((long)R << s_log2))));
        s_log2 += (uint32_t)ilog2((uint32_t)R);
    }
    return 0;
}

// first_log2: length 2^first_log2 of the first (contiguous) pass when it does
// not cover the whole line.  A first pass followed by strided passes folds
// their twiddle, which the kernels implement for lines of 256..4096 points
// (k_rows) and 65536 points (k_big<16>): first_log2 in 8..12 or 16.
int build_layout_1d(int n, int batch, Layout& out, int first_log2 = 16) {
    if (!is_pow2(n) || n < 256 || n > (1 << 27)) return TCFFT_INVALID_SIZE;
    if (batch < 1 || (long)n * batch >= (1L << 31)) return TCFFT_INVALID_BATCH;
    if (!((first_log2 >= 8 && first_log2 <= 12) || first_log2 == 16)) return TCFFT_INVALID_VALUE;
    out = Layout{};
    out.dims = 1;
    out.n = n;
    out.batch = batch;
    build_axis_rows(n, batch, out.rad_y, out.passes, first_log2);
    return TCFFT_SUCCESS;
}

int build_layout_2d(int nx, int ny, int batch, Layout& out) {
    if (!is_pow2(nx) || !is_pow2(ny) || ny < 256 || ny > (1 << 16) || nx < 2 || nx > (1 << 16))
        return TCFFT_INVALID_SIZE;
    if (batch < 1 || (long)nx * ny * batch >= (1L << 31)) return TCFFT_INVALID_BATCH;
    out = Layout{};
    out.dims = 2;
    out.nx = nx;
    out.ny = ny;
    out.batch = batch;
    // rows: length ny, nx*batch lines; no twiddle between the two axes
    build_axis_rows(ny, (long)nx * batch, out.rad_y, out.passes);
    // columns: strided passes along x with memory step ny * s_x
    const uint32_t ny_log2 = (uint32_t)ilog2((uint32_t)ny);
    uint32_t sx_log2 = 0;
    bool first = true;
    for (int R : split_bits(ilog2((uint32_t)nx))) {
        if (!first) set_epi(out.passes.back(), sx_log2, R, ny_log2);
        first = false;
        pass_digits(R, out.rad_x);
        out.passes.push_back(
            strided_pass(R, ny_log2 + sx_log2, (uint32_t)((long)nx * batch / ((long)R << sx_log2))));
        sx_log2 += (uint32_t)ilog2((uint32_t)R);
    }
    return TCFFT_SUCCESS;
}

}  // namespace

struct tcfft_plan_s {
    uint32_t magic = kMagic;
    Layout lay;
    int device = 0;
    float2* w4096 = nullptr;
    std::map<uint32_t, std::pair<float2*, float2*>> epi_tables;  // M_log2 -> (hi, lo)
    std::vector<void*> allocs;
    // Staging copy of the input for in-place tcfft_exec_natural on layouts
    // whose first pass cannot read its input in place (see
    // natural_needs_stage); allocated with the plan so that no exec call
    // allocates.  One per plan: in-place natural-order calls on one plan
    // must not overlap.
    void* workspace = nullptr;
    // 2D: output line of input row x for the natural-order row pass (nx
    // words, the digit reversal over the x radices in reverse order)
    uint32_t* xpos = nullptr;
    size_t workspace_bytes = 0;
    size_t total = 0;  // elements in the buffer
    // signals per pass pair in tcfft_exec_split, 0 = the whole batch (2^16 x
    // 256: 99.6 us whole against 112.9 us in chunks of 128 on one box)
    int split_chunk = 0;
    int cus = 0;          // compute units of the plan's device
    int big_delay = -1;   // start schedule of the first-pass kernels: -1 = default
    int big_groups = 3;
    // waves per workgroup of the contiguous-row passes (1, 2, 4; 0 = by the
    // pass, see rows_wg); one-wave workgroups measured fastest for one round
    // of waves (4096 x 1024: 7.2 us against 8.1 with 4, 1024-point rows of
    // 2D 1024^2 x 8: 14.7 against 15.1)
    int rows_waves = 0;
    int rows_tiles = 0;  // tiles per wave of a row first pass (rows_nt; 0 = by the grid)
    // The schedule options as the caller set them.  The tuner, which times
    // tcfft_exec, changes only the fields above: the natural-order row passes
    // and k_lines_nat have other optima (256 x 16384: 8 tiles win the drop-in
    // call, 8.0 us against 8.7 with 4; natural order 10.8 with 8, 9.5 with 4)
    struct {
        int delay = -1, groups = 3, waves = 0, tiles = 0;
    } set;
    int cols_delay = 1;   // start delay of the radix-256*W column pass (3 groups; 2D 1024^2 x 8: 36.0 -> 33.8 us)
    int split_delay = 2;  // start delay of the split-precision passes (3 groups; 2^16 x 256: 110.6 -> 106.6 us)
    // first pass's output stores of a multi-pass plan: -1 = cached while the
    // buffer is at most 256 MiB (cached_out), 0 = non-temporal, 1 = cached
    int first_cached = -1;
    // batch chunk of a multi-pass transform larger than the MALL, in MiB
    // (chunk_signals; 0 = the whole batch at once)
    int mall_chunk_mib = 256;
    // Split precision at every size (tcfft_plan_prepare_split): the column
    // passes in order, and a workspace of total * 8 bytes (FP32 complex)
    // for the passes whose transposed store cannot go in place.
    struct SplitStep {
        int R;
        int row_tiles;     // > 0: one pass over contiguous lines of 256*row_tiles points (k_split_rows), a.units lines
        bool row;          // Qlo = 1 (transposed row store)
        bool transposing;  // not the last pass of its axis: src != dst
        tcfft::SplitPassArgs a;
    };
    std::vector<SplitStep> split_steps;
    bool split_ready = false;
    float2* split_ws = nullptr;
    int real_n = 0;       // real-input plan: the real length (its complex layout has n = real_n / 2)
    float2* w_real = nullptr;  // W_{real_n}^0..64 (n <= 8192) or ^0..64W (n = 8192 W <= 65536)
    std::pair<float2*, float2*> w_real_pair{};  // n > 65536: two-level table of W_n
    uint32_t* real_ws = nullptr;                // n > 65536: the n/2-point spectrum between the two steps
};

namespace {

int hip_fail(hipError_t e) {
    g_last_hip_error = (int)e;
    return TCFFT_HIP_ERROR;
}

// exp(-2*pi*i*k/M) for k in [k0, k0 + count) with stride `step`, computed in
// FP64 and rounded to FP32.
std::vector<float2> host_table(uint32_t M_log2, uint64_t step, uint32_t count) {
    std::vector<float2> t(count);
    const double M = std::ldexp(1.0, (int)M_log2);
    for (uint32_t k = 0; k < count; ++k) {
        const double a = 2.0 * M_PI * (double)((uint64_t)k * step) / M;
        t[k] = make_float2((float)std::cos(a), (float)-std::sin(a));
    }
    return t;
}

int upload(tcfft_plan_s* p, const std::vector<float2>& h, float2** dst) {
    void* d = nullptr;
    hipError_t e = hipMalloc(&d, h.size() * sizeof(float2));
    if (e != hipSuccess) return hip_fail(e);
    p->allocs.push_back(d);
    e = hipMemcpy(d, h.data(), h.size() * sizeof(float2), hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(e);
    *dst = (float2*)d;
    return TCFFT_SUCCESS;
}

// Position of input row x (0 <= x < nx) among the rows of a 2D natural-order
// row pass's output: the digits of x taken from the low end by the x radices
// in reverse order and reassembled most significant first (the digit
// reversal the column passes consume, as gen_rev, tcfft_doit_half_2d.cpp:40-50).
uint32_t xpos_of(uint32_t x, const std::vector<int>& rad_x) {
    uint32_t idx = 0, rest = x;
    std::vector<uint32_t> digits;
    for (auto it = rad_x.rbegin(); it != rad_x.rend(); ++it) {
        digits.push_back(rest % (uint32_t)*it);
        rest /= (uint32_t)*it;
    }
    size_t i = 0;
    for (auto it = rad_x.rbegin(); it != rad_x.rend(); ++it, ++i) idx = idx * (uint32_t)*it + digits[i];
    return idx;
}

int upload_xpos(tcfft_plan_s* p) {
    const uint32_t nx = (uint32_t)p->lay.nx;
    std::vector<uint32_t> h(nx);
    for (uint32_t x = 0; x < nx; ++x) h[x] = xpos_of(x, p->lay.rad_x);
    void* d = nullptr;
    hipError_t e = hipMalloc(&d, nx * sizeof(uint32_t));
    if (e != hipSuccess) return hip_fail(e);
    p->allocs.push_back(d);
    e = hipMemcpy(d, h.data(), nx * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(e);
    p->xpos = (uint32_t*)d;
    return TCFFT_SUCCESS;
}

void free_plan(tcfft_plan_s* p) {
    for (void* a : p->allocs) (void)hipFree(a);
    p->magic = 0;
    delete p;
}

// Whether in-place tcfft_exec_natural stages a copy of its input: 2D plans
// (the first pass writes the x reversal as a permutation of whole lines, so a
// workgroup would overwrite lines others have not read yet) and 1D plans
// whose first pass does not read natural order itself (the reversal pass
// before it gathers from the whole line).
bool natural_needs_stage(const Layout& L) {
    const Pass& f = L.passes[0];
    const bool fused = (f.kind == 0 || f.kind == 2) && !f.has_epi;
    return L.dims == 2 || !fused;
}

// Two-level table of W_M, M = 2^M_log2: hi[k] = W_M^{k*2^lo}, lo[k] = W_M^k,
// lo = floor(M_log2 / 2) (the split every kernel uses).
int table_pair(tcfft_plan_s* p, uint32_t M, std::pair<float2*, float2*>& out) {
    auto it = p->epi_tables.find(M);
    if (it == p->epi_tables.end()) {
        const uint32_t lo = M / 2;
        float2 *hi_d = nullptr, *lo_d = nullptr;
        int rc = upload(p, host_table(M, 1ull << lo, 1u << (M - lo)), &hi_d);
        if (rc) return rc;
        rc = upload(p, host_table(M, 1, 1u << lo), &lo_d);
        if (rc) return rc;
        it = p->epi_tables.emplace(M, std::make_pair(hi_d, lo_d)).first;
    }
    out = it->second;
    return TCFFT_SUCCESS;
}

// Split-precision passes for the M-point DFTs along the first index of
// `signals` arrays [M][L] (M = 2^m_log2, L = 2^l_log2): one pass of radix M
// when L >= 16 and M <= 256 (radix 2..8 on VALU), else ceil(m_log2 / 8)
// passes (at least two when L = 1, whose first pass needs >= 16 columns) of
// 4..8 bits, balanced.  Pass i sees R_i rows by Q = M*L/R_i columns with
// Qlo = L * R_0 * ... * R_{i-1}, and all but the last take the twiddle of
// the remaining M' = M / (R_0 ... R_{i-1}) points.
int split_axis(int m_log2, int l_log2, uint32_t signals, std::vector<tcfft_plan_s::SplitStep>& out) {
    std::vector<int> bits;
    if (m_log2 <= 3) {
        if (l_log2 < 4 || m_log2 < 1) return TCFFT_INVALID_SIZE;
        bits.push_back(m_log2);
    } else {
        int passes = (m_log2 + 7) / 8;
        if (l_log2 == 0 && passes < 2) passes = 2;
        for (int i = 0; i < passes; ++i) bits.push_back((m_log2 + i) / passes);
        for (int b : bits)
            if (b < 4 || b > 8) return TCFFT_INVALID_SIZE;
    }
    int done = 0;
    for (size_t i = 0; i < bits.size(); ++i) {
        const int b = bits[i];
        const int cur_l = l_log2 + done, cur_m = m_log2 - done;
        tcfft_plan_s::SplitStep s{};
        s.R = 1 << b;
        s.row = cur_l == 0;
        s.transposing = cur_m > b;
        s.a.q_log2 = (uint32_t)(m_log2 + l_log2 - b);
        s.a.qlo_log2 = (uint32_t)cur_l;
        s.a.units = signals << (s.a.q_log2 - 4);
        if (s.transposing) {
            s.a.m_mask = (1u << cur_m) - 1u;
            s.a.lo_bits = (uint32_t)cur_m / 2u;  // the split of table_pair
        }
        out.push_back(s);
        done += b;
    }
    return TCFFT_SUCCESS;
}

// The split-precision pass list of a shape (host only): 1D n (ny = 0) or 2D
// nx x ny, batch signals; n = 65536 has none (its own two-pass kernel).
int split_steps_of(int dims, int n_or_nx, int ny, int batch, std::vector<tcfft_plan_s::SplitStep>& steps) {
    if (dims == 1) return n_or_nx == 65536 ? TCFFT_SUCCESS : split_axis(ilog2((uint32_t)n_or_nx), 0, (uint32_t)batch, steps);
    // rows: the contiguous ny axis of every one of the nx lines; then the nx
    // axis with the ny columns of each image
    const int rc = split_axis(ilog2((uint32_t)ny), 0, (uint32_t)batch * (uint32_t)n_or_nx, steps);
    return rc ? rc : split_axis(ilog2((uint32_t)n_or_nx), ilog2((uint32_t)ny), (uint32_t)batch, steps);
}

// The passes tcfft_exec_split runs for that list.  Fewer round trips where a
// kernel holds more than a pass of the list:
//   a contiguous axis of 256..4096 points: whole lines (k_split_rows);
//   1D 2^17..2^22 points: two passes of radix 256..2048 instead of three;
//   a strided axis of 512..2048 points: one pass (k_split_colsw), at every
//   grid: whole calls with the list's two passes there / with one, 512 x 256 x 1
//   34.0 / 13.1 us, x 16 40.9 / 22.4, 1024 x 256 x 1 30.8 / 15.8, 2048 x 256 x 1 31.6 /
//   22.6, x 4 40.9 / 29.0, 2048 x 1024 x 4 80.2 / 57.7 (both without a start delay).
int split_exec_steps_of(int dims, int n_or_nx, int ny, int batch, std::vector<tcfft_plan_s::SplitStep>& steps) {
    std::vector<tcfft_plan_s::SplitStep> list;
    const int rc = split_steps_of(dims, n_or_nx, ny, batch, list);
    if (rc) return rc;
    const int line = dims == 1 ? n_or_nx : ny;
    const uint32_t lines = (uint32_t)batch * (dims == 1 ? 1u : (uint32_t)n_or_nx);
    size_t i = 0;
    while (i < list.size() && list[i].transposing) ++i;  // an axis's passes end with the first one without a twiddle
    ++i;
    tcfft_plan_s::SplitStep s{};
    if (line <= 4096) {
        s.R = line;
        s.row_tiles = line / 256;
        s.a.units = lines;
        steps.push_back(s);
    } else if (dims == 1 && line >= (1 << 17) && line <= (1 << 22)) {
        const int m = ilog2((uint32_t)line), b = m == 17 ? 9 : m / 2;  // R = 2^b rows, then 2^(m-b)
        s.R = 1 << b;
        s.row = s.transposing = true;
        s.a.q_log2 = (uint32_t)(m - b);
        s.a.units = lines << (s.a.q_log2 - 4);
        s.a.m_mask = (uint32_t)line - 1u;
        s.a.lo_bits = (uint32_t)m / 2u;  // the split of table_pair
        steps.push_back(s);
        s = {};
        s.R = 1 << (m - b);
        s.a.q_log2 = s.a.qlo_log2 = (uint32_t)b;
        s.a.units = lines << (b - 4);
        steps.push_back(s);
    } else {
        steps.insert(steps.end(), list.begin(), list.begin() + (long)std::min(i, list.size()));
    }
    if (dims == 2 && n_or_nx >= 512 && n_or_nx <= 2048) {
        s = {};
        s.R = n_or_nx;
        s.a.q_log2 = s.a.qlo_log2 = (uint32_t)ilog2((uint32_t)ny);
        s.a.units = (uint32_t)batch << (s.a.q_log2 - 4);
        steps.push_back(s);
    } else if (dims == 2) {
        steps.insert(steps.end(), list.begin() + (long)i, list.end());
    }
    return TCFFT_SUCCESS;
}

int finish_plan(tcfft_plan_s* p) {
    hipError_t e = hipGetDevice(&p->device);
    if (e != hipSuccess) return hip_fail(e);
    e = hipDeviceGetAttribute(&p->cus, hipDeviceAttributeMultiprocessorCount, p->device);
    if (e != hipSuccess) return hip_fail(e);
    int rc = upload(p, host_table(12, 1, 4096), &p->w4096);
    if (rc) return rc;
    for (Pass& ps : p->lay.passes) {
        if (ps.kind == 2) {
            std::pair<float2*, float2*> t;
            rc = table_pair(p, ps.big_M_log2, t);
            if (rc) return rc;
            ps.big_hi = t.first;
            ps.big_lo = t.second;
        }
        if (!ps.has_epi) continue;
        std::pair<float2*, float2*> t;
        rc = table_pair(p, ps.epi_M_log2, t);
        if (rc) return rc;
        ps.epi.hi = t.first;
        ps.epi.lo = t.second;
    }
    return TCFFT_SUCCESS;
}

// stage_ws: allocate the staging workspace of in-place natural order when
// the layout needs one (real-input plans pass false and lend their own
// workspace of the same size instead).
int create_common(tcfft_plan* plan, const Layout& lay, bool stage_ws = true) {
    tcfft_plan_s* p = new (std::nothrow) tcfft_plan_s;
    if (!p) return TCFFT_ALLOC_FAILED;
    p->lay = lay;
    p->total = lay.dims == 1 ? (size_t)lay.n * lay.batch : (size_t)lay.nx * lay.ny * lay.batch;
    int rc = finish_plan(p);
    if (!rc && lay.dims == 2) rc = upload_xpos(p);
    if (!rc && stage_ws && natural_needs_stage(lay)) {
        const hipError_t e = hipMalloc(&p->workspace, p->total * 4u);
        if (e != hipSuccess) {
            p->workspace = nullptr;
            rc = hip_fail(e);
        } else {
            p->allocs.push_back(p->workspace);
            p->workspace_bytes = p->total * 4u;
        }
    }
    if (rc) {
        free_plan(p);
        return rc;
    }
    *plan = p;
    return TCFFT_SUCCESS;
}

bool valid(tcfft_plan p) { return p && p->magic == kMagic; }

// Start schedule of the single-pass kernel of width W.  Defaults measured on
// MI355X (3 groups; 2^15 x 512: 26.2 -> 24.0 us with delay 1, 2^16 x 256:
// 28.9 -> 26.5 us with delay 2, 2^14 x 2048: 53.9 -> 50.4 us with delay 1).
// Checked again on finite data (input restored before every timed run,
// 40 graph-replayed execs, medians of 3 rounds), 2^16 x 256: 3 groups with
// delay 2 27.60 us, delay 3 27.43, 5 groups delay 1 27.46, 7 groups delay 1
// 27.66, no stagger 28.13; natural order 5 groups delay 3 37.40 us, 7 groups
// delay 2 37.11, 3 groups delay 2 38.59.
// A grid of less than one wave per SIMD has nothing to stagger (natural order,
// 8192 x 100: 8.9 us with the delay, 7.1 without; 16384 x 64 10.6 and 9.8;
// drop-in behind a copy of its input, 8192 x 128 10.6 and 8.9, 16384 x 64 11.5
// and 10.3, 32768 x 32 16.1 and 14.9, both passes of 2^20 x 2 32.0 and 30.2).
tcfft::StartSched big_sched(const tcfft_plan_s* p, int W, uint32_t lines) {
    const bool small = (uint64_t)lines * (uint32_t)W < 4u * (uint64_t)p->cus;
    const int delay = p->big_delay >= 0 ? p->big_delay : small ? 0 : (W == 4 || W == 8 ? 1 : 2);
    return tcfft::StartSched{(uint32_t)delay, (uint32_t)p->big_groups, 0u};
}

// The same for the natural-order single-pass kernel.  Its workgroups stage
// the whole signal through LDS before any compute, so the 65536-point kernel
// wants a longer stagger: with the start delay left at its default it runs 5
// groups with a delay of 3 (2^16 x 256 natural, two runs: 3 groups with
// delays 2, 3, 4, 5: 38.6-38.8, 38.2-38.4, 37.9-38.4, 37.1-37.4 us; 5 groups
// with delay 2: 37.5-37.9, delay 3: 36.7-37.1; 7 groups with delay 2:
// 36.8-37.0); for W = 2, 4, 8 the drop-in defaults stay within 2% of the best.
tcfft::StartSched nat_big_sched(const tcfft_plan_s* p, int W, uint32_t lines) {
    const tcfft::StartSched s = big_sched(p, W, lines);
    if (p->big_delay >= 0 || W != 16 || s.delay == 0) return s;
    return tcfft::StartSched{3u, 5u, 0u};
}

// Start schedule of the contiguous-row first pass.  By default a delay of 1
// only when the grid is at most one 4-wave workgroup per CU (4096 x 1024:
// 10.0 -> 9.2 us); with more workgroups per CU they desynchronise by
// themselves and a delay only costs time (1024 x 8192: 15.9 -> 16.2 us).
// Waves per workgroup of a contiguous-row first pass: the plan's `setting`, or
// by default 4 for 4096-point lines over at least 32 waves per CU and 1
// otherwise.  Measured (rotated buffers): 4096 x 1024 7.7 us with one wave
// against 8.6 with four; even at 2048-4096 lines; four ahead from 8192
// lines (47.7 against 48.6 us) to 65536 (352 against 369 us); for 2048-point
// and shorter lines one wave stays ahead at every batch (2048 x 131072: 369
// against 403 us).
uint32_t rows_wg(const tcfft_plan_s* p, const Pass& ps, int setting) {
    if (setting > 0) return (uint32_t)setting;
    const uint32_t waves = (ps.n_tiles + 15u) / 16u;
    return ps.radix == 16 && waves >= 32u * (uint32_t)p->cus ? 4u : 1u;
}

// Tiles (of 256 points) per wave of a contiguous-row first pass: 16 for
// passes with an epilogue; for 4096-point lines the plan's setting, or by
// default 4 (four waves per line, k_rows_half) up to one line per CU, 8
// (two waves) up to four lines per CU, and 16 above (random input, input
// restored before every timed run, one / two / four waves per line: 4096 x
// 256 6.55 / 5.39 / 5.31 us, 4096 x 1024 7.8-8.1 / 7.35 / 9.3, 4096 x 2048
// 13.9 / 14.2 / 16.0, 4096 x 4096 26.4 / 25.9 / 27.5; 2D 256 x 4096 x 8,
// 2048 lines, 27.9 / 28.8 on inf/NaN data); otherwise the plan's setting,
// or by default the largest of 16, 8, 4 (at least the line's tiles) that
// still gives every SIMD two waves, so that a small grid spreads over the
// chip.  Measured (random input; 16 / 8 / 4 tiles): 1024 x 1024 6.17 / 5.23
// / 4.86 us, 256 x 1024 4.59 / 3.75 / 3.37, 1024 x 4096 9.68 / 9.00 / 10.27,
// 256 x 16384 9.02 / 8.04 / 8.68; at two waves per SIMD or more, 16 (2D
// 1024^2 x 8 31.3 us against 34.0 at 8 and 36.0 at 4; 1024 x 8192 14.2
// against 16.7 and 18.3).
uint32_t rows_nt(const tcfft_plan_s* p, const Pass& ps, int setting) {
    const uint32_t T = (uint32_t)ps.radix;
    if (ps.has_epi) return 16u;
    if (T >= 16) {
        if (setting > 0) return (uint32_t)setting;
        const uint32_t lines = ps.n_tiles / 16u, cus = (uint32_t)p->cus;
        return lines <= cus ? 4u : lines <= 4u * cus ? 8u : 16u;
    }
    const uint32_t lo = T <= 4 ? 4u : 8u;
    if (setting > 0) return std::max((uint32_t)setting, lo);
    const uint32_t want = 8u * (uint32_t)p->cus;  // two waves per SIMD
    for (uint32_t nt = 16u; nt > lo; nt /= 2)
        if ((ps.n_tiles + nt - 1u) / nt >= want) return nt;
    return lo;
}

// The same for the natural-order pass.  4096-point lines: four waves per line
// up to two lines per CU, two above (out of place, random input; one / two /
// four waves per line: 4096 x 256 5.9 / 4.9 / 4.8 us, 4096 x 512 6.7 / 6.5 /
// 5.8, 4096 x 1024 9.0 / 7.7 / 8.0, 4096 x 2048 13.2 / 12.0 / 13.8, 4096 x
// 4096 27.0 / 22.8 / 23.9, 4096 x 16384 96 / 93 / 110).  2D lines go to
// permuted places: one wave per line from 6 to below 16 lines per CU (whole
// transforms, one / two waves: 16 x 4096 x 96 22.9 / 23.4 us, x 128 27.6 / 28.9,
// x 192 36.6 / 39.3, x 256 48.7 / 48.2, x 384 69.7 / 68.7; 1024 x 4096 x 2 31.9 /
// 33.3, x 3 39.9 / 43.7), except for nx = 128..512, where two stay ahead (128 x
// 4096 x 16 28.4 / 26.7, 256 x 4096 x 16 51.2 / 48.2, 512 x 4096 x 4 32.8 /
// 30.6; the same at nx = 2..64 and at 1024, 2048; why these three differ was not
// found).  256-point lines: 16 or 4, never 8 (256 x 16384 9.4 us with 4, 10.5
// with 8; 256 x 65536 26.9 with 4, 35 with 8, 26.8 with 16).  Else as rows_nt
// (1024 x 1024 5.6 / 4.4 / 4.2 us with 16 / 8 / 4 tiles, 1024 x 4096 9.3 / 8.4 /
// 9.7, 1024 x 16384 25.7 / 25.7 / 28.8).
uint32_t rows_nt_nat(const tcfft_plan_s* p, const Pass& ps) {
    if (ps.radix < 16) {
        const uint32_t nt = rows_nt(p, ps, p->set.tiles);
        return ps.radix == 1 && nt == 8u && !p->set.tiles ? 4u : nt;
    }
    if (p->set.tiles > 0) return (uint32_t)p->set.tiles;
    const uint32_t lines = ps.n_tiles / 16u, cus = (uint32_t)p->cus;
    const bool mid_nx = p->lay.nx >= 128 && p->lay.nx <= 512;
    if (p->lay.dims == 2 && !mid_nx && lines >= 6u * cus && lines < 16u * cus) return 16u;
    return lines <= 2u * cus ? 4u : 8u;
}

// Waves per workgroup of the natural-order pass: as rows_wg, but four for 2D
// rows that fill the chip, whose stores go to permuted lines (2D 1024 x 1024
// x 8 29.4 us against 30.7 with one; 1D 1024 x 16384 26.7 against 26.1).
uint32_t rows_wg_nat(const tcfft_plan_s* p, const Pass& ps) {
    if (p->set.waves > 0) return (uint32_t)p->set.waves;
    return p->lay.dims == 2 && (ps.n_tiles + 15u) / 16u >= 4u * (uint32_t)p->cus ? 4u : rows_wg(p, ps, 0);
}

// Start schedule of the natural-order row pass, and of k_lines_nat: the
// caller's, or none.  The row pass has no load phase of its own to stagger:
// with a delay of 1, 1024 x 64 takes 3.37 us against 2.50 without, 4096 x 256
// 5.17 and 4.74, 1024 x 4096 8.8 and 8.4, 2048 x 2048 9.6 and 8.9, 2D 32 x
// 2048 x 64 16.8 and 15.9.
tcfft::StartSched nat_sched(const tcfft_plan_s* p) {
    return tcfft::StartSched{(uint32_t)std::max(p->set.delay, 0), (uint32_t)p->set.groups, 0u};
}

// Start schedule of a contiguous-row first pass run with nt tiles per wave.
tcfft::StartSched rows_sched(const tcfft_plan_s* p, const Pass& ps, uint32_t nt) {
    const uint32_t waves = (ps.n_tiles + nt - 1u) / nt;  // at most one wave per SIMD: a delay of 1
    const int delay = p->big_delay >= 0 ? p->big_delay : (waves <= 4u * (uint32_t)p->cus ? 1 : 0);
    return tcfft::StartSched{(uint32_t)delay, (uint32_t)p->big_groups, 0u};
}

// Whether pass i stores its output through the caches: only the first pass of
// a multi-pass plan (the next pass reads its output back), and by default
// only while the signals it covers (`nsig`, one batch chunk) take at most the
// 256 MiB of the MALL.  Measured per exec on random input, non-temporal ->
// cached: 2^20 x 16 (64 MiB) 56.1 -> 51.7 us, 2^21 x 16 105.8 -> 95.1,
// 2^22 x 16 (256 MiB) 202 -> 186, 2D 4096 x 4096 87.4 -> 77.4; at 2^24 x 8 in
// one piece (512 MiB) cached stores cost 5% (481 -> 504 us).  A single-pass
// plan keeps its non-temporal stores (2^16 x 256: 27.7 us, 29.5 cached).
uint32_t cached_out(const tcfft_plan_s* p, size_t i, uint32_t nsig) {
    if (i != 0 || p->lay.passes.size() < 2 || p->first_cached == 0) return 0u;
    const size_t bytes = p->total / (size_t)p->lay.batch * nsig * 4u;
    return p->first_cached == 1 || bytes <= ((size_t)256 << 20) ? 1u : 0u;
}

// Signals per batch chunk.  A multi-pass transform larger than the MALL runs
// all its passes on one chunk of at most mall_chunk_mib MiB of signals before
// the next, so that each later pass reads what the pass before has just
// written from the MALL instead of HBM.  Measured per exec on random input,
// whole batch -> chunks of 256 MiB: 2^24 x 8 491 -> 429 us, 2^17 x 2048
// 780 -> 716 us, 2^18 x 2048 1571 -> 1442 us, 2D 256 x 256 x 2048 468 -> 338
// us, 2D 4096 x 4096 x 16 1336 -> 1003 us (128 and 64 MiB chunks gained
// less).  Plans with a k_cols_big pass keep the whole batch: 2D 1024 x 1024
// x 128 and 512 x 1024 x 2048 measured 2% slower in chunks.
uint32_t chunk_signals(const tcfft_plan_s* p) {
    const Layout& L = p->lay;
    const uint32_t B = (uint32_t)L.batch;
    if (p->mall_chunk_mib == 0 || L.passes.size() < 2 || B < 2) return B;
    for (const Pass& ps : L.passes)
        if (ps.kind == 3) return B;
    const size_t lim = (size_t)p->mall_chunk_mib << 20, per = p->total / B * 4u;
    if (per * B <= lim || per > lim) return B;
    const size_t chunks = (per * B + lim - 1) / lim;
    size_t cs = (B + chunks - 1) / chunks;
    if (cs * per > lim) cs = lim / per;
    return (uint32_t)cs;
}

// The plan's passes [first, first + count) on signals [sig0, sig0 + nsig) of
// the batch (nsig = 0: the whole batch).  Every pass is uniform over the
// signals, so a chunk is the same launch with its counts scaled.
int run_passes(tcfft_plan_s* p, uint32_t* buf, int sign, hipStream_t st, size_t first = 0, size_t count = ~(size_t)0,
               uint32_t sig0 = 0, uint32_t nsig = 0) {
    const uint32_t B = (uint32_t)p->lay.batch;
    if (nsig == 0) nsig = B;
    buf += p->total / B * sig0;
    const size_t end = count > p->lay.passes.size() - first ? p->lay.passes.size() : first + count;
    for (size_t i = first; i < end; ++i) {
        Pass ps = p->lay.passes[i];
        ps.n_tiles = (uint32_t)((uint64_t)ps.n_tiles / B * nsig);
        ps.outer = (uint32_t)((uint64_t)ps.outer / B * nsig);
        const EpiParams* epi = ps.has_epi ? &ps.epi : nullptr;
        hipError_t e;
        if (ps.kind == 0) {
            const uint32_t nt = rows_nt(p, ps, p->rows_tiles);
            tcfft::StartSched sc = rows_sched(p, ps, nt);
            sc.cached_out = cached_out(p, i, nsig);
            e = tcfft::launch_rows(ps.radix, buf, ps.n_tiles, sign, p->w4096, epi, sc,
                                   rows_wg(p, ps, p->rows_waves), nt, st);
        } else if (ps.kind == 2) {
            tcfft::StartSched sc = big_sched(p, ps.radix, ps.n_tiles);
            sc.cached_out = cached_out(p, i, nsig);
            e = tcfft::launch_big(ps.radix, buf, ps.n_tiles, sign, p->w4096, ps.big_hi, ps.big_lo, ps.big_M_log2 / 2,
                                  epi, sc, st);
        } else if (ps.kind == 3) {
            e = epi ? hipErrorInvalidValue
                    : tcfft::launch_cols_big(ps.radix / 256, buf, ps.s_log2, ps.outer, sign, p->w4096,
                                             tcfft::StartSched{(uint32_t)p->cols_delay, 3u, 0u}, st);
        } else {
            e = tcfft::launch_cols(ps.radix, buf, ps.s_log2, ps.outer, sign, p->w4096, epi, st);
        }
        if (e != hipSuccess) return hip_fail(e);
    }
    return TCFFT_SUCCESS;
}

// body(sig0, nsig) over the batch chunks of chunk_signals, in order.
template <class F>
int for_chunks(const tcfft_plan_s* p, F&& body) {
    const uint32_t B = (uint32_t)p->lay.batch, cs = chunk_signals(p);
    for (uint32_t s0 = 0; s0 < B; s0 += cs) {
        const int rc = body(s0, std::min(cs, B - s0));
        if (rc) return rc;
    }
    return TCFFT_SUCCESS;
}

// The whole transform (drop-in order, in place), chunked as above.
int exec_all(tcfft_plan_s* p, uint32_t* buf, int sign, hipStream_t st) {
    return for_chunks(p, [&](uint32_t s0, uint32_t ns) { return run_passes(p, buf, sign, st, 0, ~(size_t)0, s0, ns); });
}

tcfft::RevSpec rev_spec(const std::vector<int>& rad) {
    tcfft::RevSpec s{};
    s.n_digits = (int)rad.size();
    for (size_t i = 0; i < rad.size() && i < 12; ++i) s.radix[i] = rad[i];
    return s;
}

// Tile of the LDS-tiled digit reversal for the radix list `rad` (powers of
// two): the largest a, b <= 6 whose bit sets are disjoint (see GatherTile).
bool gather_tile(const std::vector<int>& rad, tcfft::GatherTile& gt) {
    std::vector<uint32_t> pi;  // bit i of rev(p) = bit pi[i] of p
    std::vector<uint32_t> start(rad.size()), width(rad.size());
    uint32_t k = 0;
    for (size_t d = 0; d < rad.size(); ++d) {
        start[d] = k;
        width[d] = (uint32_t)ilog2((uint32_t)rad[d]);
        k += width[d];
    }
    for (size_t d = rad.size(); d-- > 0;)
        for (uint32_t b = 0; b < width[d]; ++b) pi.push_back(start[d] + b);
    if (k < 8) return false;
    uint32_t best_a = 0, best_b = 0;
    for (uint32_t a = 6; a >= 1; --a)
        for (uint32_t b = 6; b >= 1; --b) {
            bool ok = a + b <= k;
            for (uint32_t i = 0; i < b && ok; ++i) ok = pi[i] >= a;
            if (ok && a + b > best_a + best_b) {
                best_a = a;
                best_b = b;
            }
        }
    if (best_a + best_b < 8 || best_a < 2 || best_b < 2) return false;
    gt.a = best_a;
    gt.b = best_b;
    uint32_t used = (1u << best_a) - 1u;
    for (uint32_t i = 0; i < best_b; ++i) {
        gt.in_bit[i] = pi[i];
        used |= 1u << pi[i];
    }
    gt.free_mask = ((k >= 32) ? 0xffffffffu : ((1u << k) - 1u)) & ~used;
    for (uint32_t j = 0; j < best_a; ++j)
        for (uint32_t i = 0; i < k; ++i)
            if (pi[i] == j) gt.low_to_rev[j] = i;
    return true;
}

struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev) {
        int cur = 0;
        if (hipGetDevice(&cur) == hipSuccess && cur != dev && hipSetDevice(dev) == hipSuccess) prev = cur;
    }
    ~DeviceGuard() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

}  // namespace

extern "C" {

int tcfft_version(void) { return 100; }

const char* tcfft_status_string(int status) {
    switch (status) {
    case TCFFT_SUCCESS: return "TCFFT_SUCCESS";
    case TCFFT_INVALID_SIZE: return "TCFFT_INVALID_SIZE";
    case TCFFT_INVALID_BATCH: return "TCFFT_INVALID_BATCH";
    case TCFFT_INVALID_POINTER: return "TCFFT_INVALID_POINTER";
    case TCFFT_INVALID_PLAN: return "TCFFT_INVALID_PLAN";
    case TCFFT_INVALID_VALUE: return "TCFFT_INVALID_VALUE";
    case TCFFT_HIP_ERROR: return "TCFFT_HIP_ERROR";
    case TCFFT_ALLOC_FAILED: return "TCFFT_ALLOC_FAILED";
    default: return "TCFFT_UNKNOWN_STATUS";
    }
}

int tcfft_last_hip_error(void) { return g_last_hip_error; }

int tcfft_plan_create_1d(tcfft_plan* plan, int n, int n_batch) {
    if (!plan) return TCFFT_INVALID_POINTER;
    *plan = nullptr;
    Layout lay;
    int rc = build_layout_1d(n, n_batch, lay);
    if (rc) return rc;
    return create_common(plan, lay);
}

int tcfft_plan_create_1d_split(tcfft_plan* plan, int n, int n_batch, int first_log2) {
    if (!plan) return TCFFT_INVALID_POINTER;
    *plan = nullptr;
    Layout lay;
    int rc = build_layout_1d(n, n_batch, lay, first_log2);
    if (rc) return rc;
    return create_common(plan, lay);
}

int tcfft_plan_create_1d_tuned(tcfft_plan* plan, int n, int n_batch, int* first_log2, float* best_ms) {
    if (!plan) return TCFFT_INVALID_POINTER;
    *plan = nullptr;
    // candidate first-pass lengths: 65536 (or the whole line) and 4096
    std::vector<int> cands = {16};
    if (n > 4096) cands.push_back(12);
    Layout probe;
    int rc = build_layout_1d(n, n_batch, probe);
    if (rc) return rc;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    void* buf = nullptr;
    const size_t bytes = (size_t)n * (size_t)n_batch * 4u;
    e = hipMalloc(&buf, bytes);
    if (e != hipSuccess) return hip_fail(e);
    hipEvent_t a = nullptr, b = nullptr;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess || hipMemset(buf, 0, bytes) != hipSuccess) {
        if (a) (void)hipEventDestroy(a);
        if (b) (void)hipEventDestroy(b);
        (void)hipFree(buf);
        return TCFFT_HIP_ERROR;
    }
    tcfft_plan best = nullptr;
    float best_t = 1e30f;
    int best_c = 16;
    for (int c : cands) {
        tcfft_plan p = nullptr;
        rc = tcfft_plan_create_1d_split(&p, n, n_batch, c);
        if (rc) break;
        const int reps = 5;
        for (int i = 0; i < 2 && !rc; ++i) rc = exec_all(p, (uint32_t*)buf, -1, nullptr);
        if (!rc && hipEventRecord(a, nullptr) != hipSuccess) rc = TCFFT_HIP_ERROR;
        for (int i = 0; i < reps && !rc; ++i) rc = exec_all(p, (uint32_t*)buf, -1, nullptr);
        if (!rc && hipEventRecord(b, nullptr) != hipSuccess) rc = TCFFT_HIP_ERROR;
        if (!rc && hipEventSynchronize(b) != hipSuccess) rc = TCFFT_HIP_ERROR;
        float ms = 0.f;
        if (!rc && hipEventElapsedTime(&ms, a, b) != hipSuccess) rc = TCFFT_HIP_ERROR;
        if (rc) {
            (void)tcfft_plan_destroy(p);
            break;
        }
        ms /= reps;
        if (ms < best_t) {
            if (best) (void)tcfft_plan_destroy(best);
            best = p;
            best_t = ms;
            best_c = c;
        } else {
            (void)tcfft_plan_destroy(p);
        }
    }
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    (void)hipFree(buf);
    if (rc) {
        if (best) (void)tcfft_plan_destroy(best);
        return rc;
    }
    *plan = best;
    if (first_log2) *first_log2 = best_c;
    if (best_ms) *best_ms = best_t;
    return TCFFT_SUCCESS;
}

int tcfft_plan_create_2d(tcfft_plan* plan, int nx, int ny, int n_batch) {
    if (!plan) return TCFFT_INVALID_POINTER;
    *plan = nullptr;
    Layout lay;
    int rc = build_layout_2d(nx, ny, n_batch, lay);
    if (rc) return rc;
    return create_common(plan, lay);
}

int tcfft_plan_destroy(tcfft_plan plan) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    DeviceGuard guard(plan->device);
    free_plan(plan);
    return TCFFT_SUCCESS;
}

static int copy_radices(const std::vector<int>& rad, int* radices, int capacity, int* n_radices) {
    if (!n_radices || (capacity > 0 && !radices)) return TCFFT_INVALID_POINTER;
    *n_radices = (int)rad.size();
    if (capacity < (int)rad.size()) return TCFFT_INVALID_VALUE;
    for (size_t i = 0; i < rad.size(); ++i) radices[i] = rad[i];
    return TCFFT_SUCCESS;
}

int tcfft_plan_radices(tcfft_plan plan, int axis, int* radices, int capacity, int* n_radices) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    const Layout& L = plan->lay;
    if (L.dims == 1) {
        if (axis != 0) return TCFFT_INVALID_VALUE;
        return copy_radices(L.rad_y, radices, capacity, n_radices);
    }
    if (axis == 0) return copy_radices(L.rad_x, radices, capacity, n_radices);
    if (axis == 1) return copy_radices(L.rad_y, radices, capacity, n_radices);
    return TCFFT_INVALID_VALUE;
}

int tcfft_query_1d(int n, int n_batch, int* radices, int capacity, int* n_radices, int* n_passes) {
    Layout lay;
    int rc = build_layout_1d(n, n_batch, lay);
    if (rc) return rc;
    if (n_passes) *n_passes = (int)lay.passes.size();
    return copy_radices(lay.rad_y, radices, capacity, n_radices);
}

int tcfft_query_1d_split(int n, int n_batch, int first_log2, int* radices, int capacity, int* n_radices,
                         int* n_passes) {
    Layout lay;
    int rc = build_layout_1d(n, n_batch, lay, first_log2);
    if (rc) return rc;
    if (n_passes) *n_passes = (int)lay.passes.size();
    return copy_radices(lay.rad_y, radices, capacity, n_radices);
}

int tcfft_query_2d(int nx, int ny, int n_batch, int* radices_x, int* n_radices_x, int* radices_y, int* n_radices_y,
                   int* n_passes, int capacity) {
    Layout lay;
    int rc = build_layout_2d(nx, ny, n_batch, lay);
    if (rc) return rc;
    if (n_passes) *n_passes = (int)lay.passes.size();
    rc = copy_radices(lay.rad_x, radices_x, capacity, n_radices_x);
    if (rc) return rc;
    return copy_radices(lay.rad_y, radices_y, capacity, n_radices_y);
}

static int query_split_list(decltype(&split_steps_of) list, int dims, int n_or_nx, int ny, int n_batch, int* desc,
                            int capacity, int* n_passes) {
    if (!n_passes || (capacity > 0 && !desc)) return TCFFT_INVALID_POINTER;
    Layout lay;
    int rc = dims == 1 ? build_layout_1d(n_or_nx, n_batch, lay)
                       : dims == 2 ? build_layout_2d(n_or_nx, ny, n_batch, lay) : TCFFT_INVALID_VALUE;
    if (rc) return rc;
    std::vector<tcfft_plan_s::SplitStep> steps;
    rc = list(dims, n_or_nx, ny, n_batch, steps);
    if (rc) return rc;
    *n_passes = (int)steps.size();
    if ((int)steps.size() > capacity) return TCFFT_INVALID_VALUE;
    for (size_t i = 0; i < steps.size(); ++i) {
        const auto& s = steps[i];
        int* d = desc + 5 * i;
        d[0] = s.R;
        d[1] = (int)s.a.q_log2;
        d[2] = (int)s.a.qlo_log2;
        d[3] = s.a.m_mask ? ilog2(s.a.m_mask + 1u) : 0;
        d[4] = (int)s.a.units;
    }
    return TCFFT_SUCCESS;
}

int tcfft_query_split(int dims, int n_or_nx, int ny, int n_batch, int* desc, int capacity, int* n_passes) {
    return query_split_list(split_steps_of, dims, n_or_nx, ny, n_batch, desc, capacity, n_passes);
}

int tcfft_query_split_exec(int dims, int n_or_nx, int ny, int n_batch, int* desc, int capacity, int* n_passes) {
    return query_split_list(split_exec_steps_of, dims, n_or_nx, ny, n_batch, desc, capacity, n_passes);
}

int tcfft_exec(tcfft_plan plan, void* data, int direction, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!data || ((uintptr_t)data & 15u)) return TCFFT_INVALID_POINTER;
    if (direction != TCFFT_FORWARD && direction != TCFFT_INVERSE) return TCFFT_INVALID_VALUE;
    DeviceGuard guard(plan->device);
    return exec_all(plan, (uint32_t*)data, direction, (hipStream_t)stream);
}

}  // extern "C"

namespace {

// Real-input kernels of a real-input plan: the row kernels for n <= 8192, the
// workgroup kernels (the half-size plan's 4096W-point first pass and its
// twiddle tables) for n = 16384..65536.
hipError_t launch_real(tcfft_plan_s* p, int sign, bool adjoint, const void* in, void* out, hipStream_t st) {
    const uint32_t half = (uint32_t)p->real_n / 2, batch = (uint32_t)p->lay.batch;
    if (half <= 4096)
        return tcfft::launch_r2c((int)(half / 256), sign, adjoint, (const uint32_t*)in, (uint32_t*)out, batch * (half / 256),
                                 p->w4096, p->w_real, st);
    const Pass& ps = p->lay.passes[0];
    if (ps.kind != 2 || ps.radix != (int)(half / 4096)) return hipErrorInvalidValue;
    return tcfft::launch_r2c_big(ps.radix, sign, adjoint, (const uint32_t*)in, (uint32_t*)out, batch, p->w4096, ps.big_hi,
                                 ps.big_lo, ps.big_M_log2 / 2, p->w_real, big_sched(p, ps.radix, batch), st);
}

// n reals per signal to n/2 + 1 bins: the real-input transform or, with
// `adjoint`, the adjoint of the inverse one.
int exec_to_bins(tcfft_plan plan, bool adjoint, const void* in, void* out, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!plan->real_n) return TCFFT_INVALID_PLAN;
    const size_t half = (size_t)plan->real_n / 2, batch = (size_t)plan->lay.batch;
    const uintptr_t a = (uintptr_t)in, b = (uintptr_t)out;
    if (!in || !out || (a & 15u) || (b & 3u)) return TCFFT_INVALID_POINTER;
    if (a < b + (half + 1) * batch * 4u && b < a + half * batch * 4u) return TCFFT_INVALID_POINTER;  // overlap
    DeviceGuard guard(plan->device);
    if (plan->real_ws) {
        // n > 65536: the n/2-point transform of z into the workspace, then the split
        int rc = tcfft_exec_natural(plan, in, plan->real_ws, TCFFT_FORWARD, stream);
        if (rc) return rc;
        const hipError_t e = tcfft::launch_real_pairs(-1, adjoint, plan->real_ws, (uint32_t*)out,
                                                      (uint32_t)ilog2((uint32_t)half), (uint32_t)batch,
                                                      plan->w_real_pair.first, plan->w_real_pair.second,
                                                      (uint32_t)ilog2((uint32_t)plan->real_n) / 2, (hipStream_t)stream);
        return e == hipSuccess ? TCFFT_SUCCESS : hip_fail(e);
    }
    hipError_t e = launch_real(plan, -1, adjoint, in, out, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

// n/2 + 1 bins per signal to n reals, likewise.
int exec_from_bins(tcfft_plan plan, bool adjoint, const void* in, void* out, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!plan->real_n) return TCFFT_INVALID_PLAN;
    const size_t half = (size_t)plan->real_n / 2, batch = (size_t)plan->lay.batch;
    const uintptr_t a = (uintptr_t)in, b = (uintptr_t)out;
    if (!in || !out || (a & 3u) || (b & 15u)) return TCFFT_INVALID_POINTER;
    if (a < b + half * batch * 4u && b < a + (half + 1) * batch * 4u) return TCFFT_INVALID_POINTER;  // overlap
    DeviceGuard guard(plan->device);
    if (plan->real_ws) {
        // n > 65536: the split into the workspace, then the inverse n/2-point transform
        const hipError_t e = tcfft::launch_real_pairs(+1, adjoint, (const uint32_t*)in, plan->real_ws,
                                                      (uint32_t)ilog2((uint32_t)half), (uint32_t)batch,
                                                      plan->w_real_pair.first, plan->w_real_pair.second,
                                                      (uint32_t)ilog2((uint32_t)plan->real_n) / 2, (hipStream_t)stream);
        if (e != hipSuccess) return hip_fail(e);
        return tcfft_exec_natural(plan, plan->real_ws, out, TCFFT_INVERSE, stream);
    }
    hipError_t e = launch_real(plan, +1, adjoint, in, out, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

}  // namespace

extern "C" {

int tcfft_plan_create_r2c_1d(tcfft_plan* plan, int n, int n_batch) {
    if (!plan) return TCFFT_INVALID_POINTER;
    *plan = nullptr;
    if (!is_pow2(n) || n < 512 || n > (1 << 27)) return TCFFT_INVALID_SIZE;
    Layout lay;
    int rc = build_layout_1d(n / 2, n_batch, lay);
    if (rc) return rc;
    rc = create_common(plan, lay, false);
    if (rc) return rc;
    tcfft_plan_s* p = *plan;
    p->real_n = n;
    if (n <= 65536) {
        // W_n^0..64 for the row kernels, W_n^0..64W for the workgroup kernels (n = 8192 W)
        const uint32_t count = n <= 8192 ? 65u : 64u * (uint32_t)(n / 8192) + 1u;
        rc = upload(p, host_table((uint32_t)ilog2((uint32_t)n), 1, count), &p->w_real);
    } else {
        rc = table_pair(p, (uint32_t)ilog2((uint32_t)n), p->w_real_pair);
        if (!rc) {
            void* ws = nullptr;
            const hipError_t e = hipMalloc(&ws, (size_t)n / 2 * (size_t)n_batch * 4u);
            if (e != hipSuccess) rc = hip_fail(e);
            else {
                p->allocs.push_back(ws);
                p->real_ws = (uint32_t*)ws;
                // the half-size complex plan's in-place natural order stages
                // through the same buffer (both hold n/2 * batch words)
                p->workspace = ws;
                p->workspace_bytes = (size_t)n / 2 * (size_t)n_batch * 4u;
            }
        }
    }
    if (rc) {
        free_plan(p);
        *plan = nullptr;
    }
    return rc;
}

int tcfft_exec_r2c(tcfft_plan plan, const void* in, void* out, void* stream) {
    return exec_to_bins(plan, false, in, out, stream);
}

int tcfft_exec_c2r(tcfft_plan plan, const void* in, void* out, void* stream) {
    return exec_from_bins(plan, false, in, out, stream);
}

int tcfft_exec_c2r_adjoint(tcfft_plan plan, const void* in, void* out, void* stream) {
    return exec_to_bins(plan, true, in, out, stream);
}

int tcfft_exec_r2c_adjoint(tcfft_plan plan, const void* in, void* out, void* stream) {
    return exec_from_bins(plan, true, in, out, stream);
}

int tcfft_plan_prepare_split(tcfft_plan plan) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (plan->real_n) return TCFFT_INVALID_PLAN;
    if (plan->split_ready) return TCFFT_SUCCESS;
    DeviceGuard guard(plan->device);
    const Layout& L = plan->lay;
    std::vector<tcfft_plan_s::SplitStep> steps;
    int rc = split_exec_steps_of(L.dims, L.dims == 1 ? L.n : L.nx, L.ny, L.batch, steps);
    if (rc) return rc;
    if (L.dims == 1 && L.n == 65536) {
        std::pair<float2*, float2*> t;
        rc = table_pair(plan, 16, t);
        if (rc) return rc;
    }
    for (auto& s : steps) {
        if (!s.a.m_mask) continue;
        std::pair<float2*, float2*> t;
        rc = table_pair(plan, (uint32_t)ilog2(s.a.m_mask + 1u), t);
        if (rc) return rc;
        s.a.hi = t.first;
        s.a.lo = t.second;
    }
    // a workspace only where some pass cannot go in place
    bool need = L.dims == 1 && L.n == 65536;
    for (const auto& s : steps) need |= s.transposing;
    if (need) {
        void* ws = nullptr;
        const hipError_t e = hipMalloc(&ws, plan->total * 8u);
        if (e != hipSuccess) return hip_fail(e);
        plan->allocs.push_back(ws);
        plan->split_ws = (float2*)ws;
    }
    plan->split_steps = std::move(steps);
    plan->split_ready = true;
    return TCFFT_SUCCESS;
}

int tcfft_exec_split(tcfft_plan plan, const void* in, void* out, int direction, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (plan->real_n) return TCFFT_INVALID_PLAN;
    if (!in || !out || ((uintptr_t)in & 15u) || ((uintptr_t)out & 15u)) return TCFFT_INVALID_POINTER;
    if (direction != TCFFT_FORWARD && direction != TCFFT_INVERSE) return TCFFT_INVALID_VALUE;
    const Layout& L = plan->lay;
    const size_t bytes = plan->total * 8u;
    const uintptr_t a = (uintptr_t)in, b = (uintptr_t)out;
    if (in != out && a < b + bytes && b < a + bytes) return TCFFT_INVALID_POINTER;  // partial overlap
    const bool is65536 = L.dims == 1 && L.n == 65536;
    if (!plan->split_ready) {
        // unprepared plans: the 65536-point transform out of place only
        if (!is65536) return TCFFT_INVALID_SIZE;
        if (in == out) return TCFFT_INVALID_POINTER;
    }
    DeviceGuard guard(plan->device);
    const tcfft::StartSched sched{(uint32_t)plan->split_delay, 3u, 0u};
    hipStream_t st = (hipStream_t)stream;
    if (is65536) {
        std::pair<float2*, float2*> t;
        int rc = table_pair(plan, 16, t);
        if (rc) return rc;
        const uint32_t batch = (uint32_t)L.batch;
        const uint32_t chunk =
            plan->split_chunk <= 0 || plan->split_chunk > (int)batch ? batch : (uint32_t)plan->split_chunk;
        // out of place: the intermediate in out; in place: in the workspace
        float2* mid = in == out ? plan->split_ws : (float2*)out;
        const hipError_t e = tcfft::launch_split_65536((const float2*)in, mid, (float2*)out, batch, chunk, direction,
                                                       plan->w4096, t.first, t.second, sched, st);
        return e == hipSuccess ? TCFFT_SUCCESS : hip_fail(e);
    }
    // Buffers, from the last pass back: it writes out; a transposing pass
    // reads the other buffer than it writes, a last pass of an axis the same
    // one.  The first pass reads in; if that is where it would write (in
    // place), the last pass reads the workspace instead, which flips every
    // earlier choice.
    const auto& S = plan->split_steps;
    const int P = (int)S.size();
    std::vector<float2*> dst(P);
    float2* const OUT = (float2*)out;
    float2* const WS = plan->split_ws;
    for (int attempt = 0; attempt < 2; ++attempt) {
        float2* cur_dst = OUT;
        float2* src_last = attempt ? WS : OUT;
        for (int j = P - 1; j >= 0; --j) {
            dst[j] = cur_dst;
            const float2* src = j == P - 1 ? src_last : (S[j].transposing ? (cur_dst == OUT ? WS : OUT) : cur_dst);
            cur_dst = (float2*)src;
        }
        if (!(S[0].transposing && dst[0] == (const float2*)in)) break;
    }
    const float2* src = (const float2*)in;
    for (int j = 0; j < P; ++j) {
        const hipError_t e =
            S[j].row_tiles
                ? tcfft::launch_split_rows(S[j].row_tiles, src, dst[j], S[j].a.units, direction, plan->w4096, sched,
                                           (uint32_t)plan->cus, st)
                : tcfft::launch_split_pass(S[j].R, S[j].row, src, dst[j], S[j].a, direction, plan->w4096, sched, st);
        if (e != hipSuccess) return hip_fail(e);
        src = dst[j];
    }
    return TCFFT_SUCCESS;
}

}  // extern "C"

namespace {

// Parameters of the natural-order / convolution kernels for a 1D plan of
// n = 4096*W (W = 1, 2, 4): W and the two-level W_n table (W = 1 needs only
// its entry 0, which the 4096-point table provides).
int dif_params(tcfft_plan_s* p, int& W, const float2*& hi, const float2*& lo, uint32_t& bits) {
    const Layout& L = p->lay;
    if (L.dims != 1 || (L.n != 4096 && L.n != 8192 && L.n != 16384)) return TCFFT_INVALID_SIZE;
    W = L.n / 4096;
    if (W == 1) {
        hi = lo = p->w4096;
        bits = 6;
        return TCFFT_SUCCESS;
    }
    const Pass& ps = L.passes[0];
    if (ps.kind != 2 || ps.radix != W) return TCFFT_INVALID_SIZE;
    hi = ps.big_hi;
    lo = ps.big_lo;
    bits = ps.big_M_log2 / 2;
    return TCFFT_SUCCESS;
}

// Transforms repeated in place on one buffer grow fp16 values to inf/NaN
// within two or three transforms (a 65536-point transform scales the rms by
// 256), and such data runs a few percent faster than finite data (65536 x
// 256: 28.0 against 29.2-29.7 us).  The tuners therefore start every timed
// run from a copy of the caller's data, kept here when it can be allocated,
// and put that data back at the end.
struct KeptData {
    void* data;
    size_t bytes;
    hipStream_t st;
    void* keep = nullptr;
    KeptData(void* d, size_t n, hipStream_t s) : data(d), bytes(n), st(s) {
        if (hipMalloc(&keep, bytes) != hipSuccess) {
            keep = nullptr;
            (void)hipGetLastError();
        } else if (hipMemcpyAsync(keep, data, bytes, hipMemcpyDeviceToDevice, st) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipFree(keep);
            keep = nullptr;
        }
    }
    KeptData(const KeptData&) = delete;
    KeptData& operator=(const KeptData&) = delete;
    int restore() const {
        if (keep && hipMemcpyAsync(data, keep, bytes, hipMemcpyDeviceToDevice, st) != hipSuccess)
            return TCFFT_HIP_ERROR;
        return TCFFT_SUCCESS;
    }
    ~KeptData() {
        if (!keep) return;
        (void)restore();
        (void)hipStreamSynchronize(st);
        (void)hipFree(keep);
    }
};

bool aligned16(const void* ptr) { return ptr && !((uintptr_t)ptr & 15u); }

}  // namespace

template <class In>
static int permute_to_dropin(tcfft_plan plan, const void* in, void* out, int n_lines, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    const Layout& L = plan->lay;
    if (L.dims != 1) return TCFFT_INVALID_PLAN;
    if (n_lines < 1 || (long)L.n * n_lines >= (1L << 31)) return TCFFT_INVALID_BATCH;
    const uintptr_t a = (uintptr_t)in, b = (uintptr_t)out;
    const size_t points = (size_t)L.n * (size_t)n_lines;
    if (!in || !out || (a & 15u) || (b & 15u)) return TCFFT_INVALID_POINTER;
    if (a < b + points * 4u && b < a + points * sizeof(In)) return TCFFT_INVALID_POINTER;  // overlap
    tcfft::GatherTile gt{};
    if (!gather_tile(L.rad_y, gt)) return TCFFT_INVALID_VALUE;
    DeviceGuard guard(plan->device);
    const hipError_t e = tcfft::launch_gather_tiled_1d((const In*)in, (uint32_t*)out, (uint32_t)ilog2((uint32_t)L.n),
                                                       (uint32_t)points, rev_spec(L.rad_y), gt, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

extern "C" {

int tcfft_exec_dif(tcfft_plan plan, const void* in, void* out, int direction, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!aligned16(in) || !aligned16(out)) return TCFFT_INVALID_POINTER;
    if (direction != TCFFT_FORWARD && direction != TCFFT_INVERSE) return TCFFT_INVALID_VALUE;
    int W = 0;
    const float2 *hi = nullptr, *lo = nullptr;
    uint32_t bits = 0;
    int rc = dif_params(plan, W, hi, lo, bits);
    if (rc) return rc;
    DeviceGuard guard(plan->device);
    hipError_t e = tcfft::launch_dif(W, (const uint32_t*)in, (uint32_t*)out, (uint32_t)plan->lay.batch, direction,
                                     plan->w4096, hi, lo, bits, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

int tcfft_conv_exec(tcfft_plan plan, int channels, const void* x, const void* h_rev, void* y, int conj_filter,
                    void* spec_out, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!aligned16(x) || !aligned16(h_rev) || !aligned16(y)) return TCFFT_INVALID_POINTER;
    if (spec_out && (!aligned16(spec_out) || spec_out == x || spec_out == y)) return TCFFT_INVALID_POINTER;
    if (conj_filter != 0 && conj_filter != 1) return TCFFT_INVALID_VALUE;
    int W = 0;
    const float2 *hi = nullptr, *lo = nullptr;
    uint32_t bits = 0;
    int rc = dif_params(plan, W, hi, lo, bits);
    if (rc) return rc;
    if (channels < 1 || plan->lay.batch % channels) return TCFFT_INVALID_BATCH;
    DeviceGuard guard(plan->device);
    hipError_t e = tcfft::launch_conv(W, conj_filter == 1, (const uint32_t*)x, (const uint32_t*)h_rev, (uint32_t*)y,
                                      (uint32_t*)spec_out, (uint32_t)plan->lay.batch, (uint32_t)channels,
                                      1.0f / (float)plan->lay.n, plan->w4096, hi, lo, bits, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

int tcfft_conv_filter_grad(tcfft_plan plan, int channels, const void* x_spec, const void* g_spec, void* gh_rev,
                           void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!aligned16(x_spec) || !aligned16(g_spec) || !aligned16(gh_rev)) return TCFFT_INVALID_POINTER;
    const Layout& L = plan->lay;
    if (L.dims != 1) return TCFFT_INVALID_SIZE;
    if (channels < 1 || L.batch % channels) return TCFFT_INVALID_BATCH;
    DeviceGuard guard(plan->device);
    hipError_t e = tcfft::launch_conv_wgrad((const uint32_t*)x_spec, (const uint32_t*)g_spec, (float2*)gh_rev,
                                            (uint32_t)L.n, (uint32_t)channels, (uint32_t)(L.batch / channels),
                                            1.0f / (float)L.n, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

int tcfft_conv_filter_grad_natural(tcfft_plan plan, int channels, const void* x_spec, const void* g_spec, void* gh,
                                   void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!aligned16(x_spec) || !aligned16(g_spec) || !aligned16(gh)) return TCFFT_INVALID_POINTER;
    int W = 0;
    const float2 *hi = nullptr, *lo = nullptr;
    uint32_t bits = 0;
    int rc = dif_params(plan, W, hi, lo, bits);
    if (rc) return rc;
    const Layout& L = plan->lay;
    if (channels < 1 || L.batch % channels) return TCFFT_INVALID_BATCH;
    DeviceGuard guard(plan->device);
    hipError_t e = tcfft::launch_conv_wgrad_nat(W, (const uint32_t*)x_spec, (const uint32_t*)g_spec, (float2*)gh,
                                                (uint32_t)channels, (uint32_t)(L.batch / channels),
                                                1.0f / (float)L.n, (uint32_t)plan->cus, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

int tcfft_plan_set_option(tcfft_plan plan, int option, int value) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    switch (option) {
    case TCFFT_OPT_SPLIT_CHUNK:
        if (value < 0) return TCFFT_INVALID_VALUE;
        plan->split_chunk = value;
        return TCFFT_SUCCESS;
    case TCFFT_OPT_BIG_DELAY:
        if (value < -1 || value > 64) return TCFFT_INVALID_VALUE;
        plan->big_delay = plan->set.delay = value;
        return TCFFT_SUCCESS;
    case TCFFT_OPT_COLS_DELAY:
        if (value < 0 || value > 64) return TCFFT_INVALID_VALUE;
        plan->cols_delay = value;
        return TCFFT_SUCCESS;
    case TCFFT_OPT_BIG_GROUPS:
        if (value < 1 || value > 8) return TCFFT_INVALID_VALUE;
        plan->big_groups = plan->set.groups = value;
        return TCFFT_SUCCESS;
    case TCFFT_OPT_SPLIT_DELAY:
        if (value < 0 || value > 64) return TCFFT_INVALID_VALUE;
        plan->split_delay = value;
        return TCFFT_SUCCESS;
    case TCFFT_OPT_ROWS_WAVES:
        if (value != 0 && value != 1 && value != 2 && value != 4) return TCFFT_INVALID_VALUE;
        plan->rows_waves = plan->set.waves = value;
        return TCFFT_SUCCESS;
    case TCFFT_OPT_FIRST_CACHED:
        if (value < -1 || value > 1) return TCFFT_INVALID_VALUE;
        plan->first_cached = value;
        return TCFFT_SUCCESS;
    case TCFFT_OPT_ROWS_TILES:
        if (value != 0 && value != 4 && value != 8 && value != 16) return TCFFT_INVALID_VALUE;
        plan->rows_tiles = plan->set.tiles = value;
        return TCFFT_SUCCESS;
    case TCFFT_OPT_MALL_CHUNK:
        if (value != 0 && (value < 16 || value > 65536)) return TCFFT_INVALID_VALUE;
        plan->mall_chunk_mib = value;
        return TCFFT_SUCCESS;
    default: return TCFFT_INVALID_VALUE;
    }
}

int tcfft_plan_autotune(tcfft_plan plan, void* data, void* stream, int* best_groups, int* best_delay,
                        float* best_ms) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!data || ((uintptr_t)data & 15u)) return TCFFT_INVALID_POINTER;
    DeviceGuard guard(plan->device);
    hipStream_t st = (hipStream_t)stream;
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess) return TCFFT_HIP_ERROR;
    if (hipEventCreate(&b) != hipSuccess) {
        (void)hipEventDestroy(a);
        return TCFFT_HIP_ERROR;
    }
    int rc = TCFFT_SUCCESS;
    // Back to back on one buffer, a transform of up to a few hundred MiB
    // finds its data in the 256 MB last-level cache, and the schedule that
    // wins there is not the one that wins on cold data (a caller's previous
    // work has evicted it).  Each timed run therefore follows a write of a
    // buffer of that size (when one can be allocated) and is timed alone.
    const size_t flush_bytes = size_t(256) << 20;
    void* flush = nullptr;
    if (hipMalloc(&flush, flush_bytes) != hipSuccess) {
        flush = nullptr;
        (void)hipGetLastError();
    }
    const KeptData kept(data, plan->total * sizeof(uint32_t), st);
    // mean of five single cold executions after two warm-up ones, each timed
    // one on the caller's data
    auto time_current = [&](float& ms) {
        for (int i = 0; i < 2 && !rc; ++i) rc = exec_all(plan, (uint32_t*)data, -1, st);
        float total = 0.f;
        for (int i = 0; i < 5 && !rc; ++i) {
            rc = kept.restore();
            if (!rc && flush && hipMemsetAsync(flush, i + 1, flush_bytes, st) != hipSuccess) rc = TCFFT_HIP_ERROR;
            if (!rc && hipEventRecord(a, st) != hipSuccess) rc = TCFFT_HIP_ERROR;
            if (!rc) rc = exec_all(plan, (uint32_t*)data, -1, st);
            if (!rc && hipEventRecord(b, st) != hipSuccess) rc = TCFFT_HIP_ERROR;
            if (!rc && hipEventSynchronize(b) != hipSuccess) rc = TCFFT_HIP_ERROR;
            float t = 0.f;
            if (!rc && hipEventElapsedTime(&t, a, b) != hipSuccess) rc = TCFFT_HIP_ERROR;
            total += t;
        }
        ms = total / 5.f;
    };
    // Each candidate is timed once, then the four fastest again in three
    // alternating rounds, each keeping its best: neighbouring schedules
    // differ by a few percent, less than one sweep's noise.
    struct Cand {
        int a, b;  // (groups, delay) of the first pass, or (cols delay, 0)
        float ms;
    };
    auto tune = [&](std::vector<Cand>& cands, const std::function<void(const Cand&)>& apply) {
        for (Cand& c : cands) {
            if (rc) return;
            apply(c);
            time_current(c.ms);
        }
        std::sort(cands.begin(), cands.end(), [](const Cand& x, const Cand& y) { return x.ms < y.ms; });
        if (cands.size() > 4) cands.resize(4);
        for (int round = 0; round < 3 && !rc; ++round)
            for (Cand& c : cands) {
                float ms = 0.f;
                apply(c);
                time_current(ms);
                if (!rc) c.ms = std::min(c.ms, ms);
            }
        std::sort(cands.begin(), cands.end(), [](const Cand& x, const Cand& y) { return x.ms < y.ms; });
    };
    // start schedule of the first pass: no stagger, or 3, 5 or 7 groups
    // (counts coprime with 2, see big_sched) with delays of 1..4 quanta
    const int saved_groups = plan->big_groups, saved_delay = plan->big_delay;
    std::vector<Cand> first{{3, 0, 0.f}};
    for (int g : {3, 5, 7})
        for (int d = 1; d <= 4; ++d) first.push_back({g, d, 0.f});
    tune(first, [&](const Cand& c) {
        plan->big_groups = c.a;
        plan->big_delay = c.b;
    });
    float best_t = rc ? 0.f : first[0].ms;
    if (rc) {
        plan->big_groups = saved_groups;
        plan->big_delay = saved_delay;
    } else {
        plan->big_groups = first[0].a;
        plan->big_delay = first[0].b;
        if (best_groups) *best_groups = first[0].a;
        if (best_delay) *best_delay = first[0].b;
    }
    // then the workgroup size of a contiguous-row first pass (1, 2 or 4
    // waves), with the chosen start schedule
    if (!rc && plan->lay.passes[0].kind == 0) {
        const int saved = plan->rows_waves;
        std::vector<Cand> wg{{4, 0, 0.f}, {2, 0, 0.f}, {1, 0, 0.f}};
        tune(wg, [&](const Cand& c) { plan->rows_waves = c.a; });
        plan->rows_waves = rc ? saved : wg[0].a;
        if (!rc) best_t = std::min(best_t, wg[0].ms);
    }
    // then the tiles per wave of such a pass of lines up to 2048 points
    // (4096-point lines keep the choice by the grid, see rows_nt)
    const Pass& p0 = plan->lay.passes[0];
    if (!rc && p0.kind == 0 && p0.radix < 16 && !p0.has_epi) {
        const int saved = plan->rows_tiles;
        std::vector<Cand> tiles{{16, 0, 0.f}, {8, 0, 0.f}};
        if (p0.radix <= 4) tiles.push_back({4, 0, 0.f});
        tune(tiles, [&](const Cand& c) { plan->rows_tiles = c.a; });
        plan->rows_tiles = rc ? saved : tiles[0].a;
        if (!rc) best_t = std::min(best_t, tiles[0].ms);
    }
    // then the start delay of a radix-256*W column pass, if the plan has one
    bool has_cols_big = false;
    for (const Pass& ps : plan->lay.passes) has_cols_big |= ps.kind == 3;
    if (has_cols_big && !rc) {
        const int saved = plan->cols_delay;
        std::vector<Cand> cols;
        for (int cd = 0; cd <= 4; ++cd) cols.push_back({cd, 0, 0.f});
        tune(cols, [&](const Cand& c) { plan->cols_delay = c.a; });
        plan->cols_delay = rc ? saved : cols[0].a;
        if (!rc) best_t = std::min(best_t, cols[0].ms);
    }
    if (flush) (void)hipFree(flush);
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    if (rc) return rc;
    if (best_ms) *best_ms = best_t;
    return TCFFT_SUCCESS;
}

int tcfft_plan_num_passes(tcfft_plan plan, int* n_passes) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!n_passes) return TCFFT_INVALID_POINTER;
    *n_passes = (int)plan->lay.passes.size();
    return TCFFT_SUCCESS;
}

int tcfft_exec_passes(tcfft_plan plan, void* data, int direction, int first, int count, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!data || ((uintptr_t)data & 15u)) return TCFFT_INVALID_POINTER;
    if (direction != TCFFT_FORWARD && direction != TCFFT_INVERSE) return TCFFT_INVALID_VALUE;
    const int np = (int)plan->lay.passes.size();
    if (first < 0 || count < 0 || first > np || count > np - first) return TCFFT_INVALID_VALUE;
    DeviceGuard guard(plan->device);
    return run_passes(plan, (uint32_t*)data, direction, (hipStream_t)stream, (size_t)first, (size_t)count);
}

int tcfft_exec_natural(tcfft_plan plan, const void* in, void* out, int direction, void* stream) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    return tcfft::exec_natural_staged(plan, in, out, direction, stream, plan->workspace, plan->workspace_bytes);
}

}  // extern "C"

namespace tcfft {

size_t natural_stage_bytes(tcfft_plan plan, const void* in, const void* out) {
    if (!valid(plan) || in != out || !natural_needs_stage(plan->lay)) return 0;
    return plan->total * 4u;
}

int plan_device(tcfft_plan plan) { return valid(plan) ? plan->device : -1; }

int exec_natural_staged(tcfft_plan plan, const void* in, void* out, int direction, void* stream, void* stage_buf,
                        size_t stage_cap) {
    if (!valid(plan)) return TCFFT_INVALID_PLAN;
    if (!in || !out || ((uintptr_t)in & 15u) || ((uintptr_t)out & 15u)) return TCFFT_INVALID_POINTER;
    if (direction != TCFFT_FORWARD && direction != TCFFT_INVERSE) return TCFFT_INVALID_VALUE;
    DeviceGuard guard(plan->device);
    hipStream_t st = (hipStream_t)stream;
    const Layout& L0 = plan->lay;
    const Pass& first = L0.passes[0];
    const size_t bytes = plan->total * 4;
    auto stage = [&](const uint32_t*& src) -> int {  // copy of the input in the staging buffer
        if (!stage_buf || stage_cap < bytes) return TCFFT_INVALID_PLAN;
        hipError_t e = hipMemcpyAsync(stage_buf, in, bytes, hipMemcpyDeviceToDevice, st);
        if (e != hipSuccess) return hip_fail(e);
        src = (const uint32_t*)stage_buf;
        return TCFFT_SUCCESS;
    };
    // First pass over lines of up to 4096 points (k_rows) or of 8192..32768
    // points (k_big<W <= 8>): the digit reversal is done in that pass's load
    // (1D in place or not; 2D with its x reversal as a line permutation of the
    // stores, from a staged copy when in place), so natural order costs no
    // extra pass.
    const bool fused_rows = first.kind == 0 && !first.has_epi;
    const bool fused_big = first.kind == 2 && !first.has_epi;
    if (fused_rows || fused_big) {
        const uint32_t* rsrc = (const uint32_t*)in;
        if (L0.dims == 2 && in == out) {
            int rc = stage(rsrc);
            if (rc) return rc;
        }
        uint32_t nx_log2 = 0;
        tcfft::RevSpec x_pos{};
        if (L0.dims == 2) {
            nx_log2 = (uint32_t)ilog2((uint32_t)L0.nx);
            std::vector<int> rx(L0.rad_x.rbegin(), L0.rad_x.rend());
            x_pos = rev_spec(rx);
        }
        // per batch chunk (chunk_signals): the fused first pass, then the rest
        const uint32_t B = (uint32_t)L0.batch;
        const size_t per = plan->total / B;
        return for_chunks(plan, [&](uint32_t s0, uint32_t ns) -> int {
            Pass fp = first;
            fp.n_tiles = (uint32_t)((uint64_t)first.n_tiles / B * ns);
            const uint32_t nt = fused_rows ? rows_nt_nat(plan, fp) : 16u;
            tcfft::StartSched sc = fused_rows ? nat_sched(plan) : nat_big_sched(plan, fp.radix, fp.n_tiles);
            sc.cached_out = cached_out(plan, 0, ns);
            const uint32_t* ci = rsrc + per * s0;
            uint32_t* co = (uint32_t*)out + per * s0;
            hipError_t e = fused_rows ? tcfft::launch_rows_nat(fp.radix, ci, co, fp.n_tiles, direction, plan->w4096,
                                                               nx_log2, plan->xpos, sc, nt, rows_wg_nat(plan, fp), st)
                                      : tcfft::launch_big_nat(fp.radix, ci, co, fp.n_tiles, direction, plan->w4096,
                                                              fp.big_hi, fp.big_lo, fp.big_M_log2 / 2, nx_log2, x_pos,
                                                              sc, st);
            if (e != hipSuccess) return hip_fail(e);
            return run_passes(plan, (uint32_t*)out, direction, st, 1, ~(size_t)0, s0, ns);
        });
    }
    // 1D lines above 65536 points: the LDS-tiled reversal pass, then the
    // plan's passes (every plan takes one of these two routes: 2D rows are
    // at most 65536 points, and a longer line's radix list always admits a
    // reversal tile).
    const Layout& L = plan->lay;
    tcfft::GatherTile gt{};
    if (L.dims != 1 || !gather_tile(L.rad_y, gt)) return TCFFT_INVALID_VALUE;
    const uint32_t* src = (const uint32_t*)in;
    if (in == out) {
        int rc = stage(src);
        if (rc) return rc;
    }
    // 2^17..2^20 points (n = 65536*R): two passes that read natural order
    // themselves, or, for the fewest signals, the reversal and the plan's own
    // passes.  k_lines_nat's R workgroups a signal each pull 256 KiB through
    // one CU, which a small grid waits for when the input is not in L2; where
    // they are a multiple of 16, the two that share 128-byte lines run on one
    // XCD.  Input in the MALL, reversal + plan / two passes: 2^17 x 1 25.6 /
    // 26.6 us, x 4 26.6 / 27.0, x 5 27.3 / 27.2, x 8 28.3 / 25.3; 2^18 x 1 26.2 /
    // 28.9, x 3 27.7 / 29.4, x 4 28.5 / 27.1, x 5 30.2 / 30.2; 2^19 x 1 27.3 /
    // 31.8, x 2 29.0 / 29.5, x 3 32.0 / 33.7, x 4 34.0 / 33.6, x 5 36.6 / 36.8;
    // 2^20 x 1 29.1 / 33.1, x 2 34.1 / 37.4, x 3 38.8 / 39.5, x 4 45.5 / 41.0.
    // Between the split pass and this transform of a real-input plan, r2c and
    // c2r of twice the points: 2^17 x 4 30.3 / 29.9 and 29.6 / 29.8, x 5 31.6 /
    // 30.3 and 30.6 / 30.3; 2^18 x 3 32.3 / 32.5 and 31.5 / 32.8, x 4 33.9 / 30.8
    // and 32.8 / 29.2; 2^19 x 1 31.1 / 34.4 and 30.7 / 34.5, x 2 34.9 / 33.3 and
    // 33.8 / 31.3, x 3 40.2 / 38.3 and 38.5 / 39.4; 2^20 x 1 33.8 / 36.4 and 33.5 /
    // 34.7, x 2 43.1 / 42.8 and 40.4 / 38.7, x 3 51.2 / 47.6 and 46.1 / 42.6.
    const bool two_pass = L.passes.size() == 2 && first.kind == 2 && first.radix == 16 && first.has_epi &&
                          L.passes[1].kind == 1 && L.passes[1].radix <= 16;
    auto enough = [&](uint32_t ns) {
        const uint32_t R = (uint32_t)L.passes[1].radix;
        if (plan->real_n) return ns >= (R == 2u ? 5u : R == 4u ? 4u : 2u);
        return ns >= (R <= 4u ? 5u : R == 8u ? 6u : 4u) || (R <= 8u && ns * R % 16u == 0u);
    };
    // per batch chunk (chunk_signals)
    const tcfft::RevSpec spec = rev_spec(L.rad_y);
    return for_chunks(plan, [&](uint32_t s0, uint32_t ns) -> int {
        const size_t off = (size_t)L.n * s0;
        if (two_pass && enough(ns)) {
            // no stagger but the caller's: 2^20 x 16 66 us with the 65536-point
            // kernel's schedule, 59 without, 2^17 x 128 59 and 53
            tcfft::StartSched sc = nat_sched(plan);
            sc.cached_out = cached_out(plan, 0, ns);
            const hipError_t e = tcfft::launch_nat_two_pass(L.passes[1].radix, src + off, (uint32_t*)out + off, ns,
                                                            direction, plan->w4096, first.epi, sc, st);
            return e == hipSuccess ? TCFFT_SUCCESS : hip_fail(e);
        }
        hipError_t e = tcfft::launch_gather_tiled_1d(src + off, (uint32_t*)out + off, (uint32_t)ilog2((uint32_t)L.n),
                                                     (uint32_t)((size_t)L.n * ns), spec, gt, st);
        if (e != hipSuccess) return hip_fail(e);
        return run_passes(plan, (uint32_t*)out, direction, st, 0, ~(size_t)0, s0, ns);
    });
}

}  // namespace tcfft

extern "C" {

int tcfft_permute_to_dropin(tcfft_plan plan, const void* in, void* out, int n_lines, void* stream) {
    return permute_to_dropin<uint32_t>(plan, in, out, n_lines, stream);
}

int tcfft_permute_to_dropin_f32(tcfft_plan plan, const void* in, void* out, int n_lines, void* stream) {
    return permute_to_dropin<float2>(plan, in, out, n_lines, stream);
}

int tcfft_gen_rev(int n, const int* radices, int n_radices, int* rev) {
    if (!radices || !rev) return TCFFT_INVALID_POINTER;
    if (n_radices < 0 || n_radices > 64) return TCFFT_INVALID_VALUE;
    long prod = 1;
    for (int i = 0; i < n_radices; ++i) {
        if (radices[i] < 2) return TCFFT_INVALID_VALUE;
        prod *= radices[i];
    }
    if (prod != n) return TCFFT_INVALID_SIZE;
    for (int p = 0; p < n; ++p) {
        int q = p, idx = 0;
        int digits[64];
        for (int i = 0; i < n_radices; ++i) {
            digits[i] = q % radices[i];
            q /= radices[i];
        }
        for (int i = 0; i < n_radices; ++i) idx = idx * radices[i] + digits[i];
        rev[p] = idx;
    }
    return TCFFT_SUCCESS;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Uneven batches (no counterpart in the reference): many signals of sizes
// 2^8 .. 2^16 packed back to back, transformed by one persistent launch.
namespace {
constexpr uint32_t kMultiMagic = 0x7cff3a17u;
}

struct tcfft_multi_s {
    uint32_t magic = kMultiMagic;
    int device = 0;
    std::vector<int> sizes;
    std::vector<uint32_t> offsets;  // element offset of every signal
    size_t total = 0;
    std::vector<tcfft::MultiTask> tasks;
    std::vector<uint32_t> task_offsets;  // offsets in task order
    tcfft::MultiTask* d_tasks = nullptr;
    uint32_t* d_offsets = nullptr;
    float2* w4096 = nullptr;
    tcfft::MultiTables tb{};
    uint32_t grid = 256;
    int order = 0;
    uint32_t cus = 256;  // compute units of the device
    int delay = 0;  // start delay of the resident workgroups (3 groups, quanta of 1024 cycles)
    std::vector<void*> allocs;
};

namespace {

bool valid_multi(tcfft_multi_s* p) { return p && p->magic == kMultiMagic; }

int multi_alloc(tcfft_multi_s* p, size_t bytes, void** out) {
    hipError_t e = hipMalloc(out, bytes);
    if (e != hipSuccess) return hip_fail(e);
    p->allocs.push_back(*out);
    return TCFFT_SUCCESS;
}

// Build the task list for an ordering policy:
//   0: size classes from the largest to the smallest (longest tasks first)
//   1: classes interleaved task by task
//   2: size classes from the smallest to the largest
void multi_build_tasks(tcfft_multi_s* p, int order) {
    std::vector<std::vector<uint32_t>> byclass(17);
    for (size_t i = 0; i < p->sizes.size(); ++i) byclass[ilog2((uint32_t)p->sizes[i])].push_back((uint32_t)i);
    std::vector<std::vector<tcfft::MultiTask>> cls_tasks(17);
    std::vector<std::vector<std::vector<uint32_t>>> cls_offs(17);
    for (int m = 8; m <= 16; ++m) {
        const auto& ids = byclass[m];
        const int per_task = m <= 12 ? 256 / (1 << (m - 8)) : 16 / (1 << (m - 12));
        for (size_t s0 = 0; s0 < ids.size(); s0 += per_task) {
            const size_t cnt = std::min(ids.size() - s0, (size_t)per_task);
            std::vector<uint32_t> offs;
            for (size_t k = 0; k < cnt; ++k) offs.push_back(p->offsets[ids[s0 + k]]);
            cls_tasks[m].push_back(tcfft::MultiTask{(uint32_t)m, 0u, (uint32_t)cnt, 0u});
            cls_offs[m].push_back(offs);
        }
    }
    p->tasks.clear();
    p->task_offsets.clear();
    auto emit = [&](int m, size_t k) {
        tcfft::MultiTask t = cls_tasks[m][k];
        t.first = (uint32_t)p->task_offsets.size();
        for (uint32_t o : cls_offs[m][k]) p->task_offsets.push_back(o);
        p->tasks.push_back(t);
    };
    if (order == 1) {
        size_t most = 0;
        for (int m = 8; m <= 16; ++m) most = std::max(most, cls_tasks[m].size());
        for (size_t k = 0; k < most; ++k)
            for (int m = 16; m >= 8; --m)
                if (k < cls_tasks[m].size()) emit(m, k);
    } else {
        for (int i = 0; i < 9; ++i) {
            const int m = order == 2 ? 8 + i : 16 - i;
            for (size_t k = 0; k < cls_tasks[m].size(); ++k) emit(m, k);
        }
    }
}

int multi_upload_tasks(tcfft_multi_s* p) {
    hipError_t e = hipMemcpy(p->d_tasks, p->tasks.data(), p->tasks.size() * sizeof(tcfft::MultiTask),
                             hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(e);
    e = hipMemcpy(p->d_offsets, p->task_offsets.data(), p->task_offsets.size() * sizeof(uint32_t),
                  hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

void multi_free(tcfft_multi_s* p) {
    for (void* a : p->allocs) (void)hipFree(a);
    p->magic = 0;
    delete p;
}

}  // namespace

extern "C" {

int tcfft_multi_create(tcfft_multi* plan, int n_signals, const int* sizes) {
    if (!plan || !sizes) return TCFFT_INVALID_POINTER;
    *plan = nullptr;
    if (n_signals < 1) return TCFFT_INVALID_BATCH;
    size_t total = 0;
    for (int i = 0; i < n_signals; ++i) {
        if (!is_pow2(sizes[i]) || sizes[i] < 256 || sizes[i] > 65536) return TCFFT_INVALID_SIZE;
        total += (size_t)sizes[i];
    }
    if (total >= (1ull << 31)) return TCFFT_INVALID_BATCH;
    tcfft_multi_s* p = new (std::nothrow) tcfft_multi_s;
    if (!p) return TCFFT_ALLOC_FAILED;
    p->sizes.assign(sizes, sizes + n_signals);
    p->offsets.resize(n_signals);
    size_t acc = 0;
    for (int i = 0; i < n_signals; ++i) {
        p->offsets[i] = (uint32_t)acc;
        acc += (size_t)sizes[i];
    }
    p->total = total;
    int rc = TCFFT_SUCCESS;
    hipError_t e = hipGetDevice(&p->device);
    if (e != hipSuccess) rc = hip_fail(e);
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, p->device) == hipSuccess && cus > 0)
        p->cus = (uint32_t)cus;
    multi_build_tasks(p, 0);
    void* d = nullptr;
    if (!rc) rc = multi_alloc(p, p->tasks.size() * sizeof(tcfft::MultiTask), &d);
    p->d_tasks = (tcfft::MultiTask*)d;
    if (!rc) rc = multi_alloc(p, std::max<size_t>(p->task_offsets.size(), 1) * sizeof(uint32_t), &d);
    p->d_offsets = (uint32_t*)d;
    if (!rc) rc = multi_upload_tasks(p);
    // tables: W_4096 and two-level W_N for N = 2^13 .. 2^16
    auto up = [&](const std::vector<float2>& h, const float2** dst) {
        if (rc) return;
        void* dd = nullptr;
        rc = multi_alloc(p, h.size() * sizeof(float2), &dd);
        if (rc) return;
        hipError_t ee = hipMemcpy(dd, h.data(), h.size() * sizeof(float2), hipMemcpyHostToDevice);
        if (ee != hipSuccess) rc = hip_fail(ee);
        *dst = (const float2*)dd;
    };
    const float2* w = nullptr;
    up(host_table(12, 1, 4096), &w);
    p->w4096 = (float2*)w;
    for (int m = 13; m <= 16; ++m) {
        const uint32_t lo = (uint32_t)m / 2;
        up(host_table((uint32_t)m, 1ull << lo, 1u << (m - lo)), &p->tb.hi[m - 13]);
        up(host_table((uint32_t)m, 1, 1u << lo), &p->tb.lo[m - 13]);
    }
    if (rc) {
        multi_free(p);
        return rc;
    }
    *plan = p;
    return TCFFT_SUCCESS;
}

int tcfft_multi_destroy(tcfft_multi plan) {
    if (!valid_multi(plan)) return TCFFT_INVALID_PLAN;
    DeviceGuard guard(plan->device);
    multi_free(plan);
    return TCFFT_SUCCESS;
}

int tcfft_multi_info(tcfft_multi plan, int* n_tasks, long long* total_elements) {
    if (!valid_multi(plan)) return TCFFT_INVALID_PLAN;
    if (n_tasks) *n_tasks = (int)plan->tasks.size();
    if (total_elements) *total_elements = (long long)plan->total;
    return TCFFT_SUCCESS;
}

int tcfft_multi_set_start_delay(tcfft_multi plan, int delay) {
    if (!valid_multi(plan)) return TCFFT_INVALID_PLAN;
    if (delay < 0 || delay > 64) return TCFFT_INVALID_VALUE;
    plan->delay = delay;
    return TCFFT_SUCCESS;
}

int tcfft_multi_get_schedule(tcfft_multi plan, int* grid, int* order, int* delay) {
    if (!valid_multi(plan)) return TCFFT_INVALID_PLAN;
    if (grid) *grid = (int)plan->grid;
    if (order) *order = plan->order;
    if (delay) *delay = plan->delay;
    return TCFFT_SUCCESS;
}

int tcfft_multi_set_schedule(tcfft_multi plan, int grid, int order) {
    if (!valid_multi(plan)) return TCFFT_INVALID_PLAN;
    if (grid < 0 || order < 0 || order > 2) return TCFFT_INVALID_VALUE;
    DeviceGuard guard(plan->device);
    plan->grid = (uint32_t)grid;
    if (order != plan->order) {
        plan->order = order;
        multi_build_tasks(plan, order);
        return multi_upload_tasks(plan);
    }
    return TCFFT_SUCCESS;
}

int tcfft_multi_exec(tcfft_multi plan, void* data, int direction, void* stream) {
    if (!valid_multi(plan)) return TCFFT_INVALID_PLAN;
    if (!data || ((uintptr_t)data & 15u)) return TCFFT_INVALID_POINTER;
    if (direction != TCFFT_FORWARD && direction != TCFFT_INVERSE) return TCFFT_INVALID_VALUE;
    DeviceGuard guard(plan->device);
    hipError_t e = tcfft::launch_multi((uint32_t*)data, plan->d_tasks, (uint32_t)plan->tasks.size(), plan->d_offsets,
                                       plan->grid, direction, plan->w4096, plan->tb,
                                       tcfft::StartSched{(uint32_t)plan->delay, 3u, 0u}, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

int tcfft_multi_exec_natural(tcfft_multi plan, const void* in, void* out, int direction, void* stream) {
    if (!valid_multi(plan)) return TCFFT_INVALID_PLAN;
    if (!in || !out || ((uintptr_t)in & 15u) || ((uintptr_t)out & 15u)) return TCFFT_INVALID_POINTER;
    const uintptr_t a = (uintptr_t)in, b = (uintptr_t)out;
    const size_t bytes = plan->total * 4u;
    if (in != out && a < b + bytes && b < a + bytes) return TCFFT_INVALID_POINTER;  // partial overlap
    if (direction != TCFFT_FORWARD && direction != TCFFT_INVERSE) return TCFFT_INVALID_VALUE;
    DeviceGuard guard(plan->device);
    // Order 0 with more than a task per CU is walked from its end: the small
    // signals' tasks first, whose different lengths spread the workgroups'
    // phases.  Natural order, largest first -> smallest first: 2048 signals
    // (480 tasks) 68.5 -> 63.6 us on a grid of 256, 102.6 -> 96.9 on 128, 68.0
    // -> 63.9 on 512; 4096 signals 131.8 -> 122.1, but 190.1 -> 193.1 on 128;
    // 1100 signals 35.9 -> 35.4.  With a task per CU or fewer the longest go
    // first (700 signals 26.6 against 26.9).  The drop-in call gains nothing
    // from it.  A property of the list alone, so that setting the current
    // schedule again changes nothing.
    const bool reverse = plan->order == 0 && plan->tasks.size() > plan->cus;
    hipError_t e = tcfft::launch_multi_nat((const uint32_t*)in, (uint32_t*)out, plan->d_tasks,
                                           (uint32_t)plan->tasks.size(), plan->d_offsets, plan->grid, direction,
                                           plan->w4096, plan->tb, reverse,
                                           tcfft::StartSched{(uint32_t)plan->delay, 3u, 0u}, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return TCFFT_SUCCESS;
}

int tcfft_multi_autotune(tcfft_multi plan, void* data, void* stream, int* best_grid, int* best_order,
                         float* best_ms) {
    if (!valid_multi(plan)) return TCFFT_INVALID_PLAN;
    if (!data || ((uintptr_t)data & 15u)) return TCFFT_INVALID_POINTER;
    DeviceGuard guard(plan->device);
    hipStream_t st = (hipStream_t)stream;
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess) return TCFFT_HIP_ERROR;
    if (hipEventCreate(&b) != hipSuccess) {
        (void)hipEventDestroy(a);
        return TCFFT_HIP_ERROR;
    }
    int cu = 256;
    (void)hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, plan->device);
    const int grids[] = {cu / 2, cu, 2 * cu};
    struct Cand {
        int grid, order, delay;
        float ms;
    };
    std::vector<Cand> cands;
    int rc = TCFFT_SUCCESS;
    // Back to back on one buffer, a run finds part of the data still in the
    // 256 MB last-level cache, which favours some schedules over others.
    // Before each timed run the tuner therefore writes a buffer of that size
    // (when it can allocate one), as a caller's previous work would.
    const size_t flush_bytes = size_t(256) << 20;
    void* flush = nullptr;
    if (hipMalloc(&flush, flush_bytes) != hipSuccess) {
        flush = nullptr;
        (void)hipGetLastError();
    }
    const KeptData kept(data, plan->total * sizeof(uint32_t), st);
    // mean of five single timed executions after two warm-up ones, on the
    // current schedule, each timed one on the caller's data
    auto time_current = [&](float& ms) {
        for (int i = 0; i < 2 && !rc; ++i) rc = tcfft_multi_exec(plan, data, TCFFT_FORWARD, stream);
        float total = 0.f;
        for (int i = 0; i < 5 && !rc; ++i) {
            rc = kept.restore();
            if (!rc && flush && hipMemsetAsync(flush, i + 1, flush_bytes, st) != hipSuccess) rc = TCFFT_HIP_ERROR;
            if (!rc && hipEventRecord(a, st) != hipSuccess) rc = TCFFT_HIP_ERROR;
            if (!rc) rc = tcfft_multi_exec(plan, data, TCFFT_FORWARD, stream);
            if (!rc && hipEventRecord(b, st) != hipSuccess) rc = TCFFT_HIP_ERROR;
            if (!rc && hipEventSynchronize(b) != hipSuccess) rc = TCFFT_HIP_ERROR;
            float t = 0.f;
            if (!rc && hipEventElapsedTime(&t, a, b) != hipSuccess) rc = TCFFT_HIP_ERROR;
            total += t;
        }
        ms = total / 5.f;
    };
    auto apply = [&](const Cand& c) {
        if (!rc) rc = tcfft_multi_set_schedule(plan, c.grid, c.order);
        plan->delay = c.delay;
    };
    // every (task order, grid, start delay) once
    for (int order = 0; order < 3 && !rc; ++order)
        for (int gsz : grids)
            for (int delay = 0; delay <= 2 && !rc; ++delay) {
                Cand c{gsz, order, delay, 0.f};
                apply(c);
                time_current(c.ms);
                if (!rc) cands.push_back(c);
            }
    // the four fastest again, three rounds in turn, each keeping its best
    // round: one sweep's timings differ by several percent between
    // neighbouring candidates, enough to pick a slower schedule
    if (!rc) {
        std::sort(cands.begin(), cands.end(), [](const Cand& x, const Cand& y) { return x.ms < y.ms; });
        if (cands.size() > 4) cands.resize(4);
        for (int round = 0; round < 3 && !rc; ++round)
            for (Cand& c : cands) {
                float ms = 0.f;
                apply(c);
                time_current(ms);
                if (!rc) c.ms = std::min(c.ms, ms);
            }
    }
    float best = 1e30f;
    int bg = cu, bo = 0, bd = 0;
    for (const Cand& c : cands)
        if (c.ms < best) {
            best = c.ms;
            bg = c.grid;
            bo = c.order;
            bd = c.delay;
        }
    if (flush) (void)hipFree(flush);
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    if (rc) return rc;
    rc = tcfft_multi_set_schedule(plan, bg, bo);
    plan->delay = bd;
    if (best_grid) *best_grid = bg;
    if (best_order) *best_order = bo;
    if (best_ms) *best_ms = best;
    return rc;
}

}  // extern "C"

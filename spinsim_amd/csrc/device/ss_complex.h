// Complex float64 scalars and d x d (d = 2, 3) matrices held in registers.
// Shared by the hipRTC-compiled integrator and the ahead-of-time kernels.
#pragma once

struct ss_cd {
    double x, y;
};

static __host__ __device__ __forceinline__ ss_cd ss_c(double x, double y)
{
    ss_cd r;
    r.x = x;
    r.y = y;
    return r;
}
static __device__ __forceinline__ ss_cd ss_mul(ss_cd a, ss_cd b)
{
    return ss_c(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
static __device__ __forceinline__ ss_cd ss_conj(ss_cd a) { return ss_c(a.x, -a.y); }
static __device__ __forceinline__ ss_cd ss_add(ss_cd a, ss_cd b) { return ss_c(a.x + b.x, a.y + b.y); }
static __device__ __forceinline__ ss_cd ss_sub(ss_cd a, ss_cd b) { return ss_c(a.x - b.x, a.y - b.y); }
static __device__ __forceinline__ ss_cd ss_scale(ss_cd a, double s) { return ss_c(a.x * s, a.y * s); }
// acc + a*b as four fused multiply-adds
static __device__ __forceinline__ ss_cd ss_mac(ss_cd acc, ss_cd a, ss_cd b)
{
    acc.x = fma(a.x, b.x, acc.x);
    acc.x = fma(-a.y, b.y, acc.x);
    acc.y = fma(a.x, b.y, acc.y);
    acc.y = fma(a.y, b.x, acc.y);
    return acc;
}

template <int D>
static __device__ __forceinline__ void ss_set_identity(ss_cd m[D][D])
{
#pragma unroll
    for (int r = 0; r < D; ++r)
#pragma unroll
        for (int c = 0; c < D; ++c) m[r][c] = ss_c(r == c ? 1.0 : 0.0, 0.0);
}

template <int D>
static __device__ __forceinline__ void ss_copy(const ss_cd a[D][D], ss_cd out[D][D])
{
#pragma unroll
    for (int r = 0; r < D; ++r)
#pragma unroll
        for (int c = 0; c < D; ++c) out[r][c] = a[r][c];
}

// out = a * b, each entry summed in k order.  The k loop is outermost so
// consecutive fused multiply-adds update different entries: a single wave
// then issues back to back without waiting on its own results.
template <int D>
static __device__ __forceinline__ void ss_matmul(const ss_cd a[D][D], const ss_cd b[D][D], ss_cd out[D][D])
{
#pragma unroll
    for (int r = 0; r < D; ++r)
#pragma unroll
        for (int c = 0; c < D; ++c) out[r][c] = ss_mul(a[r][0], b[0][c]);
#pragma unroll
    for (int k = 1; k < D; ++k)
#pragma unroll
        for (int r = 0; r < D; ++r)
#pragma unroll
            for (int c = 0; c < D; ++c) out[r][c] = ss_mac(out[r][c], a[r][k], b[k][c]);
}

// u <- e * u
template <int D>
static __device__ __forceinline__ void ss_left_multiply(const ss_cd e[D][D], ss_cd u[D][D])
{
    ss_cd t[D][D];
    ss_matmul<D>(e, u, t);
    ss_copy<D>(t, u);
}

// u <- u * e
template <int D>
static __device__ __forceinline__ void ss_right_multiply(ss_cd u[D][D], const ss_cd e[D][D])
{
    ss_cd t[D][D];
    ss_matmul<D>(u, e, t);
    ss_copy<D>(t, u);
}

// out = m v
template <int D>
static __device__ __forceinline__ void ss_matvec(const ss_cd m[D][D], const ss_cd v[D], ss_cd out[D])
{
#pragma unroll
    for (int r = 0; r < D; ++r) {
        ss_cd acc = ss_mul(m[r][0], v[0]);
#pragma unroll
        for (int k = 1; k < D; ++k) acc = ss_mac(acc, m[r][k], v[k]);
        out[r] = acc;
    }
}

#ifndef SS_HOST
// Moves of a wave's inclusive scan by data-parallel primitives: a lane takes a
// value from s lanes before it in its row of 16 (row_shr), from the last lane of
// the row before (row_bcast:15) or of the first half (row_bcast:31).  They are
// register moves at the rate of any other vector instruction, where a shuffle
// goes through the LDS crossbar, which the four waves of a workgroup share: 36
// of them a step for a spin-one matrix took longer than its product.  Scans of
// 1e5 spin-one rows: 18.7 -> 16.1 us (one simulation), 1.35e5 in a batch 40.1 ->
// 32.9; 2.6e5 spin-half rows 15.9 -> 14.1 and 31.5 -> 28.0.
#define SS_DPP_ROW_SHR(s) (0x110 + (s))
#define SS_DPP_WAVE_SHR1 0x138
#define SS_DPP_ROW_BCAST15 0x142
#define SS_DPP_ROW_BCAST31 0x143

// (lanes without a source get 0)
template <int CTRL>
static __device__ __forceinline__ double ss_dpp(double x)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

template <int D, int CTRL>
static __device__ __forceinline__ void ss_dpp_mat(const ss_cd m[D][D], ss_cd out[D][D])
{
#pragma unroll
    for (int r = 0; r < D; ++r)
#pragma unroll
        for (int c = 0; c < D; ++c) out[r][c] = ss_c(ss_dpp<CTRL>(m[r][c].x), ss_dpp<CTRL>(m[r][c].y));
}

// step(control, applies) for each step of an inclusive scan over the first
// `count` lanes (uniform; the lanes from there on are left with products of
// theirs): x_l <- x_l o x_source where `applies`, after which lane l holds
// x_l o ... o x_0.
template <int CTRL> struct ss_dpp_ctrl {
    static constexpr int value = CTRL;
};
template <class Step>
static __device__ __forceinline__ void ss_scan_steps(int lane, int count, Step step)
{
    if (count > 1) step(ss_dpp_ctrl<SS_DPP_ROW_SHR(1)>(), (lane & 15) >= 1);
    if (count > 2) step(ss_dpp_ctrl<SS_DPP_ROW_SHR(2)>(), (lane & 15) >= 2);
    if (count > 4) step(ss_dpp_ctrl<SS_DPP_ROW_SHR(4)>(), (lane & 15) >= 4);
    if (count > 8) step(ss_dpp_ctrl<SS_DPP_ROW_SHR(8)>(), (lane & 15) >= 8);
    if (count > 16) step(ss_dpp_ctrl<SS_DPP_ROW_BCAST15>(), (lane & 16) != 0);
    if (count > 32) step(ss_dpp_ctrl<SS_DPP_ROW_BCAST31>(), (lane & 32) != 0);
}

// q_l <- q_l q_{l-1} ... q_0 over the first `count` lanes of a wave.
template <int D>
static __device__ __forceinline__ void ss_wave_scan(ss_cd q[D][D], int lane, int count)
{
    ss_scan_steps(lane, count, [&](auto ctrl, bool applies) {
        ss_cd p[D][D];
        ss_dpp_mat<D, decltype(ctrl)::value>(q, p);
        if (applies) ss_right_multiply<D>(q, p);
    });
}
#endif

// Training-mode kernels for gfx950: relaxed forward, backward_w, backward_x.
//
// Layout: activations are feature-major [features, batch]; lanes run along the batch so that
// every gathered row segment is one coalesced access (16 bytes per lane where the batch length
// and the base addresses allow it).  Everything indexed by the neuron (connection indices, the
// 16 gate weights) is wave-uniform and read through the scalar cache.
//
// The mixture of the 16 relaxed gates is bilinear in (a, b).  With
//     P_st = sum_i w_i * [gate i is true at (s, t)]            (four sums of eight weights)
// it is  y = (1-a)(1-b) P00 + (1-a) b P01 + a (1-b) P10 + a b P11, evaluated as two
// interpolations along b followed by one along a.
#include <hip/hip_fp16.h>

#include "dl_common.h"

namespace {

template <typename T> struct Acc { typedef float type; };
template <> struct Acc<double> { typedef double type; };

// VEC consecutive elements of a row.  RAG: the rows are not whole vectors (or a base address is not aligned to one), so a
// vector is only aligned to its elements; the hardware takes such loads and stores as they are, whole (dwordx4).
template <typename T, int N, bool RAG = false> struct alignas(RAG ? sizeof(T) : sizeof(T) * N) Pack { T v[N]; };

// Rows of `batch` elements are read and written as vectors 0 .. ceil(batch / VEC) - 1.  RAG: the last vector of a row is
// moved back to end with the row, so it repeats `dup` elements of the vector before it.  Elementwise results are then
// written twice with the same value (the conversion to half by round_fma, which does not depend on an element's place in
// its vector); sums over the batch leave the repeated elements out (own_part).  What that buys
// over one element per lane: half rows of 500 elements on six 64000-wide layers, forward + backward 2.11 -> 0.61 ms.
template <int VEC> __device__ __forceinline__ int64_t vec_count(int64_t batch) {
    return (int64_t) ((uint64_t) (batch + VEC - 1) / VEC);
}
template <int VEC, bool RAG> __device__ __forceinline__ int64_t vec_at(int64_t col, int64_t batch) {
    const int64_t at = col * VEC;
    return RAG && at + VEC > batch ? batch - VEC : at;
}
template <int VEC, bool RAG> __device__ __forceinline__ int vec_dup(int64_t col, int64_t batch) {
    return RAG && col * VEC + VEC > batch ? (int) (col * VEC + VEC - batch) : 0;
}
template <bool RAG, typename C> __device__ __forceinline__ C own_part(C g, int e, int dup) {
    return RAG && e < dup ? (C) 0 : g;
}
// Vector `col` of row `row` (whole rows are addressed in vectors: one shift less per access, 2 % of a one-pass backward).
template <typename P, int VEC, bool RAG, typename T>
__device__ __forceinline__ const P &row_vec(const T *base, int64_t row, int64_t batch, int64_t ncols, int64_t col) {
    if constexpr (RAG) return *reinterpret_cast<const P *>(base + row * batch + vec_at<VEC, RAG>(col, batch));
    else return reinterpret_cast<const P *>(base)[row * ncols + col];
}
template <typename P, int VEC, bool RAG, typename T>
__device__ __forceinline__ P &row_vec(T *base, int64_t row, int64_t batch, int64_t ncols, int64_t col) {
    return const_cast<P &>(row_vec<P, VEC, RAG>(const_cast<const T *>(base), row, batch, ncols, col));
}

// A vector read past the caches (NT: the row will not be read again soon, so it takes no place in the Infinity Cache).
template <bool NT, typename P> __device__ __forceinline__ P load_vec(const P &at) {
    if constexpr (!NT) {
        return at;
    } else {
        constexpr size_t A = alignof(P) < 4 ? 2 : 4;
        typedef std::conditional_t<A == 2, uint16_t, uint32_t> E;
        typedef E V __attribute__((ext_vector_type(sizeof(P) / A), aligned(alignof(P))));
        return __builtin_bit_cast(P, __builtin_nontemporal_load(reinterpret_cast<const V *>(&at)));
    }
}

// Vector `col` of row `row` of a matrix of short rows, zeros where the row has no such vector, by every lane and without a
// branch: behind one the compiler cannot count the loads in flight, and waits for all of them.  Whole rows are read through a
// buffer resource that ends with the row: nothing is fetched, and zeros come back, where `valid` (wave-uniform) is false.
// RAG: lanes past the row read its last vector; `row` must be there, and `valid` is the caller's to apply.
template <typename P, int VEC, bool RAG, bool NT, typename T>
__device__ __forceinline__ P row_part(const T *base, int64_t row, bool valid, int64_t batch, int64_t ncols, int64_t col) {
    if constexpr (RAG) {
        P v = load_vec<NT>(row_vec<P, VEC, RAG>(base, row, batch, ncols, col));
#pragma unroll
        for (int e = 0; e < VEC; ++e) v.v[e] = col < ncols ? v.v[e] : (T) 0;
        return v;
    } else {
        static_assert(sizeof(P) == 16 || sizeof(P) == 8, "one buffer load per vector");
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T *>(base + row * batch), 0, valid ? (int) (batch * (int64_t) sizeof(T)) : 0, 0x00027000);
        const int at = (int) col * (int) sizeof(P);
        constexpr int policy = NT ? 2 : 0;
        if constexpr (sizeof(P) == 16) return __builtin_bit_cast(P, __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, 0, policy));
        else return __builtin_bit_cast(P, __builtin_amdgcn_raw_buffer_load_b64(rsrc, at, 0, policy));
    }
}

template <typename T> __device__ __forceinline__ typename Acc<T>::type up(T v) { return (typename Acc<T>::type) v; }
template <> __device__ __forceinline__ float up<__half>(__half v) { return __half2float(v); }
template <typename T, typename C> __device__ __forceinline__ T down(C v) { return (T) v; }
template <> __device__ __forceinline__ __half down<__half, float>(float v) { return __float2half(v); }
template <typename T> __device__ __forceinline__ T from_double(double v) {
    if constexpr (sizeof(T) == 2) return __builtin_bit_cast(T, (_Float16) v);        // (not by way of float)
    else return (T) v;
}

__device__ __forceinline__ float dl_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double dl_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// fma(a, b, c) as a T, and v * s as a T.  Left to itself the compiler folds the conversion to half into the multiply-add
// for some elements of a vector (v_fma_mixlo_f16: one rounding) and not for others (two); ONCE says which it is: one
// rounding for every element, as the kernels that take one element per lane have it.
template <typename T, bool ONCE, typename C> __device__ __forceinline__ T round_fma(C a, C b, C c) {
    if constexpr (ONCE && sizeof(T) == 2) {
        uint32_t r;                                              // (the instruction writes the low half)
        asm("v_fma_mixlo_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
        return __builtin_bit_cast(T, (uint16_t) r);
    } else {
        return down<T, C>(dl_fma(a, b, c));
    }
}
template <typename T, bool ONCE, typename C> __device__ __forceinline__ T round_scaled(C v, C s) {
    if constexpr (ONCE && sizeof(T) == 2) return round_fma<T, ONCE, C>(v, s, (C) -0.0);      // (keeps the sign of a zero)
    else return down<T, C>(v * s);
}

// Gate weights (probabilities or logits) and their gradients sit next to activations of type T either in T as well
// or, `w32`, in fp32 whatever T is: what a layer with fp32 weights needs for half / double activations (the
// reference's --training-bit-count 16 / 64).  The pointers keep the type T* and are reinterpreted.
template <typename T> __device__ __forceinline__ typename Acc<T>::type wload(const T *__restrict__ w, int64_t at, bool w32) {
    typedef typename Acc<T>::type C;
    if constexpr (sizeof(T) == sizeof(float)) return w[at];
    else return w32 ? (C) reinterpret_cast<const float *>(w)[at] : up<T>(w[at]);
}
template <bool NT, typename E> __device__ __forceinline__ void store_elem(E *at, E v) {
    typedef std::conditional_t<sizeof(E) == 2, uint16_t, std::conditional_t<sizeof(E) == 4, uint32_t, uint64_t>> U;
    if constexpr (NT) __builtin_nontemporal_store(__builtin_bit_cast(U, v), reinterpret_cast<U *>(at));
    else *at = v;
}
// (NT: past the Infinity Cache, as load_vec)
template <typename T, bool NT = false>
__device__ __forceinline__ void wstore(T *__restrict__ w, int64_t at, typename Acc<T>::type v, bool w32) {
    typedef typename Acc<T>::type C;
    if constexpr (sizeof(T) == sizeof(float)) store_elem<NT, T>(w + at, v);
    else if (w32) store_elem<NT>(reinterpret_cast<float *>(w) + at, (float) v);
    else store_elem<NT>(w + at, down<T, C>(v));
}

// y = lerp(lerp(P00, P01, b), lerp(P10, P11, b), a), three fused multiply-adds.
template <typename T, bool ONCE, typename C> __device__ __forceinline__ T mix(C av, C bv, C p00, C p10, C d0, C d1) {
    const C lo = dl_fma(bv, d0, p00);
    const C hi = dl_fma(bv, d1, p10);
    return round_fma<T, ONCE, C>(av, hi - lo, lo);
}

// The four corner values of neuron n's gate mixture.
template <typename C> struct Corners { C p00, p01, p10, p11; };

template <typename C> __device__ __forceinline__ Corners<C> corners_of(const C (&g)[16]) {
    Corners<C> c;
    c.p00 = ((g[8] + g[9]) + (g[10] + g[11])) + ((g[12] + g[13]) + (g[14] + g[15]));
    c.p01 = ((g[4] + g[5]) + (g[6] + g[7])) + ((g[12] + g[13]) + (g[14] + g[15]));
    c.p10 = ((g[2] + g[3]) + (g[6] + g[7])) + ((g[10] + g[11]) + (g[14] + g[15]));
    c.p11 = ((g[1] + g[3]) + (g[5] + g[7])) + ((g[9] + g[11]) + (g[13] + g[15]));
    return c;
}

template <typename T>
__device__ __forceinline__ Corners<typename Acc<T>::type> corners(const T *__restrict__ w, int64_t n, bool w32) {
    typedef typename Acc<T>::type C;
    C g[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) g[i] = wload<T>(w, n * 16 + i, w32);
    return corners_of<C>(g);
}

// ------------------------------------------------------------------------------------------
// Wave-wide sums with a fixed association order (deterministic).
// ------------------------------------------------------------------------------------------
template <int CTRL> __device__ __forceinline__ float dpp_f32(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

__device__ __forceinline__ float lane_value(float v, int i) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}

__device__ __forceinline__ double lane_value(double v, int i) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t) __builtin_amdgcn_readlane((int) (uint32_t) u, i);
    const uint32_t hi = (uint32_t) __builtin_amdgcn_readlane((int) (uint32_t) (u >> 32), i);
    return __builtin_bit_cast(double, ((uint64_t) hi << 32) | lo);
}

// Wave-wide sums of FOUR values at once, each replaced by its total (wave-uniform).  A butterfly
// that halves the number of live values at each of its first two steps: after exchanging with
// lane ^ 1 a lane keeps the first or the second value of each pair, after lane ^ 2 it keeps one
// value, index lane & 3, summed over its quad; the quads of a 16-lane row are then added with
// row rotations (which keep lane & 3), rows 0+1 and 2+3 with v_permlane16_swap and the two
// halves with v_permlane32_swap (gfx950).  19 vector instructions instead of 44 for four
// separate reductions; the order of the additions is fixed.
__device__ __forceinline__ float swap_add16(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);     // rows (0,0,2,2) and (1,1,3,3)
    return __builtin_bit_cast(float, (unsigned) r[0]) + __builtin_bit_cast(float, (unsigned) r[1]);
}

__device__ __forceinline__ float swap_add32(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);     // lower half twice, upper half twice
    return __builtin_bit_cast(float, (unsigned) r[0]) + __builtin_bit_cast(float, (unsigned) r[1]);
}

// (in every lane the total of value lane & 3)
__device__ __forceinline__ float wave_sum4_lane(float s0, float s1, float s2, float s3, int lane) {
    const bool odd = lane & 1, high = lane & 2;
    const float x = (odd ? s1 : s0) + dpp_f32<0xB1>(odd ? s0 : s1);          // quad_perm [1,0,3,2]: lane ^ 1
    const float y = (odd ? s3 : s2) + dpp_f32<0xB1>(odd ? s2 : s3);
    float z = (high ? y : x) + dpp_f32<0x4E>(high ? x : y);                  // quad_perm [2,3,0,1]: lane ^ 2
    z += dpp_f32<0x124>(z);                                                  // row_ror:4
    z += dpp_f32<0x128>(z);                                                  // row_ror:8
    return swap_add32(swap_add16(z));
}

__device__ __forceinline__ void wave_sum4(float &s0, float &s1, float &s2, float &s3, int lane) {
    const float z = wave_sum4_lane(s0, s1, s2, s3, lane);
    s0 = lane_value(z, 0);
    s1 = lane_value(z, 1);
    s2 = lane_value(z, 2);
    s3 = lane_value(z, 3);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int m = 1; m < DL_WAVE; m <<= 1) v += __shfl_xor(v, m, DL_WAVE);
    return v;
}

__device__ __forceinline__ void wave_sum4(double &s0, double &s1, double &s2, double &s3, int) {
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    s3 = wave_sum(s3);
}

__device__ __forceinline__ double wave_sum4_lane(double s0, double s1, double s2, double s3, int lane) {
    wave_sum4(s0, s1, s2, s3, lane);
    return (lane & 2) ? ((lane & 1) ? s3 : s2) : ((lane & 1) ? s1 : s0);
}

// The value of lane I of the lane's 16-lane row (wave_sum4_lane: one of four sums; the quads of a row add in different orders).
template <int I> __device__ __forceinline__ float row_value(float v) { return dpp_f32<0x150 + I>(v); }         // row_newbcast
template <int I> __device__ __forceinline__ double row_value(double v) { return __shfl(v, (dl_lane() & ~15) | I, DL_WAVE); }

// Sum over each aligned group of 16 lanes, result in every lane of the group.
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_f32<0xB1>(v);
    v += dpp_f32<0x4E>(v);
    v += dpp_f32<0x141>(v);
    v += dpp_f32<0x140>(v);
    return v;
}

__device__ __forceinline__ double row16_sum(double v) {
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) v += __shfl_xor(v, m, DL_WAVE);
    return v;
}

__device__ __forceinline__ float dl_exp(float v) { return expf(v); }
__device__ __forceinline__ double dl_exp(double v) { return exp(v); }

__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp_f32<0xB1>(v));
    v = fmaxf(v, dpp_f32<0x4E>(v));
    v = fmaxf(v, dpp_f32<0x141>(v));
    v = fmaxf(v, dpp_f32<0x140>(v));
    return v;
}

__device__ __forceinline__ double row16_max(double v) {
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) v = fmax(v, __shfl_xor(v, m, DL_WAVE));
    return v;
}

// Row of the gradient matrix that belongs to neuron n.  gdiv == 0: grad_y is [out_dim, batch] and
// the row is n.  gdiv > 0: the layer feeds a GroupSum and grad_y is its [k, batch] gradient (already
// divided by tau): all gdiv = out_dim / k neurons of a class share one row, and the broadcast
// [out_dim, batch] matrix is never materialised.
__device__ __forceinline__ int64_t grad_row(int64_t n, int64_t gdiv) {
    return gdiv ? (int64_t) ((uint32_t) n / (uint32_t) gdiv) : n;
}

// What a kernel makes of the [out, 16] weights: gate probabilities as they are (0, false), the softmax of logits (1, true),
// or all of the argmax gate (the discretised net on float inputs; taken here instead of in four torch launches per layer
// that make a one-hot matrix: 784 -> 6 x 64000, batch 1000: 834 -> 705 us).
constexpr int GATES_LOGITS = 1, GATES_ARGMAX = 2;

// Corner coefficients of FOUR neurons at once: the 16-lane row r of the wave works on neuron n[r]
// (n[r] < 0: none), lane i of the row on gate i.  LOGITS (GATES_LOGITS): `w` holds logits, the row computes their
// softmax (and stores it to `probs` if asked); otherwise `w` holds the probabilities.  The corner
// sums are masked row sums whose association order is that of corners_of(), so the results are
// bit-identical to it.  Returns, per neuron, the wave-uniform P00, P10, P01 - P00, P11 - P10.
template <typename T, int GATES, bool NT = false>
__device__ __forceinline__ void corners4(const T *__restrict__ w, const int32_t (&n)[4], int lane, bool store_probs,
                                         T *__restrict__ probs, typename Acc<T>::type (&p00)[4],
                                         typename Acc<T>::type (&p10)[4], typename Acc<T>::type (&d0)[4],
                                         typename Acc<T>::type (&d1)[4], bool w32 = false) {
    typedef typename Acc<T>::type C;
    const int row = lane >> 4, gate = lane & 15;
    const int32_t mine = row == 0 ? n[0] : row == 1 ? n[1] : row == 2 ? n[2] : n[3];
    const bool valid = mine >= 0;
    const int64_t at = (int64_t) (valid ? mine : 0) * 16 + gate;
    C p = wload<T>(w, at, w32);
    if (GATES == GATES_LOGITS) {
        const C e = dl_exp(p - row16_max(p));
        p = e / row16_sum(e);
        if (store_probs && valid) wstore<T, NT>(probs, at, p, w32);
    } else if (GATES == GATES_ARGMAX) {
        // as argmax: the first of the largest, a NaN above every number (row16_max passes NaNs over)
        const uint32_t nans = (uint32_t) (__ballot(p != p) >> (16 * row)) & 0xffffu;
        const uint32_t tops = (uint32_t) (__ballot(p == row16_max(p)) >> (16 * row)) & 0xffffu;
        p = gate == __ffs((int) (nans ? nans : tops)) - 1 ? (C) 1 : (C) 0;
    }
    const C zero = (C) 0;
    const C q00 = row16_sum((gate & 8) ? p : zero), q01 = row16_sum((gate & 4) ? p : zero);
    const C q10 = row16_sum((gate & 2) ? p : zero), q11 = row16_sum((gate & 1) ? p : zero);
    const C e0 = q01 - q00, e1 = q11 - q10;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        p00[i] = lane_value(q00, 16 * i);
        p10[i] = lane_value(q10, 16 * i);
        d0[i] = lane_value(e0, 16 * i);
        d1[i] = lane_value(e1, 16 * i);
    }
}

// ------------------------------------------------------------------------------------------
// forward: one wave = NPW neurons x 64 vectors of the batch.
// ------------------------------------------------------------------------------------------
// LOGITS: `w` holds the raw gate logits; the kernel applies the softmax itself and (column tile 0
// only) stores the probabilities to `probs` for the backward pass.
template <typename T, int VEC, int NPW, int GATES, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void forward_kernel(const T *__restrict__ x, const int64_t *__restrict__ a,
                                                           const int64_t *__restrict__ b, const T *__restrict__ w,
                                                           T *__restrict__ y, T *__restrict__ probs, int64_t out_dim,
                                                           int64_t batch, bool w32) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t n0 = ((int64_t) blockIdx.x * 4 + wave) * NPW;
    if (n0 >= out_dim) return;
    const int64_t ncols = vec_count<VEC>(batch);

    static_assert(NPW == 4, "corners4 serves four neurons per wave");
    int64_t ia[NPW], ib[NPW];
    C p00[NPW], p10[NPW], d0[NPW], d1[NPW];
    int32_t ids[NPW];
#pragma unroll
    for (int j = 0; j < NPW; ++j) {
        const int64_t n = (n0 + j < out_dim) ? n0 + j : out_dim - 1;
        ia[j] = a[n];
        ib[j] = b[n];
        ids[j] = n0 + j < out_dim ? (int32_t) (n0 + j) : -1;
    }
    corners4<T, GATES>(w, ids, lane, blockIdx.y == 0, probs, p00, p10, d0, d1, w32);
    for (int64_t col = (int64_t) blockIdx.y * DL_WAVE + lane; col < ncols; col += (int64_t) gridDim.y * DL_WAVE) {
        P va[NPW], vb[NPW];
#pragma unroll
        for (int j = 0; j < NPW; ++j) {
            va[j] = row_vec<P, VEC, RAG>(x, ia[j], batch, ncols, col);
            vb[j] = row_vec<P, VEC, RAG>(x, ib[j], batch, ncols, col);
        }
#pragma unroll
        for (int j = 0; j < NPW; ++j) {
            if (n0 + j < out_dim) {
                P r;
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    r.v[e] = mix<T, RAG, C>(up<T>(va[j].v[e]), up<T>(vb[j].v[e]), p00[j], p10[j], d0[j], d1[j]);
                }
                row_vec<P, VEC, RAG>(y, (n0 + j), batch, ncols, col) = r;
            }
        }
    }
}

// Lane i < 16 holds gate i: its gradient is the sum of the corner sums at which gate i is true.
// probs != nullptr chains the softmax backward, p_i * (g_i - sum_j p_j g_j).  Called by whole
// waves (the 16-lane row sum needs every lane).
template <typename T>
__device__ __forceinline__ void store_grad_w(int lane, bool neuron_valid, int64_t n, typename Acc<T>::type s00,
                                             typename Acc<T>::type s01, typename Acc<T>::type s10,
                                             typename Acc<T>::type s11, const T *__restrict__ probs,
                                             T *__restrict__ gw, bool w32 = false) {
    typedef typename Acc<T>::type C;
    const bool valid = lane < 16 && neuron_valid;
    C r = (C) 0;
    if (lane & 8) r += s00;
    if (lane & 4) r += s01;
    if (lane & 2) r += s10;
    if (lane & 1) r += s11;
    if (probs != nullptr) {
        const C p = valid ? wload<T>(probs, n * 16 + lane, w32) : (C) 0;
        const C dot = row16_sum(p * r);
        r = p * (r - dot);
    }
    if (valid) wstore<T>(gw, n * 16 + lane, r, w32);
}

// The same for four neurons at once: the 16-lane row r of the wave holds neuron r's sums as wave_sum4_lane leaves them and, in
// `p`, its probabilities (read only with `softmax`).  Same values, same order of additions.
template <typename T, bool NT>
__device__ __forceinline__ void store_grad_w4(int lane, bool valid, int64_t n, typename Acc<T>::type sums,
                                              typename Acc<T>::type p, bool softmax, T *__restrict__ gw, bool w32) {
    typedef typename Acc<T>::type C;
    const C s00 = row_value<0>(sums), s01 = row_value<1>(sums), s10 = row_value<2>(sums), s11 = row_value<3>(sums);
    C r = (C) 0;
    if (lane & 8) r += s00;
    if (lane & 4) r += s01;
    if (lane & 2) r += s10;
    if (lane & 1) r += s11;
    if (softmax) {
        const C dot = row16_sum(p * r);
        r = p * (r - dot);
    }
    if (valid) wstore<T, NT>(gw, n * 16 + (lane & 15), r, w32);
}

// ------------------------------------------------------------------------------------------
// backward_w: per neuron, the four corner-weighted batch sums
//     S_st = sum_r g[r] * a^s (1-a)^(1-s) * b^t (1-b)^(1-t)
// and grad_w[n, i] = sum of the S_st at which gate i is true.
// WPN = waves that share one neuron's batch (1: a wave owns NPW neurons; 4: the workgroup's
// four waves split the batch of NPW neurons and combine through LDS in wave order).
// ------------------------------------------------------------------------------------------
// probs != nullptr: chain the softmax backward, gw[n,i] = p_i * (g_i - sum_j p_j g_j), i.e. the
// gradient with respect to the logits that `probs` (forward_kernel's LOGITS output) came from.
template <typename T, int VEC, int NPW, int WPN, bool RAG>
__device__ __forceinline__ void backward_w_block(int64_t block, typename Acc<T>::type (*partial)[NPW][4],
                                                 const T *__restrict__ x, const int64_t *__restrict__ a,
                                                 const int64_t *__restrict__ b, const T *__restrict__ gy,
                                                 const T *__restrict__ probs, T *__restrict__ gw, int64_t out_dim,
                                                 int64_t batch, int64_t gdiv, bool w32) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t n0 = (WPN == 1) ? (block * 4 + wave) * NPW : block * NPW;
    const int part = (WPN == 1) ? 0 : wave;

    C s00[NPW], s01[NPW], s10[NPW], s11[NPW];
#pragma unroll
    for (int j = 0; j < NPW; ++j) s00[j] = s01[j] = s10[j] = s11[j] = (C) 0;

    if (n0 < out_dim) {
        int64_t ia[NPW], ib[NPW], nn[NPW];
#pragma unroll
        for (int j = 0; j < NPW; ++j) {
            const int64_t n = (n0 + j < out_dim) ? n0 + j : out_dim - 1;
            ia[j] = a[n];
            ib[j] = b[n];
            nn[j] = grad_row(n, gdiv);
        }
        for (int64_t base = (int64_t) part * DL_WAVE; base < ncols; base += (int64_t) WPN * DL_WAVE) {
            const int64_t col = base + lane;
            if (col < ncols) {
                const int dup = vec_dup<VEC, RAG>(col, batch);
                P va[NPW], vb[NPW], vg[NPW];
#pragma unroll
                for (int j = 0; j < NPW; ++j) {
                    va[j] = row_vec<P, VEC, RAG>(x, ia[j], batch, ncols, col);
                    vb[j] = row_vec<P, VEC, RAG>(x, ib[j], batch, ncols, col);
                    vg[j] = row_vec<P, VEC, RAG>(gy, nn[j], batch, ncols, col);
                }
#pragma unroll
                for (int j = 0; j < NPW; ++j) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        const C av = up<T>(va[j].v[e]), bv = up<T>(vb[j].v[e]), g = own_part<RAG>(up<T>(vg[j].v[e]), e, dup);
                        const C ga = g * av, gna = g - ga;       // g*a, g*(1-a)
                        const C t11 = ga * bv, t01 = gna * bv;
                        s11[j] += t11;
                        s10[j] += ga - t11;
                        s01[j] += t01;
                        s00[j] += gna - t01;
                    }
                }
            }
        }
    }

#pragma unroll
    for (int j = 0; j < NPW; ++j) {
        wave_sum4(s00[j], s01[j], s10[j], s11[j], lane);
    }

    if (WPN != 1) {
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < NPW; ++j) {
                partial[wave][j][0] = s00[j];
                partial[wave][j][1] = s01[j];
                partial[wave][j][2] = s10[j];
                partial[wave][j][3] = s11[j];
            }
        }
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int j = 0; j < NPW; ++j) {
            s00[j] = (partial[0][j][0] + partial[1][j][0]) + (partial[2][j][0] + partial[3][j][0]);
            s01[j] = (partial[0][j][1] + partial[1][j][1]) + (partial[2][j][1] + partial[3][j][1]);
            s10[j] = (partial[0][j][2] + partial[1][j][2]) + (partial[2][j][2] + partial[3][j][2]);
            s11[j] = (partial[0][j][3] + partial[1][j][3]) + (partial[2][j][3] + partial[3][j][3]);
        }
    }

#pragma unroll
    for (int j = 0; j < NPW; ++j)
        store_grad_w<T>(lane, n0 + j < out_dim, n0 + j, s00[j], s01[j], s10[j], s11[j], probs, gw, w32);
}

template <typename T, int VEC, int NPW, int WPN, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void backward_w_kernel(const T *__restrict__ x, const int64_t *__restrict__ a,
                                                              const int64_t *__restrict__ b,
                                                              const T *__restrict__ gy, const T *__restrict__ probs,
                                                              T *__restrict__ gw, int64_t out_dim, int64_t batch,
                                                              int64_t gdiv, bool w32) {
    __shared__ typename Acc<T>::type partial[4][NPW][4];
    backward_w_block<T, VEC, NPW, WPN, RAG>(blockIdx.x, partial, x, a, b, gy, probs, gw, out_dim, batch, gdiv, w32);
}

// ------------------------------------------------------------------------------------------
// backward_x: one wave = one input row x 64 vectors of the batch; it walks the row's fan-out
// list (reverse index) and gathers, so every grad_x element has a single writer.
//     dy/da = (P10 - P00) + b * ((P11 - P10) - (P01 - P00))
//     dy/db = (P01 - P00) + a * ((P11 - P10) - (P01 - P00))
// A neuron wired twice to this input appears twice in the list; each visit adds half of
// dy/da + dy/db.
// ------------------------------------------------------------------------------------------
template <typename T, int VEC, bool RAG>
__device__ __forceinline__ void backward_x_block(int64_t block, int64_t tile, int64_t tiles, const T *__restrict__ x,
                                                 const int64_t *__restrict__ a, const int64_t *__restrict__ b,
                                                 const T *__restrict__ w, const T *__restrict__ gy,
                                                 const int64_t *__restrict__ start, const int64_t *__restrict__ idx,
                                                 T *__restrict__ gx, int64_t in_dim, int64_t batch,
                                                 typename Acc<T>::type scale, int64_t gdiv, bool w32) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t c = block * 4 + wave;
    if (c >= in_dim) return;
    const int64_t e0 = start[c], e1 = start[c + 1];

    for (int64_t col = tile * DL_WAVE + lane; col < ncols; col += tiles * DL_WAVE) {
        C acc[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = (C) 0;
        for (int64_t e = e0; e < e1; e += 2) {
            // two fan-out entries per trip so that their loads overlap
            const bool two = e + 1 < e1;
            const int64_t nA = idx[e], nB = two ? idx[e + 1] : nA;
            const int64_t iaA = a[nA], ibA = b[nA], iaB = a[nB], ibB = b[nB];
            const bool isaA = iaA == c, isaB = iaB == c;
            const P gA = row_vec<P, VEC, RAG>(gy, grad_row(nA, gdiv), batch, ncols, col), oA = row_vec<P, VEC, RAG>(x, (isaA ? ibA : iaA), batch, ncols, col);
            const P gB = row_vec<P, VEC, RAG>(gy, grad_row(nB, gdiv), batch, ncols, col), oB = row_vec<P, VEC, RAG>(x, (isaB ? ibB : iaB), batch, ncols, col);
            const Corners<C> kA = corners<T>(w, nA, w32), kB = corners<T>(w, nB, w32);
            {
                const C d0 = kA.p01 - kA.p00, d1 = kA.p11 - kA.p10, dd = d1 - d0, da = kA.p10 - kA.p00;
                const C k0 = (isaA && ibA == c) ? (C) 0.5 * (da + d0) : (isaA ? da : d0);
#pragma unroll
                for (int q = 0; q < VEC; ++q) acc[q] += up<T>(gA.v[q]) * (k0 + up<T>(oA.v[q]) * dd);
            }
            if (two) {
                const C d0 = kB.p01 - kB.p00, d1 = kB.p11 - kB.p10, dd = d1 - d0, da = kB.p10 - kB.p00;
                const C k0 = (isaB && ibB == c) ? (C) 0.5 * (da + d0) : (isaB ? da : d0);
#pragma unroll
                for (int q = 0; q < VEC; ++q) acc[q] += up<T>(gB.v[q]) * (k0 + up<T>(oB.v[q]) * dd);
            }
        }
        P r;
#pragma unroll
        for (int q = 0; q < VEC; ++q) r.v[q] = round_scaled<T, RAG, C>(acc[q], scale);
        row_vec<P, VEC, RAG>(gx, c, batch, ncols, col) = r;
    }
}

template <typename T, int VEC, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void backward_x_kernel(const T *__restrict__ x, const int64_t *__restrict__ a,
                                                              const int64_t *__restrict__ b, const T *__restrict__ w,
                                                              const T *__restrict__ gy,
                                                              const int64_t *__restrict__ start,
                                                              const int64_t *__restrict__ idx, T *__restrict__ gx,
                                                              int64_t in_dim, int64_t batch,
                                                              typename Acc<T>::type scale, int64_t gdiv, bool w32) {
    backward_x_block<T, VEC, RAG>(blockIdx.x, blockIdx.y, gridDim.y, x, a, b, w, gy, start, idx, gx, in_dim, batch, scale,
                                  gdiv, w32);
}

// Both gradients of a layer in one launch, the first `x_blocks` workgroups (input rows x column tiles) as
// backward_x_kernel, the others as backward_w_kernel: the two do not depend on each other, and on the small layers that
// have no schedule each takes about as long as its launch and one chain of dependent loads.
// 8000 -> 8000 at batch 128: 6.8 + 3.8 us and a second launch -> 8.0; 30000 -> 30000 at 1024: 91 + 53 -> 138.
template <typename T, int VEC, int NPW, int WPN, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void backward_both_kernel(
    const T *__restrict__ x, const int64_t *__restrict__ a, const int64_t *__restrict__ b, const T *__restrict__ w,
    const T *__restrict__ gy, const T *__restrict__ probs, const int64_t *__restrict__ start,
    const int64_t *__restrict__ idx, T *__restrict__ gw, T *__restrict__ gx, uint32_t row_blocks, uint32_t x_blocks,
    int64_t in_dim, int64_t out_dim, int64_t batch, typename Acc<T>::type scale, int64_t gdiv, bool w32) {
    __shared__ typename Acc<T>::type partial[4][NPW][4];
    if (blockIdx.x < x_blocks)
        backward_x_block<T, VEC, RAG>(blockIdx.x % row_blocks, blockIdx.x / row_blocks, x_blocks / row_blocks, x, a, b, w, gy,
                                      start, idx, gx, in_dim, batch, scale, gdiv, w32);
    else
        backward_w_block<T, VEC, NPW, WPN, RAG>(blockIdx.x - x_blocks, partial, x, a, b, gy, probs, gw, out_dim, batch, gdiv,
                                                w32);
}

// ------------------------------------------------------------------------------------------
// Chained forward / backward_w.  The layer's neurons are walked along the trails of an
// evaluation schedule (schedule.cpp): step s brings in input row verts[s + 1] and evaluates
// neuron[s] from (verts[s], verts[s + 1]); flip[s] tells which of the two is the neuron's `a`
// input.  The shared row stays in registers, so a neuron costs one gathered row instead of two.
// Arithmetic and summation order per element are those of the unchained kernels: the fp32 and
// fp64 results are bit-identical, and so are half results on rows that end inside a vector (on rows of whole vectors
// they can differ in the last bit, where the compiler folds the final conversion into a fused multiply-add in one
// kernel and not in the other).
// ------------------------------------------------------------------------------------------
template <typename T, int VEC, int CHUNK, int GATES, bool RAG, bool NT>
__global__ __launch_bounds__(DL_BLOCK) void forward_chain_kernel(const T *__restrict__ x,
                                                                 const int32_t *__restrict__ verts,
                                                                 const int32_t *__restrict__ neuron,
                                                                 const uint8_t *__restrict__ flip,
                                                                 const T *__restrict__ w, T *__restrict__ y,
                                                                 T *__restrict__ probs, int64_t nchunks, int64_t batch,
                                                                 bool w32) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t c = (int64_t) blockIdx.x * 4 + wave;
    if (c >= nchunks) return;
    static_assert(CHUNK % 4 == 0, "neurons are served four at a time");
    const int64_t s0 = c * CHUNK;

    for (int64_t ct = blockIdx.y; ct * DL_WAVE < ncols; ct += gridDim.y) {
        const int64_t col = ct * DL_WAVE + lane;
        const bool live = col < ncols;
        const int64_t cl = live ? col : 0;
        // every row of the chunk is requested before the first one is used
        P rows[CHUNK + 1];
#pragma unroll
        for (int j = 0; j <= CHUNK; ++j)
            rows[j] = load_vec<NT>(row_vec<P, VEC, RAG>(x, (int64_t) verts[s0 + j], batch, ncols, cl));
#pragma unroll
        for (int j0 = 0; j0 < CHUNK; j0 += 4) {
            int32_t n[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) n[i] = neuron[s0 + j0 + i];
            C p00[4], p10[4], d0[4], d1[4];
            corners4<T, GATES, NT>(w, n, lane, ct == 0, probs, p00, p10, d0, d1, w32);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = j0 + i;
                const bool f = flip[s0 + j] != 0;
                P r;
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const C u0 = up<T>(rows[j].v[e]), u1 = up<T>(rows[j + 1].v[e]);
                    r.v[e] = mix<T, RAG, C>(f ? u1 : u0, f ? u0 : u1, p00[i], p10[i], d0[i], d1[i]);
                }
                if (live && n[i] >= 0) row_vec<P, VEC, RAG>(y, (int64_t) n[i], batch, ncols, cl) = r;
            }
        }
    }
}

// forward_chain_kernel for a layer whose input is the output of the layer below, with that output
// recomputed instead of read: input row v = forward of neuron v of the lower layer, from lower input
// rows low_a[v], low_b[v] of `lx` (a small matrix that stays in the L2 caches) and its gate weights
// (LOGITS: logits, whose softmax goes to `lprobs`).  Values and rounding are those of forward_kernel
// on the lower layer, so the result equals running the two layers one after the other bit for bit,
// but the activation between them is neither written nor read.
template <typename T, int VEC, int CHUNK, bool LOGITS, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void forward_chain_lower_kernel(
    const T *__restrict__ lx, const int64_t *__restrict__ low_a, const int64_t *__restrict__ low_b,
    const T *__restrict__ lw, T *__restrict__ lprobs, const int32_t *__restrict__ verts,
    const int32_t *__restrict__ neuron, const uint8_t *__restrict__ flip, const T *__restrict__ w, T *__restrict__ y,
    T *__restrict__ probs, int64_t nchunks, int64_t batch) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t c = (int64_t) blockIdx.x * 4 + wave;
    if (c >= nchunks) return;
    static_assert(CHUNK % 4 == 0, "neurons are served four at a time");
    const int64_t s0 = c * CHUNK;

    // corner coefficients of the chunk's CHUNK + 1 lower neurons and CHUNK neurons, once for all column tiles
    constexpr int NV = CHUNK + 4;
    int32_t v[NV], n[CHUNK];
    C lp00[NV], lp10[NV], ld0[NV], ld1[NV], p00[CHUNK], p10[CHUNK], d0[CHUNK], d1[CHUNK];
#pragma unroll
    for (int j0 = 0; j0 <= CHUNK; j0 += 4) {
        int32_t v4[4];
        C q00[4], q10[4], e0[4], e1[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v4[i] = j0 + i <= CHUNK ? verts[s0 + j0 + i] : -1;
        corners4<T, LOGITS>(lw, v4, lane, blockIdx.y == 0, lprobs, q00, q10, e0, e1);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j0 + i] = v4[i], lp00[j0 + i] = q00[i], lp10[j0 + i] = q10[i], ld0[j0 + i] = e0[i], ld1[j0 + i] = e1[i];
    }
#pragma unroll
    for (int j0 = 0; j0 < CHUNK; j0 += 4) {
        int32_t n4[4];
        C q00[4], q10[4], e0[4], e1[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) n4[i] = neuron[s0 + j0 + i];
        corners4<T, LOGITS>(w, n4, lane, blockIdx.y == 0, probs, q00, q10, e0, e1);
#pragma unroll
        for (int i = 0; i < 4; ++i) n[j0 + i] = n4[i], p00[j0 + i] = q00[i], p10[j0 + i] = q10[i], d0[j0 + i] = e0[i], d1[j0 + i] = e1[i];
    }
    int64_t ia[CHUNK + 1], ib[CHUNK + 1];
#pragma unroll
    for (int j = 0; j <= CHUNK; ++j) ia[j] = low_a[v[j]], ib[j] = low_b[v[j]];

    for (int64_t ct = blockIdx.y; ct * DL_WAVE < ncols; ct += gridDim.y) {
        const int64_t col = ct * DL_WAVE + lane;
        const bool live = col < ncols;
        const int64_t cl = live ? col : 0;
        // the chunk's CHUNK + 1 input rows, recomputed four at a time
        P rows[CHUNK + 1];
#pragma unroll
        for (int j0 = 0; j0 <= CHUNK; j0 += 4) {
            P va[4], vb[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (j0 + i <= CHUNK) {
                    va[i] = row_vec<P, VEC, RAG>(lx, ia[j0 + i], batch, ncols, cl);
                    vb[i] = row_vec<P, VEC, RAG>(lx, ib[j0 + i], batch, ncols, cl);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = j0 + i;
                if (j <= CHUNK) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e)
                        rows[j].v[e] = mix<T, RAG, C>(up<T>(va[i].v[e]), up<T>(vb[i].v[e]), lp00[j], lp10[j], ld0[j], ld1[j]);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < CHUNK; ++j) {
            const bool f = flip[s0 + j] != 0;
            P r;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const C u0 = up<T>(rows[j].v[e]), u1 = up<T>(rows[j + 1].v[e]);
                r.v[e] = mix<T, RAG, C>(f ? u1 : u0, f ? u0 : u1, p00[j], p10[j], d0[j], d1[j]);
            }
            if (live && n[j] >= 0) row_vec<P, VEC, RAG>(y, (int64_t) n[j], batch, ncols, cl) = r;
        }
    }
}

// Forward along the schedule for long rows: one wave owns `chunk` steps and a segment of
// CPL * 64 consecutive vectors of the row (blockIdx.y picks the segment; lane l holds its vectors
// l, l + 64, ...), so every gathered row is one contiguous request of up to 4 KB, and the next
// step's row is requested before this step's arithmetic.
template <typename T, int VEC, int CPL, int GATES, bool RAG, bool NT>
__global__ __launch_bounds__(DL_BLOCK) void forward_chain_rows_kernel(const T *__restrict__ x,
                                                                      const int32_t *__restrict__ verts,
                                                                      const int32_t *__restrict__ neuron,
                                                                      const uint8_t *__restrict__ flip,
                                                                      const T *__restrict__ w, T *__restrict__ y,
                                                                      T *__restrict__ probs, int64_t steps, int chunk,
                                                                      int64_t batch, bool w32) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t s0 = ((int64_t) blockIdx.x * 4 + wave) * chunk;
    if (s0 >= steps) return;
    const int64_t s1 = s0 + chunk < steps ? s0 + chunk : steps;
    const int64_t col0 = (int64_t) blockIdx.y * (CPL * DL_WAVE);
    auto load_row = [&](int64_t row, bool valid, P *out) {
#pragma unroll
        for (int q = 0; q < CPL; ++q)
            out[q] = row_part<P, VEC, RAG, NT>(x, row, valid, batch, ncols, col0 + lane + q * DL_WAVE);
    };
    // the chunk's schedule entries, one per lane (chunk <= 64), handed out by readlane: no scalar loads in the step loop
    const int cnt = (int) (s1 - s0);
    const bool has = lane < cnt;
    const int32_t sch_n = has ? neuron[s0 + lane] : -1;
    const int32_t sch_v = has ? verts[s0 + 1 + lane] : 0;
    const int32_t sch_f = has ? (int32_t) flip[s0 + lane] : 0;
    constexpr int AHEAD = 3, SLOTS = AHEAD + 1;     // rows requested before their step; step i is in slot i % SLOTS
    P prev[CPL], cur[SLOTS][CPL];
    auto fetch = [&](int i, P *out) {
        const bool there = i < cnt;
        load_row(__builtin_amdgcn_readlane(sch_v, there ? i : cnt - 1), there, out);
    };
    load_row(verts[s0], true, prev);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(i, cur[i]);
#pragma unroll 1
    for (int i0 = 0; i0 < cnt; i0 += 4) {            // four steps per trip: their corners are computed together
        int32_t n[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) n[j] = __builtin_amdgcn_readlane(sch_n, (i0 + j) & 63);
        C p00[4], p10[4], d0[4], d1[4];
        corners4<T, GATES, NT>(w, n, lane, col0 == 0, probs, p00, p10, d0, d1, w32);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = i0 + j;
            if (i < cnt) {                           // wave-uniform
                const int now = j % SLOTS;
                fetch(i + AHEAD, cur[(j + AHEAD) % SLOTS]);
                const bool f = __builtin_amdgcn_readlane(sch_f, i) != 0;
#pragma unroll
                for (int q = 0; q < CPL; ++q) {
                    const int64_t col = col0 + lane + q * DL_WAVE;
                    P r;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        const C u0 = up<T>(prev[q].v[e]), u1 = up<T>(cur[now][q].v[e]);
                        r.v[e] = mix<T, RAG, C>(f ? u1 : u0, f ? u0 : u1, p00[j], p10[j], d0[j], d1[j]);
                    }
                    if (n[j] >= 0 && col < ncols) row_vec<P, VEC, RAG>(y, (int64_t) n[j], batch, ncols, col) = r;
                }
#pragma unroll
                for (int q = 0; q < CPL; ++q) prev[q] = cur[now][q];
            }
        }
    }
}

// One wave owns CHUNK steps and the whole batch: lane l holds vectors l, l + 64, ... (CPL of them).
template <typename T, int VEC, int CPL, int CHUNK, bool RAG, bool NT>
__global__ __launch_bounds__(DL_BLOCK) void backward_w_chain_kernel(const T *__restrict__ x,
                                                                    const int32_t *__restrict__ verts,
                                                                    const int32_t *__restrict__ neuron,
                                                                    const uint8_t *__restrict__ flip,
                                                                    const T *__restrict__ gy,
                                                                    const T *__restrict__ probs, T *__restrict__ gw,
                                                                    int64_t nchunks, int64_t batch, int64_t gdiv, bool w32) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t c = (int64_t) blockIdx.x * 4 + wave;
    if (c >= nchunks) return;
    const int64_t s0 = c * CHUNK;
    auto load_row = [&](const T *base, int64_t row, P *dst) {
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
            const int64_t col = lane + q * DL_WAVE;
            dst[q] = row_part<P, VEC, RAG, NT>(base, row, true, batch, ncols, col);
        }
    };
    static_assert(CHUNK % 4 == 0, "neurons are finished four at a time");
    const int quarter = lane >> 4;                   // which of four neurons this lane finishes
    P prev[CPL];
    load_row(x, verts[s0], prev);
#pragma unroll 1
    for (int j0 = 0; j0 < CHUNK; j0 += 4) {
        int32_t n[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) n[i] = neuron[s0 + j0 + i];
        const int32_t mine = quarter == 0 ? n[0] : quarter == 1 ? n[1] : quarter == 2 ? n[2] : n[3];
        const C p = probs != nullptr && mine >= 0 ? wload<T>(probs, (int64_t) mine * 16 + (lane & 15), w32) : (C) 0;
        C sums = (C) 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool f = flip[s0 + j0 + i] != 0;
            P cur[CPL], g[CPL];
            load_row(x, verts[s0 + j0 + i + 1], cur);
            load_row(gy, grad_row(n[i] >= 0 ? n[i] : 0, gdiv), g);
            C s00 = (C) 0, s01 = (C) 0, s10 = (C) 0, s11 = (C) 0;
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
                const int dup = vec_dup<VEC, RAG>(lane + q * DL_WAVE, batch);
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const C u0 = up<T>(prev[q].v[e]), u1 = up<T>(cur[q].v[e]), gg = own_part<RAG>(up<T>(g[q].v[e]), e, dup);
                    const C av = f ? u1 : u0, bv = f ? u0 : u1;
                    const C ga = gg * av, gna = gg - ga;
                    const C t11 = ga * bv, t01 = gna * bv;
                    s11 += t11;
                    s10 += ga - t11;
                    s01 += t01;
                    s00 += gna - t01;
                }
            }
            const C z = wave_sum4_lane(s00, s01, s10, s11, lane);
            sums = quarter == i ? z : sums;
#pragma unroll
            for (int q = 0; q < CPL; ++q) prev[q] = cur[q];
        }
        store_grad_w4<T, NT>(lane, mine >= 0, mine, sums, p, probs != nullptr, gw, w32);
    }
}

// ------------------------------------------------------------------------------------------
// Chained backward: grad_w AND grad_x of a layer in one pass along the schedule.  Step s reads
// input row verts[s + 1] and grad_y row neuron[s] (the other input row is still in registers),
// which is all that backward_w and both directions of backward_x need for that neuron:
//     to a:  g * ((P10 - P00) + b * dd)      to b:  g * ((P01 - P00) + a * dd)
//     dd = (P11 - P10) - (P01 - P00)
// A vertex in the middle of a trail collects the share of the neuron before it (kept in
// `carry`) and of the neuron after it and is written once: position p of the schedule goes to
// row dst[p] (-1: nothing to write; >= in_dim: row dst[p] - in_dim of `overflow`, for vertices
// that occur at several positions and are summed afterwards by backward_fix_kernel; the parts are kept in the type
// that sums are taken in, and half results are rounded once, after the sum and the scale).  Rows longer
// than CPL * 64 vectors are cut into segments (blockIdx.y); the corner sums of the segments then
// go to `partial` and backward_w_finish_kernel adds them.  A wave
// owns `chunk` positions [s0, s0 + chunk); it recomputes the last neuron of the chunk before it to get
// the carry into its first position, so chunks do not exchange partial rows.
// ------------------------------------------------------------------------------------------
// LOWER >= 1: the layer BELOW this one (whose output x is) needs no grad_x of its own and gets its
// grad_w here: a vertex's finished grad_x row is the grad_y row of neuron `vertex` of the layer below,
// so its four corner sums are taken on the spot from the row in registers and the two input rows of
// that neuron (`low.x`, gathered through `low.a`, `low.b`), and the row is not stored at all.  Only the
// vertices that finish in backward_fix_kernel still go through memory (backward_w_rows_kernel).
// LOWER == 2: x itself is not read either: row v of x is recomputed as the lower layer's forward pass
// computed it (same arithmetic, same rounding) from the two lower input rows that the vertex's
// backward_w needs anyway, so the activation between the two layers never exists in memory.
template <typename T> struct LowerLayer {
    const T *x;                 // [in_dim of the layer below, batch]
    const int64_t *a, *b;       // its wiring, [in_dim]
    const T *w;                 // its gate probabilities [in_dim, 16]
    const T *probs;             // == w: chain the softmax backward into gw; null: gw is the plain grad_w
    T *gw;                      // [in_dim, 16]
};

// Vertices of several positions (or none) that further workgroups of the launch finish, a wave each, forming their parts
// anew: `vertex` [count] with positions[start[i]] .. positions[start[i + 1] - 1].  positions == nullptr: the walks store the
// parts to overflow rows and backward_fix_kernel adds them.
struct FixHere {
    const int32_t *vertex, *start, *positions;
    int count;
    uint32_t first_block;
};

// A vector of an overflow row.  (Eight floats for half rows: two 16-byte accesses, no 32-byte alignment asked for.)
template <typename T, int VEC, bool RAG>
using OverflowPack = Pack<typename Acc<T>::type, VEC, RAG || sizeof(T) != sizeof(typename Acc<T>::type)>;

// dy/da or dy/db of a neuron, k + u * dd.  SPLIT: in two roundings, as backward_x_kernel has it.
template <bool SPLIT, typename C> __device__ __forceinline__ C slope(C u, C dd, C k) {
    if constexpr (SPLIT) return k + u * dd;
    else return dl_fma(u, dd, k);
}

template <typename T, int VEC, int CPL, int LOWER, bool RAG, bool NT>
__global__ __launch_bounds__(DL_BLOCK) void backward_chain_kernel(
    const T *__restrict__ x, const int32_t *__restrict__ verts, const int32_t *__restrict__ neuron,
    const uint8_t *__restrict__ flip, const int32_t *__restrict__ dst, const T *__restrict__ w,
    const T *__restrict__ gy, const T *__restrict__ probs, T *__restrict__ gw,
    typename Acc<T>::type *__restrict__ partial, T *__restrict__ gx, typename Acc<T>::type *__restrict__ overflow,
    int64_t steps, int chunk, int64_t in_dim, int64_t out_dim, int64_t batch, typename Acc<T>::type scale, int64_t gdiv, LowerLayer<T> low,
    FixHere fix, bool w32) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    constexpr bool RECOMPUTE = LOWER == 2;
    // a last-bit difference in fp32 turns a half result by 2^-11 now and then: with SPLIT, half rows of any length get the
    // bits of backward_x_kernel whether or not their layer is walked along its schedule
    constexpr bool SPLIT = RAG && sizeof(T) == 2;
    constexpr int LCPL = LOWER ? CPL : 1;                       // registers for lower rows only where they are used
    // steps whose rows are requested before they are walked: three on short fp32 rows (64000 -> 64000, one / three: batch 100
    // 27.6 / 25.8 us, 128 28.6 / 26.2); half rows, whose steps hold more registers, lose by it (500: 45.8 / 47.4)
    constexpr int AHEAD = CPL == 1 && LOWER == 0 && sizeof(T) == 4 ? 3 : 1, SLOTS = AHEAD + 1;
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const bool fixes = blockIdx.x >= fix.first_block;            // (uniform) a workgroup that finishes vertices of several positions
    const int64_t s0 = ((int64_t) (fixes ? 0 : blockIdx.x) * 4 + wave) * chunk;
    if (!fixes && s0 >= steps) return;
    const int64_t s1 = s0 + chunk < steps ? s0 + chunk : steps;
    const int64_t col0 = (int64_t) blockIdx.y * (CPL * DL_WAVE);   // this wave's segment of the rows
    const int gate = lane & 15;
    auto load_row_as = [&](auto once, const T *base, int64_t row, bool valid, P *out) {
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
            const int64_t col = col0 + lane + q * DL_WAVE;
            out[q] = row_part<P, VEC, RAG, decltype(once)::value>(base, row, valid, batch, ncols, col);
        }
    };
    auto load_row = [&](const T *base, int64_t row, bool valid, P *out) {          // of x or grad_y
        load_row_as(std::bool_constant<NT>(), base, row, valid, out);
    };
    // the two input rows of neuron v of the layer below (v wave-uniform)
    auto lower_rows = [&](int64_t v, bool valid, P *la, P *lb) {
        if constexpr (LOWER != 0) {
            const int64_t r = valid ? v : 0;
            load_row_as(std::false_type(), low.x, low.a[r], valid, la);
            load_row_as(std::false_type(), low.x, low.b[r], valid, lb);
        }
    };
    // Corner sums of the probabilities in the lanes' 16-lane rows, in the association order of corners_of().
    const C zc = (C) 0;
    const int quarter = lane >> 4;                   // which of four steps this lane's row serves
    auto corner_rows = [&](C p, C &q00, C &q10, C &d0, C &d1) {
        q00 = row16_sum((gate & 8) ? p : zc);
        q10 = row16_sum((gate & 2) ? p : zc);
        d0 = row16_sum((gate & 4) ? p : zc) - q00;
        d1 = row16_sum((gate & 1) ? p : zc) - q10;
    };
    auto pick = [&](const int32_t (&v)[4]) { return quarter == 0 ? v[0] : quarter == 1 ? v[1] : quarter == 2 ? v[2] : v[3]; };
    // row v of x as the lower layer's forward kernel stored it, from its two input rows and corner coefficients
    auto lower_forward = [&](const P *la, const P *lb, C p00, C p10, C d0, C d1, P *out) {
#pragma unroll
        for (int q = 0; q < CPL; ++q)
#pragma unroll
            for (int e = 0; e < VEC; ++e)
                out[q].v[e] = mix<T, RAG, C>(up<T>(la[q].v[e]), up<T>(lb[q].v[e]), p00, p10, d0, d1);
    };
    // ... of a single vertex
    auto lower_row = [&](int64_t v, P *la, P *lb, P *out) {
        lower_rows(v, true, la, lb);
        C q00, q10, d0, d1;
        corner_rows(up<T>(low.w[v * 16 + gate]), q00, q10, d0, d1);
        lower_forward(la, lb, lane_value(q00, 0), lane_value(q10, 0), lane_value(d0, 0), lane_value(d1, 0), out);
    };
    // (LOWER) corner sums of the layer below for a finished vertex, whose lower rows are la, lb: as backward_w_kernel on the
    // row that would have been stored, same values, same order of additions
    auto lower_sums = [&](const C (&val)[CPL][VEC], const P *la, const P *lb, C scale) {
        C s00 = (C) 0, s01 = (C) 0, s10 = (C) 0, s11 = (C) 0;
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
            const int dup = vec_dup<VEC, RAG>(col0 + lane + q * DL_WAVE, batch);
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const C g = own_part<RAG>(up<T>(round_scaled<T, RAG, C>(val[q][e], scale)), e, dup);
                const C av = up<T>(la[q].v[e]), bv = up<T>(lb[q].v[e]);
                const C ga = g * av, gna = g - ga;
                const C t11 = ga * bv, t01 = gna * bv;
                s11 += t11;
                s10 += ga - t11;
                s01 += t01;
                s00 += gna - t01;
            }
        }
        return wave_sum4_lane(s00, s01, s10, s11, lane);
    };
    // a finished position's row to where dst says; with LOWER only parts of sums are stored
    auto store_row = [&](int32_t row, const C (&val)[CPL][VEC]) {
        if (row < 0 || (LOWER != 0 && row < in_dim)) return;
        if (row >= in_dim) {                                     // a part of a sum: in C, scaled here only if that is T
            if (fix.positions != nullptr) return;                // ... or formed where the sum is taken
            typedef OverflowPack<T, VEC, RAG> O;
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
                const int64_t col = col0 + lane + q * DL_WAVE;
                O r;
#pragma unroll
                for (int e = 0; e < VEC; ++e) r.v[e] = sizeof(T) == sizeof(C) ? val[q][e] * scale : val[q][e];
                if (col < ncols) row_vec<O, VEC, RAG>(overflow, (int64_t) row - in_dim, batch, ncols, col) = r;
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < CPL; ++q) {
            const int64_t col = col0 + lane + q * DL_WAVE;
            P r;
#pragma unroll
            for (int e = 0; e < VEC; ++e) r.v[e] = round_scaled<T, RAG, C>(val[q][e], scale);
            if (col < ncols) row_vec<P, VEC, RAG>(gx, row, batch, ncols, col) = r;
        }
    };

    // The share of neuron n = neuron[s], between positions s and s + 1, of the vertex at `own`, from the row of the other.
    auto share_of = [&](int64_t s, bool own_first, C (&share)[CPL][VEC]) {
        const int32_t n = neuron[s];
        const bool f = flip[s] != 0;
        P other[CPL], g[CPL];
        const int64_t v = verts[own_first ? s + 1 : s];
        if constexpr (RECOMPUTE) {
            P oa[LCPL], ob[LCPL];
            lower_row(v, oa, ob, other);
        } else {
            load_row(x, v, true, other);
        }
        load_row(gy, grad_row(n, gdiv), true, g);
        const Corners<C> k = corners<T>(w, n, w32);
        const C d0 = k.p01 - k.p00, dd = (k.p11 - k.p10) - d0, da = k.p10 - k.p00;
        const C kk = f == own_first ? d0 : da;
#pragma unroll
        for (int q = 0; q < CPL; ++q)
#pragma unroll
            for (int e = 0; e < VEC; ++e) share[q][e] = up<T>(g[q].v[e]) * slope<SPLIT, C>(up<T>(other[q].v[e]), dd, kk);
    };
    if (fixes) {
        // a wave per vertex: the parts of its positions as the walks form them, added in the order of the overflow rows
        const int i = (int) (blockIdx.x - fix.first_block) * 4 + wave;
        if (i >= fix.count) return;
        const int64_t v = fix.vertex[i];
        C acc[CPL][VEC];
#pragma unroll
        for (int q = 0; q < CPL; ++q)
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[q][e] = (C) 0;
        const int32_t r1 = fix.start[i + 1];
#pragma unroll 1
        for (int32_t r = fix.start[i]; r < r1; ++r) {
            const int64_t p = fix.positions[r];
            C part[CPL][VEC], next[CPL][VEC];
#pragma unroll
            for (int q = 0; q < CPL; ++q)
#pragma unroll
                for (int e = 0; e < VEC; ++e) part[q][e] = next[q][e] = (C) 0;
            if (p > 0 && neuron[p - 1] >= 0) share_of(p - 1, false, part);
            if (p < steps && neuron[p] >= 0) share_of(p, true, next);
#pragma unroll
            for (int q = 0; q < CPL; ++q)
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const C both = part[q][e] + next[q][e];
                    acc[q][e] += sizeof(T) == sizeof(C) ? both * scale : both;
                }
        }
        const C rest = sizeof(T) == sizeof(C) ? (C) 1 : scale;
        if constexpr (LOWER != 0) {
            P fa[LCPL], fb[LCPL];
            lower_rows(v, true, fa, fb);
            const C lz = lower_sums(acc, fa, fb, rest);
            const C p = low.probs != nullptr ? up<T>(low.probs[v * 16 + gate]) : zc;
            store_grad_w4<T, NT>(lane, quarter == 0, v, lz, p, low.probs != nullptr, low.gw, false);
        } else {
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
                const int64_t col = col0 + lane + q * DL_WAVE;
                P r;
#pragma unroll
                for (int e = 0; e < VEC; ++e) r.v[e] = round_scaled<T, RAG, C>(acc[q][e], rest);
                if (col < ncols) row_vec<P, VEC, RAG>(gx, v, batch, ncols, col) = r;
            }
        }
        return;
    }

    // prev: row of the vertex at the chunk's first position; pla, plb: (RECOMPUTE) the lower rows it came from,
    // which also serve that vertex's backward_w at step 0
    P prev[CPL], pla[LCPL], plb[LCPL];
    C carry[CPL][VEC];
    if constexpr (RECOMPUTE) lower_row(verts[s0], pla, plb, prev);
    else load_row(x, verts[s0], true, prev);
#pragma unroll
    for (int q = 0; q < CPL; ++q)
#pragma unroll
        for (int e = 0; e < VEC; ++e) carry[q][e] = (C) 0;
    // the share of the neuron that ends at this chunk's first vertex
    if (s0 > 0 && neuron[s0 - 1] >= 0) share_of(s0 - 1, false, carry);
    // The chunk's schedule entries are fetched once, one per lane (chunk <= 64), and handed out by
    // readlane, so the step loop waits for no scalar loads; the rows of step i + 1 are requested
    // before the arithmetic of step i.
    const int cnt = (int) (s1 - s0);
    const bool has = lane < cnt;
    const int32_t sch_n = has ? neuron[s0 + lane] : -1;
    const int32_t sch_v = has ? verts[s0 + 1 + lane] : 0;
    const int32_t sch_d = has ? dst[s0 + lane] : -1;
    const int32_t sch_f = has ? (int32_t) flip[s0 + lane] : 0;
    // Rows of step i: the new input row (RECOMPUTE: the two lower rows it is recomputed from) and the neuron's grad_y
    // row (zero for a step without a neuron).  LOWER == 1: la, lb are the lower rows of the vertex that step i
    // finishes (dst[i]); RECOMPUTE: of the vertex that step i brings in.
    auto fetch = [&](int i, P *row, P *grad, P *la, P *lb) {
        const bool there = i < cnt;
        if (!there) i = cnt - 1;
        const int32_t n = __builtin_amdgcn_readlane(sch_n, i);
        const int32_t v = __builtin_amdgcn_readlane(sch_v, i);
        if constexpr (RECOMPUTE) {
            lower_rows(v, there, la, lb);
        } else {
            load_row(x, v, there, row);
            if constexpr (LOWER == 1) {
                const int32_t d = __builtin_amdgcn_readlane(sch_d, i);
                lower_rows(d, there && d >= 0 && d < in_dim, la, lb);
            }
        }
        load_row(gy, grad_row(n >= 0 ? n : 0, gdiv), there && n >= 0, grad);
    };
    // What is needed once per neuron is done for four steps at a time, a 16-lane row each: of the group that starts at
    // step i the neurons' probabilities, (RECOMPUTE) those of the vertices the steps bring in, and (LOWER) those of the
    // vertices they finish.
    auto entries = [&](int32_t sch, int i, int32_t (&v)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __builtin_amdgcn_readlane(sch, (i + j) & 63);
    };
    auto fetch_probs = [&](int i, C &p, C &lp, C &dp) {
        int32_t v[4];
        entries(sch_n, i, v);
        const int32_t n = pick(v);
        p = wload<T>(w, (int64_t) (n >= 0 ? n : 0) * 16 + gate, w32);
        if constexpr (RECOMPUTE) {
            entries(sch_v, i, v);
            lp = up<T>(low.w[(int64_t) pick(v) * 16 + gate]);
        }
        if constexpr (LOWER != 0) {
            entries(sch_d, i, v);
            const int32_t d = pick(v);
            if (low.probs != nullptr) dp = up<T>(low.probs[(int64_t) (d >= 0 && d < in_dim ? d : 0) * 16 + gate]);
        }
    };
    P cur[SLOTS][CPL], g[SLOTS][CPL], la[SLOTS][LCPL], lb[SLOTS][LCPL];       // step i is in slot i % SLOTS
    C pw, lpw = zc, dpw = zc;
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(i, cur[i], g[i], la[i], lb[i]);
    fetch_probs(0, pw, lpw, dpw);
#pragma unroll 1
    for (int i0 = 0; i0 < cnt; i0 += 4) {
        int32_t n[4], d[4], fl[4];
        entries(sch_n, i0, n);
        entries(sch_d, i0, d);
        entries(sch_f, i0, fl);
        C npw = zc, nlpw = zc, ndpw = zc;
        if (i0 + 4 < cnt) fetch_probs(i0 + 4, npw, nlpw, ndpw);
        C c00, c10, cd0, cd1, l00 = zc, l10 = zc, ld0 = zc, ld1 = zc;
        corner_rows(pw, c00, c10, cd0, cd1);
        const C cdd = cd1 - cd0, cda = c10 - c00;
        const bool frow = pick(fl) != 0;
        const C cku = frow ? cd0 : cda, ckv = frow ? cda : cd0;
        if constexpr (RECOMPUTE) corner_rows(lpw, l00, l10, ld0, ld1);
        C sums = zc, lsums = zc;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = i0 + j;
            if (i < cnt) {                               // (wave-uniform)
                const int now = j % SLOTS, ahead = (j + AHEAD) % SLOTS;
                fetch(i + AHEAD, cur[ahead], g[ahead], la[ahead], lb[ahead]);
                if constexpr (RECOMPUTE)
                    lower_forward(la[now], lb[now], lane_value(l00, 16 * j), lane_value(l10, 16 * j), lane_value(ld0, 16 * j),
                                  lane_value(ld1, 16 * j), cur[now]);
                if (RAG && n[j] < 0)
#pragma unroll
                    for (int q = 0; q < CPL; ++q) g[now][q] = P{};
                const bool f = fl[j] != 0;
                const C dd = lane_value(cdd, 16 * j), ku = lane_value(cku, 16 * j), kv = lane_value(ckv, 16 * j);
                C s00 = zc, s01 = zc, s10 = zc, s11 = zc;
                C out[CPL][VEC];
#pragma unroll
                for (int q = 0; q < CPL; ++q) {
                    const int dup = vec_dup<VEC, RAG>(col0 + lane + q * DL_WAVE, batch);
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        const C u0 = up<T>(prev[q].v[e]), u1 = up<T>(cur[now][q].v[e]), gg = up<T>(g[now][q].v[e]);
                        const C av = f ? u1 : u0, bv = f ? u0 : u1;
                        const C gs = own_part<RAG>(gg, e, dup);
                        const C ga = gs * av, gna = gs - ga;
                        const C t11 = ga * bv, t01 = gna * bv;
                        s11 += t11;
                        s10 += ga - t11;
                        s01 += t01;
                        s00 += gna - t01;
                        out[q][e] = carry[q][e] + gg * slope<SPLIT, C>(u1, dd, ku);
                        carry[q][e] = gg * slope<SPLIT, C>(u0, dd, kv);
                    }
                }
                const C z = wave_sum4_lane(s00, s01, s10, s11, lane);
                sums = quarter == j ? z : sums;
                // the vertex at position s0 + i is finished: RECOMPUTE keeps its lower rows from the step that brought it in
                if constexpr (LOWER != 0) {
                    if (d[j] >= 0 && d[j] < in_dim) {
                        const C lz = lower_sums(out, RECOMPUTE ? pla : la[now], RECOMPUTE ? plb : lb[now], scale);
                        lsums = quarter == j ? lz : lsums;
                    }
                }
                store_row(d[j], out);
#pragma unroll
                for (int q = 0; q < CPL; ++q) prev[q] = cur[now][q];
                if constexpr (RECOMPUTE) {
#pragma unroll
                    for (int q = 0; q < LCPL; ++q) pla[q] = la[now][q], plb[q] = lb[now][q];
                }
            }
        }
        const int32_t mine = pick(n);                    // (-1 past the end: the lanes beyond hold no entry)
        if (partial == nullptr) {
            store_grad_w4<T, NT>(lane, mine >= 0, mine, sums, pw, probs != nullptr, gw, w32);
        } else if (mine >= 0 && gate < 4) {              // several segments: backward_w_finish_kernel adds them
            store_elem<NT>(partial + ((int64_t) blockIdx.y * out_dim + mine) * 4 + gate, sums);
        }
        if constexpr (LOWER != 0) {
            const int32_t done = pick(d);
            store_grad_w4<T, NT>(lane, done >= 0 && done < in_dim, done, lsums, dpw, low.probs != nullptr, low.gw, false);
        }
        pw = npw;
        lpw = nlpw;
        dpw = ndpw;
    }
    if (s1 == steps) {                                   // the schedule's last position
        const int32_t last = dst[steps];
        if constexpr (LOWER != 0) {
            if (last >= 0 && last < in_dim) {
                if constexpr (LOWER == 1) lower_rows(last, true, pla, plb);
                const C lz = lower_sums(carry, pla, plb, scale);
                const C p = low.probs != nullptr ? up<T>(low.probs[(int64_t) last * 16 + gate]) : zc;
                store_grad_w4<T, NT>(lane, quarter == 0, last, lz, p, low.probs != nullptr, low.gw, false);
            }
        }
        store_row(last, carry);
    }
}

// grad_x rows of the vertices that backward_chain_kernel could not finish in one write: vertex
// fix_vertex[i] is the sum, in slot order, of overflow rows [fix_start[i], fix_start[i + 1])
// (no rows: the input feeds no neuron and its gradient is zero).
// compact: row i of gx instead of row fix_vertex[i] (gx then has n_fix rows only).  scale: what the parts still lack
// (1 where backward_chain_kernel put it in).
template <typename T, int VEC, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void backward_fix_kernel(const typename Acc<T>::type *__restrict__ overflow,
                                                                const int32_t *__restrict__ fix_vertex,
                                                                const int32_t *__restrict__ fix_start,
                                                                T *__restrict__ gx, int64_t n_fix, int64_t batch,
                                                                typename Acc<T>::type scale, bool compact) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    typedef OverflowPack<T, VEC, RAG> O;
    const int64_t ncols = vec_count<VEC>(batch);
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t i = (int64_t) blockIdx.x * 4 + wave;
    if (i >= n_fix) return;
    const int64_t v = compact ? i : (int64_t) fix_vertex[i];
    const int32_t r0 = fix_start[i], r1 = fix_start[i + 1];
    for (int64_t col = (int64_t) blockIdx.y * DL_WAVE + lane; col < ncols; col += (int64_t) gridDim.y * DL_WAVE) {
        C acc[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = (C) 0;
        for (int32_t r = r0; r < r1; ++r) {
            const O part = row_vec<O, VEC, RAG>(overflow, (int64_t) r, batch, ncols, col);
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] += part.v[e];
        }
        P res;
#pragma unroll
        for (int e = 0; e < VEC; ++e) res.v[e] = round_scaled<T, RAG, C>(acc[e], scale);
        row_vec<P, VEC, RAG>(gx, v, batch, ncols, col) = res;
    }
}

// backward_w of the layer below for the few vertices whose grad_x row backward_fix_kernel finished:
// neuron list[i] of that layer, its grad_y row = row i of `rows`.  One wave per neuron, the sums in
// the order of backward_w_kernel.
template <typename T, int VEC, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void backward_w_rows_kernel(LowerLayer<T> low, const int32_t *__restrict__ list,
                                                                   const T *__restrict__ rows, int64_t n_list,
                                                                   int64_t batch) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    const int lane = dl_lane();
    const int64_t i = (int64_t) blockIdx.x * 4 + dl_wave_in_block();
    if (i >= n_list) return;
    const int64_t n = list[i];
    const int64_t ia = low.a[n], ib = low.b[n];
    C s00 = (C) 0, s01 = (C) 0, s10 = (C) 0, s11 = (C) 0;
    for (int64_t col = lane; col < ncols; col += DL_WAVE) {
        const int dup = vec_dup<VEC, RAG>(col, batch);
        const P va = row_vec<P, VEC, RAG>(low.x, ia, batch, ncols, col), vb = row_vec<P, VEC, RAG>(low.x, ib, batch, ncols, col);
        const P vg = row_vec<P, VEC, RAG>(rows, i, batch, ncols, col);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const C av = up<T>(va.v[e]), bv = up<T>(vb.v[e]), g = own_part<RAG>(up<T>(vg.v[e]), e, dup);
            const C ga = g * av, gna = g - ga;
            const C t11 = ga * bv, t01 = gna * bv;
            s11 += t11;
            s10 += ga - t11;
            s01 += t01;
            s00 += gna - t01;
        }
    }
    wave_sum4(s00, s01, s10, s11, lane);
    store_grad_w<T>(lane, true, n, s00, s01, s10, s11, low.probs, low.gw);
}

// grad_w from the per-segment corner sums of backward_chain_kernel, added in segment order.
// One 16-lane row per neuron (4 neurons per wave).
template <typename T>
__global__ __launch_bounds__(DL_BLOCK) void backward_w_finish_kernel(const typename Acc<T>::type *__restrict__ partial,
                                                                     const T *__restrict__ probs, T *__restrict__ gw,
                                                                     int64_t out_dim, int segments, bool w32) {
    typedef typename Acc<T>::type C;
    const int lane = dl_lane();
    const int64_t n = ((int64_t) blockIdx.x * 4 + dl_wave_in_block()) * 4 + (lane >> 4);
    const bool valid = n < out_dim;
    const int gate = lane & 15;
    C sum[4] = {(C) 0, (C) 0, (C) 0, (C) 0};
    if (valid)
        for (int g = 0; g < segments; ++g)
#pragma unroll
            for (int c = 0; c < 4; ++c) sum[c] += partial[((int64_t) g * out_dim + n) * 4 + c];
    C r = (C) 0;
    if (gate & 8) r += sum[0];
    if (gate & 4) r += sum[1];
    if (gate & 2) r += sum[2];
    if (gate & 1) r += sum[3];
    if (probs != nullptr) {
        const C p = valid ? wload<T>(probs, n * 16 + gate, w32) : (C) 0;
        const C dot = row16_sum(p * r);
        r = p * (r - dot);
    }
    if (valid) wstore<T>(gw, n * 16 + gate, r, w32);
}

template <typename T> struct Vec16 { static constexpr int n = 16 / (int) sizeof(T); };

// How the rows of a call are read and written: whole aligned 16-byte vectors, vectors of that size of which the last
// overlaps the one before it (RAG kernels), or one element per lane where a row is shorter than a vector.
enum class Rows { whole, ragged, single };

template <typename T> Rows rows_kind(int64_t batch, const void *p0, const void *p1 = nullptr, const void *p2 = nullptr,
                                     const void *p3 = nullptr) {
    constexpr int V = Vec16<T>::n;
    if (batch % V == 0 && dl_aligned(p0, 16) && dl_aligned(p1, 16) && dl_aligned(p2, 16) && dl_aligned(p3, 16))
        return Rows::whole;
    return batch >= V ? Rows::ragged : Rows::single;
}

// Rows up to which both gradients share a launch.  On longer ones launches do not count and the two kernels get in each
// other's way (fp32 1000 -> 1000, two launches / one: batch 4096 25.2 / 23.9 us, 8192 41.5 / 41.3, 16384 75.5 / 76.6, 65536
// 303 / 349; 2000 -> 2000 at 16384 146 / 152, half at 65536 309 / 329).
#define DL_BOTH_MAX_ROW_BYTES 32768

#define DL_GRID_MAX (0xffffffffLL / DL_BLOCK)         // workgroups along x: HIP counts the threads in 32 bits

unsigned col_tiles(int64_t ncols) {
    int64_t t = dl_ceil_div(ncols, DL_WAVE);
    return (unsigned) (t > 65535 ? 65535 : t);
}

template <typename T, int GATES>
int forward_t(const void *x, const int64_t *a, const int64_t *b, const void *w, void *y, void *probs, int64_t out_dim,
              int64_t batch, hipStream_t s, bool w32 = false) {
    constexpr int NPW = 4;
    const int64_t blocks = dl_ceil_div(out_dim, 4 * NPW);
    if (out_dim > 0x7fffffffLL) return DL_ERR_TOO_LARGE;     // neuron ids travel as int32 inside the kernel
    constexpr int V = Vec16<T>::n;
    const Rows kind = rows_kind<T>(batch, x, y);
    const dim3 grid((unsigned) blocks, col_tiles(kind == Rows::single ? batch : dl_ceil_div(batch, V)));
#define DL_LAUNCH_FORWARD(VV, RAG)                                                                                       \
    DL_LAUNCH((forward_kernel<T, VV, NPW, GATES, RAG>), grid, dim3(DL_BLOCK), 0, s, (const T *) x, a, b, (const T *) w, \
              (T *) y, (T *) probs, out_dim, batch, w32)
    if (kind == Rows::whole) DL_LAUNCH_FORWARD(V, false);
    else if (kind == Rows::ragged) DL_LAUNCH_FORWARD(V, true);
    else DL_LAUNCH_FORWARD(1, false);
#undef DL_LAUNCH_FORWARD
    return dl_launch_status();
}

template <typename T>
int backward_w_t(const void *x, const int64_t *a, const int64_t *b, const void *gy, const void *probs, void *gw,
                 int64_t out_dim, int64_t batch, hipStream_t s, int64_t gdiv = 0, bool w32 = false) {
    constexpr int NPW = 2;       // neurons per wave when the workgroup's waves split a neuron's batch
    constexpr int NPW1 = 2;      // ... when a wave owns whole rows: short rows, more neurons' loads in flight per wave
    constexpr int V = Vec16<T>::n;
    const Rows kind = rows_kind<T>(batch, x, gy);
    const int64_t ncols = kind == Rows::single ? batch : dl_ceil_div(batch, V);
    // Split one neuron's batch over the four waves once every wave still gets whole segments.
    const bool split = ncols >= 8 * DL_WAVE;
    const int64_t blocks = split ? dl_ceil_div(out_dim, NPW) : dl_ceil_div(out_dim, 4 * NPW1);
    if (blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
#define DL_LAUNCH_BACKWARD_W(VV, N, WPN, RAG)                                                                          \
    DL_LAUNCH((backward_w_kernel<T, VV, N, WPN, RAG>), dim3((unsigned) blocks), dim3(DL_BLOCK), 0, s, (const T *) x, a, \
              b, (const T *) gy, (const T *) probs, (T *) gw, out_dim, batch, gdiv, w32)
    if (kind == Rows::whole && split) DL_LAUNCH_BACKWARD_W(V, NPW, 4, false);
    else if (kind == Rows::whole) DL_LAUNCH_BACKWARD_W(V, NPW1, 1, false);
    else if (kind == Rows::ragged && split) DL_LAUNCH_BACKWARD_W(V, NPW, 4, true);
    else if (kind == Rows::ragged) DL_LAUNCH_BACKWARD_W(V, NPW1, 1, true);
    else DL_LAUNCH_BACKWARD_W(1, NPW1, 1, false);
#undef DL_LAUNCH_BACKWARD_W
    return dl_launch_status();
}

template <typename T>
int backward_x_t(const void *x, const int64_t *a, const int64_t *b, const void *w, const void *gy,
                 const int64_t *start, const int64_t *idx, void *gx, int64_t in_dim, int64_t batch, double scale,
                 hipStream_t s, int64_t gdiv = 0, bool w32 = false) {
    typedef typename Acc<T>::type C;
    constexpr int V = Vec16<T>::n;
    const int64_t blocks = dl_ceil_div(in_dim, 4);
    if (blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
    const Rows kind = rows_kind<T>(batch, x, gy, gx);
    const dim3 grid((unsigned) blocks, col_tiles(kind == Rows::single ? batch : dl_ceil_div(batch, V)));
#define DL_LAUNCH_BACKWARD_X(VV, RAG)                                                                                    \
    DL_LAUNCH((backward_x_kernel<T, VV, RAG>), grid, dim3(DL_BLOCK), 0, s, (const T *) x, a, b, (const T *) w,          \
              (const T *) gy, start, idx, (T *) gx, in_dim, batch, (C) scale, gdiv, w32)
    if (kind == Rows::whole) DL_LAUNCH_BACKWARD_X(V, false);
    else if (kind == Rows::ragged) DL_LAUNCH_BACKWARD_X(V, true);
    else DL_LAUNCH_BACKWARD_X(1, false);
#undef DL_LAUNCH_BACKWARD_X
    return dl_launch_status();
}

template <typename T>
int backward_both_t(const void *x, const int64_t *a, const int64_t *b, const void *w, const void *gy, bool softmax_backward,
                    const int64_t *start, const int64_t *idx, void *gw, void *gx, int64_t in_dim, int64_t out_dim,
                    int64_t batch, double scale, hipStream_t s, int64_t gdiv, bool w32) {
    typedef typename Acc<T>::type C;
    constexpr int V = Vec16<T>::n, NPW = 2;
    const Rows kind = rows_kind<T>(batch, x, gy, gx);
    const int64_t ncols = kind == Rows::single ? batch : dl_ceil_div(batch, V);
    const bool split = ncols >= 8 * DL_WAVE;                                         // as backward_w_t
    const int64_t row_blocks = dl_ceil_div(in_dim, 4), x_blocks = row_blocks * col_tiles(ncols);
    const int64_t blocks = x_blocks + (split ? dl_ceil_div(out_dim, NPW) : dl_ceil_div(out_dim, 4 * NPW));
    if (blocks > DL_GRID_MAX || batch * (int64_t) sizeof(T) > DL_BOTH_MAX_ROW_BYTES) {
        // a launch holds less than 2^32 threads along x, where this one has the column tiles too: one launch each
        const int st = backward_w_t<T>(x, a, b, gy, softmax_backward ? w : nullptr, gw, out_dim, batch, s, gdiv, w32);
        return st != DL_OK ? st : backward_x_t<T>(x, a, b, w, gy, start, idx, gx, in_dim, batch, scale, s, gdiv, w32);
    }
#define DL_LAUNCH_BOTH(VV, WPN, RAG)                                                                                       \
    DL_LAUNCH((backward_both_kernel<T, VV, NPW, WPN, RAG>), dim3((unsigned) blocks), dim3(DL_BLOCK), 0, s, (const T *) x, a, \
              b, (const T *) w, (const T *) gy, softmax_backward ? (const T *) w : nullptr, start, idx, (T *) gw, (T *) gx, \
              (uint32_t) row_blocks, (uint32_t) x_blocks, in_dim, out_dim, batch, (C) scale, gdiv, w32)
    if (kind == Rows::whole && split) DL_LAUNCH_BOTH(V, 4, false);
    else if (kind == Rows::whole) DL_LAUNCH_BOTH(V, 1, false);
    else if (kind == Rows::ragged && split) DL_LAUNCH_BOTH(V, 4, true);
    else if (kind == Rows::ragged) DL_LAUNCH_BOTH(V, 1, true);
    else DL_LAUNCH_BOTH(1, 1, false);
#undef DL_LAUNCH_BOTH
    return dl_launch_status();
}

// ------------------------------------------------------------------------------------------
// GroupSum on the feature-major layout.
//   forward : y[r, c] = (1/tau) * sum_{n in class c} x[n, r]       x [out, B] -> y [B, k]
//   backward: gx[n, r] = g[r, class(n)] / tau                      g [B, k]   -> gx [out, B]
// Forward is two passes with a fixed summation order: pass 1 sums SPLIT-th parts of every
// class block over the rows (lanes along the batch, the workgroup's four waves interleave
// rows and combine through LDS) into partial[s, c, r]; pass 2 adds the partials in order.
// ------------------------------------------------------------------------------------------
template <typename T, int VEC, bool RAG, bool NT>
__global__ __launch_bounds__(DL_BLOCK) void group_sum_partial_kernel(const T *__restrict__ x,
                                                                     typename Acc<T>::type *__restrict__ partial,
                                                                     int64_t per_class, int64_t batch, int64_t k,
                                                                     int64_t rows_per_split) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    __shared__ C lds[4][DL_WAVE * VEC];
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t col = (int64_t) blockIdx.x * DL_WAVE + lane;
    const int64_t cls = blockIdx.y, split = blockIdx.z;
    const int64_t at = col < ncols ? vec_at<VEC, RAG>(col, batch) : 0;
    int64_t r0 = split * rows_per_split, r1 = r0 + rows_per_split;
    if (r1 > per_class) r1 = per_class;
    C acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = (C) 0;
    if (col < ncols) {
        const T *xc = x + (cls * per_class) * batch + at;
        int64_t r = r0 + wave;
        auto row = [&](int64_t at) { return load_vec<NT>(*reinterpret_cast<const P *>(xc + at * batch)); };
        auto add = [&](const P *v) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] += (up<T>(v[0].v[e]) + up<T>(v[1].v[e])) + (up<T>(v[2].v[e]) + up<T>(v[3].v[e]));
        };
        for (; r + 28 < r1; r += 32) {      // eight independent row loads in flight per wave
            P v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = row(r + 4 * i);
            add(v);
            add(v + 4);
        }
        for (; r + 12 < r1; r += 16) {
            P v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = row(r + 4 * i);
            add(v);
        }
        for (; r < r1; r += 4) {
            const P v = row(r);
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] += up<T>(v.v[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) lds[wave][lane * VEC + e] = acc[e];
    __syncthreads();
    if (wave == 0 && col < ncols) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const int i = lane * VEC + e;
            const C sum = (lds[0][i] + lds[1][i]) + (lds[2][i] + lds[3][i]);
            partial[((int64_t) split * k + cls) * batch + at + e] = sum;
        }
    }
}

// The last LogicLayer and GroupSum in one pass: pass 1 of the sum above with the rows computed on
// the fly, y[n, r] = layer(x)[n, r] for the neurons of the class block, so the layer's output
// (and, in the backward pass, the broadcast gradient) never exists in memory.  Grid and partial
// layout as group_sum_partial_kernel; a wave takes four consecutive neurons at a time (their
// corner coefficients are computed together), the workgroup's waves interleave groups of four.
// LOGITS: `w` holds logits; the probabilities go to `probs` (column tile 0 only).
template <typename T, int VEC, bool LOGITS, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void forward_group_sum_kernel(const T *__restrict__ x, const int64_t *__restrict__ a,
                                                                     const int64_t *__restrict__ b, const T *__restrict__ w,
                                                                     T *__restrict__ probs,
                                                                     typename Acc<T>::type *__restrict__ partial,
                                                                     int64_t per_class, int64_t batch, int64_t k,
                                                                     int64_t rows_per_split) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    __shared__ C lds[4][DL_WAVE * VEC];
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t col = (int64_t) blockIdx.x * DL_WAVE + lane;
    const bool live = col < ncols;
    const int64_t cls = blockIdx.y, split = blockIdx.z;
    int64_t r0 = split * rows_per_split, r1 = r0 + rows_per_split;
    if (r1 > per_class) r1 = per_class;
    const int64_t cl = live ? col : 0;
    C acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = (C) 0;
    for (int64_t r = r0 + 4 * wave; r < r1; r += 16) {           // uniform per wave
        int64_t ia[4], ib[4];
        int32_t ids[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool valid = r + j < r1;
            const int64_t n = cls * per_class + (valid ? r + j : r);
            ia[j] = a[n];
            ib[j] = b[n];
            ids[j] = valid ? (int32_t) n : -1;
        }
        C p00[4], p10[4], d0[4], d1[4];
        corners4<T, LOGITS>(w, ids, lane, blockIdx.x == 0, probs, p00, p10, d0, d1);
        P va[4], vb[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            va[j] = row_vec<P, VEC, RAG>(x, ia[j], batch, ncols, cl);
            vb[j] = row_vec<P, VEC, RAG>(x, ib[j], batch, ncols, cl);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (ids[j] >= 0) {                                   // uniform
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    // rounded to T like the stored activation would have been
                    acc[e] += up<T>(mix<T, RAG, C>(up<T>(va[j].v[e]), up<T>(vb[j].v[e]), p00[j], p10[j], d0[j], d1[j]));
                }
            }
        }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) lds[wave][lane * VEC + e] = acc[e];
    __syncthreads();
    if (wave == 0 && live) {
        const int64_t at = vec_at<VEC, RAG>(col, batch);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const int i = lane * VEC + e;
            const C sum = (lds[0][i] + lds[1][i]) + (lds[2][i] + lds[3][i]);
            partial[((int64_t) split * k + cls) * batch + at + e] = sum;
        }
    }
}

// One wave per 64 consecutive samples of one class; the four waves of a workgroup take
// interleaved splits and are added in wave order, so the summation order is fixed.  The partial sums are added and scaled
// (by the reciprocal of tau) in double and rounded to T once: an fp32 score of 64 is 8e-6 from its neighbours, which is
// what the gradients of a net with large class sums see.  Bound by the latency of the partial sums, which come from the
// other XCDs: eight loads in flight per wave, none of them behind a branch (a load under `s < splits` is one: the compiler
// waits for each in turn).  GroupSum over 64000 rows at batch 100, 2 classes 36 -> 12 us, 10 classes 13 -> 8.
template <typename T>
__global__ __launch_bounds__(DL_BLOCK) void group_sum_finish_kernel(const typename Acc<T>::type *__restrict__ partial,
                                                                    T *__restrict__ y, int64_t batch, int64_t k,
                                                                    int splits, double inv_tau) {
    typedef typename Acc<T>::type C;
    __shared__ double lds[4][DL_WAVE];
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t r = (int64_t) blockIdx.x * DL_WAVE + lane;
    const int64_t c = blockIdx.y;
    double sum = 0.0;
    if (r < batch)
        for (int s = wave; s < splits; s += 32) {
            C v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i)                          // (past the end: the wave's own again, and not added)
                v[i] = partial[((int64_t) (s + 4 * i < splits ? s + 4 * i : s) * k + c) * batch + r];
#pragma unroll
            for (int i = 0; i < 8; ++i) sum += s + 4 * i < splits ? (double) v[i] : 0.0;
        }
    lds[wave][lane] = sum;
    __syncthreads();
    if (wave == 0 && r < batch)
        y[r * k + c] = from_double<T>(((lds[0][lane] + lds[1][lane]) + (lds[2][lane] + lds[3][lane])) * inv_tau);
}

template <typename T, int VEC, bool RAG>
__global__ __launch_bounds__(DL_BLOCK) void group_sum_backward_kernel(const T *__restrict__ g, T *__restrict__ gx,
                                                                      int64_t out_dim, int64_t per_class,
                                                                      int64_t batch, int64_t k,
                                                                      typename Acc<T>::type inv_tau) {
    typedef typename Acc<T>::type C;
    typedef Pack<T, VEC, RAG> P;
    const int64_t ncols = vec_count<VEC>(batch);
    const int wave = dl_wave_in_block();
    const int lane = dl_lane();
    const int64_t col = (int64_t) blockIdx.x * DL_WAVE + lane;
    if (col >= ncols) return;
    const int64_t at = vec_at<VEC, RAG>(col, batch);
    constexpr int ROWS = 16;                                              // rows per wave
    const int64_t n0 = ((int64_t) blockIdx.y * 4 + wave) * ROWS;
    int64_t cached_cls = -1;
    P val;
    for (int64_t n = n0; n < n0 + ROWS && n < out_dim; ++n) {
        const int64_t cls = n / per_class;
        if (cls != cached_cls) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) val.v[e] = round_scaled<T, RAG, C>(up<T>(g[(at + e) * k + cls]), inv_tau);
            cached_cls = cls;
        }
        row_vec<P, VEC, RAG>(gx, n, batch, ncols, col) = val;
    }
}

template <typename T>
int group_sum_forward_t(const void *x, void *y, void *workspace, int64_t out_dim, int64_t batch, int64_t k, int splits,
                        double tau, hipStream_t s) {
    typedef typename Acc<T>::type C;
    constexpr int V = Vec16<T>::n;
    const int64_t per_class = out_dim / k;
    const int64_t rows_per_split = dl_ceil_div(per_class, splits);
    const Rows kind = rows_kind<T>(batch, x);
    const int64_t gx = dl_ceil_div(kind == Rows::single ? batch : dl_ceil_div(batch, V), DL_WAVE);
    if (gx > 0x7fffffffLL || k > 65535) return DL_ERR_TOO_LARGE;
    const dim3 grid((unsigned) gx, (unsigned) k, (unsigned) splits);
    // More than the Infinity Cache holds is read past it: the rows of x that the layer before leaves there stay.  A training layer
    // with its GroupSum behind it, us with the sum's rows read ordinarily / past the cache: fp32 262 MB 131.5 / 129.8, 311 MB 162 / 157,
    // 344 MB 203 / 180, 410 MB 260 / 228, 524 MB 319 / 280, 819 MB 524 / 477, 1 GB 652 / 604; half 262 MB 141 / 144, 328 MB 197 / 180,
    // 524 MB 344 / 301; double 524 MB 308 / 266; whole steps of 784 -> 3 layers, fp32 303 MB 842 / 818, 393 MB 1132 / 1095, half 320 MB
    // 1104 / 1083.  (In a trace the kernel itself, 128000 rows at batch 1024, with eight rows in flight instead of four as well:
    // 134 -> 104 us.)
    const bool past = out_dim * batch * (int64_t) sizeof(T) >= 300000000;
#define DL_LAUNCH_PARTIAL_AS(VV, RAG, NT)                                                                              \
    DL_LAUNCH((group_sum_partial_kernel<T, VV, RAG, NT>), grid, dim3(DL_BLOCK), 0, s, (const T *) x, (C *) workspace,  \
              per_class, batch, k, rows_per_split)
#define DL_LAUNCH_PARTIAL(VV, RAG)                                                                                     \
    do {                                                                                                               \
        if (past) DL_LAUNCH_PARTIAL_AS(VV, RAG, true);                                                                 \
        else DL_LAUNCH_PARTIAL_AS(VV, RAG, false);                                                                     \
    } while (0)
    if (kind == Rows::whole) DL_LAUNCH_PARTIAL(V, false);
    else if (kind == Rows::ragged) DL_LAUNCH_PARTIAL(V, true);
    else DL_LAUNCH_PARTIAL(1, false);
#undef DL_LAUNCH_PARTIAL
#undef DL_LAUNCH_PARTIAL_AS
    int st = dl_launch_status();
    if (st != DL_OK) return st;
    const int64_t blocks = dl_ceil_div(batch, DL_WAVE);
    if (blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
    DL_LAUNCH((group_sum_finish_kernel<T>), dim3((unsigned) blocks, (unsigned) k), dim3(DL_BLOCK), 0, s,
                       (const C *) workspace, (T *) y, batch, k, splits, 1.0 / tau);
    return dl_launch_status();
}

template <typename T>
int group_sum_backward_t(const void *g, void *gx, int64_t out_dim, int64_t batch, int64_t k, double tau, hipStream_t s) {
    typedef typename Acc<T>::type C;
    constexpr int V = Vec16<T>::n;
    const Rows kind = rows_kind<T>(batch, gx);
    const int64_t gxd = dl_ceil_div(kind == Rows::single ? batch : dl_ceil_div(batch, V), DL_WAVE), gyd = dl_ceil_div(out_dim, 64);
    if (gxd > 0x7fffffffLL || gyd > 65535) return DL_ERR_TOO_LARGE;
    const dim3 grid((unsigned) gxd, (unsigned) gyd);
#define DL_LAUNCH_BROADCAST(VV, RAG)                                                                                    \
    DL_LAUNCH((group_sum_backward_kernel<T, VV, RAG>), grid, dim3(DL_BLOCK), 0, s, (const T *) g, (T *) gx, out_dim,   \
              out_dim / k, batch, k, (C) (1.0 / tau))
    if (kind == Rows::whole) DL_LAUNCH_BROADCAST(V, false);
    else if (kind == Rows::ragged) DL_LAUNCH_BROADCAST(V, true);
    else DL_LAUNCH_BROADCAST(1, false);
#undef DL_LAUNCH_BROADCAST
    return dl_launch_status();
}

int group_sum_splits(int64_t out_dim, int64_t batch, int64_t k);

template <typename T>
int forward_group_sum_t(const void *x, const int64_t *a, const int64_t *b, const void *w, void *probs, void *y,
                        void *workspace, int64_t out_dim, int64_t batch, int64_t k, double tau, hipStream_t s) {
    typedef typename Acc<T>::type C;
    constexpr int V = Vec16<T>::n;
    const int splits = group_sum_splits(out_dim, batch, k);
    const int64_t per_class = out_dim / k;
    const int64_t rows_per_split = dl_ceil_div(dl_ceil_div(per_class, splits), 16) * 16;     // whole groups of four per wave
    const Rows kind = rows_kind<T>(batch, x);
    const int64_t gx = dl_ceil_div(kind == Rows::single ? batch : dl_ceil_div(batch, V), DL_WAVE);
    if (gx > 0x7fffffffLL || k > 65535 || out_dim > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
    const dim3 grid((unsigned) gx, (unsigned) k, (unsigned) splits);
    const T *xp = (const T *) x, *wp = (const T *) w;
#define DL_LAUNCH_FGS(VV, RAG)                                                                                              \
    do {                                                                                                                    \
        if (probs)                                                                                                          \
            DL_LAUNCH((forward_group_sum_kernel<T, VV, true, RAG>), grid, dim3(DL_BLOCK), 0, s, xp, a, b, wp, (T *) probs,  \
                      (C *) workspace, per_class, batch, k, rows_per_split);                                                \
        else                                                                                                                \
            DL_LAUNCH((forward_group_sum_kernel<T, VV, false, RAG>), grid, dim3(DL_BLOCK), 0, s, xp, a, b, wp, (T *) probs, \
                      (C *) workspace, per_class, batch, k, rows_per_split);                                                \
    } while (0)
    if (kind == Rows::whole) DL_LAUNCH_FGS(V, false);
    else if (kind == Rows::ragged) DL_LAUNCH_FGS(V, true);
    else DL_LAUNCH_FGS(1, false);
#undef DL_LAUNCH_FGS
    int st = dl_launch_status();
    if (st != DL_OK) return st;
    const int64_t blocks = dl_ceil_div(batch, DL_WAVE);
    if (blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
    DL_LAUNCH((group_sum_finish_kernel<T>), dim3((unsigned) blocks, (unsigned) k), dim3(DL_BLOCK), 0, s,
                       (const C *) workspace, (T *) y, batch, k, splits, 1.0 / tau);
    return dl_launch_status();
}

// Number of row splits per class: enough workgroups to fill the chip, at least 32 rows each (64 / 32: layer and GroupSum on
// 8000 rows, 10 classes, batch 100 9.0 / 6.1 us; the GroupSum alone on 16000 rows at 500 7.3 / 8.5).  Twice the workgroups,
// with a finishing pass that waited for its loads one by one: GroupSum over 128000 rows at batch 1024 97 -> 90 us, but the
// finish over the partial sums of 64000 rows at 512 5.3 -> 9.0.
int group_sum_splits(int64_t out_dim, int64_t batch, int64_t k) {
    const int64_t per_class = out_dim / k;
    const int64_t col_tiles = dl_ceil_div(batch, 4 * DL_WAVE);
    int64_t want = dl_ceil_div(1024, col_tiles * k);
    const int64_t max_by_rows = per_class / 32 > 0 ? per_class / 32 : 1;
    if (want > max_by_rows) want = max_by_rows;
    if (want < 1) want = 1;
    if (want > 1024) want = 1024;
    return (int) want;
}

#define DL_TRAIN_CHUNK 8     // must equal the chunk the schedule was built with (dl_eval_schedule_chunk)
#define DL_FWD_ROWS_MIN 128  // vectors per row above which forward_chain_rows_kernel takes over

// Longest row (in 16-byte vectors) the whole-row kernels take: 16 segments of 256.
#define DL_ROWS_MAX_VECTORS (16 * 4 * DL_WAVE)

// Rows past the Infinity Cache (NT).  A walk reads every row of x (and of grad_y) once, and what it writes is what the next
// kernel reads.  Read the ordinary way, rows that nobody wants again push the new ones out of the 256 MB; written the ordinary
// way, 64 bytes of probabilities or weight gradients a neuron cost as much as half a kilobyte of rows (half a cache line each).
// Six square fp32 layers in a row, us a layer, ordinary / past the cache, by the bytes of x:
//   forward of training    31 MB 15.1 / 18.0, 51 MB 26.1 / 25.4, 66 MB 30.9 / 28.4, 131 MB 57 / 51, 262 MB 112 / 95, 524 MB 231 / 206,
//                          1 GB 452 / 452
//   discretised forward    66 MB 22.5 / 25.4, 131 MB 49.2 / 49.7, 179 MB 75 / 72, 262 MB 105 / 94, 524 MB 219 / 203, 1 GB 441 / 445
//   one-pass backward      66 MB 41.8 / 41.6, 98 MB 64 / 58, 131 MB 90 / 73, 262 MB 173 / 137, 524 MB 347 / 330, 1 GB 685 / 696
//   backward_w alone       131 MB 44 / 50, 179 MB 66 / 70, 262 MB 98 / 95, 524 MB 203 / 190, 1 GB 502 / 503
// (The discretised forward goes by the bytes of x and y: a layer that narrows, 80000 -> 40000 at batch 512, 164 MB and 82 MB,
// is still better off with both in the cache, three layers 112 / 117 us.)
// Half and double agree with that table at the same bytes (forward: half 64 MB 34.6 / 33.2, 98 MB 49 / 44, 262 MB 112 / 97, double 65 MB
// 33.0 / 30.6, 131 MB 61 / 54; one-pass backward: 131 MB 90 / 76 and 86 / 72, 262 MB 174 / 138 and 170 / 136), and so does the forward
// with given probabilities with the discretised one.  But a whole step of half or double gains by the forward pass only where its
// backward passes the cache as well, from 80 MB (784 -> 6 x 64000, a captured step: half 51 MB 435 / 443 us, 64 MB 508 / 514, 73 MB
// 637 / 643, 77 MB 657 / 650, 81 MB 657 / 637, 90 MB 795 / 776; double 51 MB 525 / 532, 76 MB 638 / 646, 81 MB 648 / 630); fp32 is
// the same either way below that (51 MB 404 / 406 as written and 341 / 343 fused, 65 MB 452 / 451 and 375 / 371, 76 MB 542 / 544 and
// 464 / 461).  In a trace, where kernels run one by one, the kernel behind one that passes the cache is up to a tenth
// longer (first layer of 9216 -> 4 x 128000 at batch 1024, backward_w 161 / 173; last layer with GroupSum 210 / 225); the step is
// shorter all the same (forward alone 2293 / 2201, backward alone 2260 / 2201).
// Smaller matrices stay in the caches from one kernel to the next; rows that are read several times (a layer much wider
// than its input, the classes' gradient rows) are read the ordinary way.
struct PastCache { int64_t from, to; };
constexpr PastCache DL_PAST_FORWARD = {50000000, INT64_MAX}, DL_PAST_FORWARD_HALF_DOUBLE = {80000000, INT64_MAX},
                    DL_PAST_ARGMAX = {280000000, 1400000000},
                    DL_PAST_BACKWARD = {80000000, 700000000}, DL_PAST_WEIGHTS = {240000000, INT64_MAX};

bool past_cache(PastCache limits, int64_t steps, int64_t in_dim, int64_t row_bytes, int64_t rows_written = 0) {
    const int64_t bytes = (in_dim + rows_written) * row_bytes;
    return 4 * steps <= 5 * in_dim && bytes >= limits.from && bytes <= limits.to;
}

int row_segments(int64_t ncols) { return (int) dl_ceil_div(ncols, 4 * DL_WAVE); }

// Steps per wave of the kernels in which a wave owns whole rows: long chunks re-read fewer rows at
// their seams, short ones give more waves to hide latency with; keep about three waves per SIMD.
int chain_chunk(int64_t steps) {
    for (int chunk = 32; chunk > 8; chunk /= 2)
        if (steps / chunk >= 3000) return chunk;
    return 8;
}

// ... of the one-pass backward of rows longer than 2 KB, whose 1024 SIMDs hold three waves each: a chunk is also long enough where
// its waves are there at once and spread evenly, at most two to a SIMD (1536 < waves <= 2048: chunks of half the length would
// need a second go) or mostly three (from 2560).  Square layers, us with chunks of 32 / 16, by the waves that 32 gives: fp32 at
// batch 1024 1500 (48000 wide) 111 / 103, 1531 112 / 105, 1562 113 / 120, 1750 120 / 129, 2000 138 / 142, 2250 181 / 171, 2500
// 193 / 190, 2562 197 / 202, 2750 211 / 222, 3000 233 / 242; at 600 1500 74 / 65, 1625 76 / 81, 2000 84 / 89, 2250 109 / 101, 2500
// 115 / 108, 2750 120 / 125; half at 1200 1750 101 / 102, 2000 103 / 105, 2500 149 / 130, 2625 149 / 148; at 2048 2562 211 / 209, 2625
// 214 / 222; double at 512 1750 121 / 131, 2500 196 / 191, 2625 202 / 215.  Chunks of 16 / 8, by the waves of 16: fp32 at 1024 1500
// (24000 wide) 58 / 55, 1750 62 / 68, 2062 84 / 80, 2500 93 / 91, 2562 93 / 94, 2750 97 / 103; half at 1200 2062 77 / 68, 2625 80 / 81.
int chain_chunk_long(int64_t steps) {
    for (int chunk = 32; chunk > 8; chunk /= 2) {
        const int64_t waves = steps / chunk;
        if (waves >= 2560 || (waves > 1536 && waves <= 2048)) return chunk;
    }
    return 8;
}

template <typename T, int GATES>
int forward_chain_t(const void *x, const int32_t *verts, const int32_t *neuron, const uint8_t *flip, int64_t steps,
                    const void *w, void *y, void *probs, int64_t in_dim, int64_t out_dim, int64_t batch, bool any_rows, hipStream_t s,
                    bool w32 = false) {
    constexpr int V = Vec16<T>::n;
    const Rows kind = rows_kind<T>(batch, x, y);
    if (kind != Rows::whole && !(any_rows && kind == Rows::ragged)) return DL_ERR_TOO_LARGE;
    const int64_t nchunks = steps / DL_TRAIN_CHUNK, ncols = dl_ceil_div(batch, V);
    const int64_t row_bytes = batch * (int64_t) sizeof(T);
    const bool past = probs ? past_cache(sizeof(T) == 4 ? DL_PAST_FORWARD : DL_PAST_FORWARD_HALF_DOUBLE, steps, in_dim, row_bytes)
                            : past_cache(DL_PAST_ARGMAX, steps, in_dim, row_bytes, out_dim);
    const T *xp = (const T *) x, *wp = (const T *) w;
    const dim3 block(DL_BLOCK);
    if (ncols > DL_FWD_ROWS_MIN && ncols <= DL_ROWS_MAX_VECTORS) {
        // rows of 2 KB and more: a wave takes whole rows, or segments of 4 KB
        const int segments = row_segments(ncols);
        const int chunk = chain_chunk(steps * segments);
        const int64_t blocks = dl_ceil_div(dl_ceil_div(steps, chunk), 4);
        if (blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
        const dim3 grid((unsigned) blocks, (unsigned) segments);
#define DL_LAUNCH_ROWS_AS(CPL, RAG, NT)                                                                                 \
    DL_LAUNCH((forward_chain_rows_kernel<T, V, CPL, GATES, RAG, NT>), grid, block, 0, s, xp, verts, neuron, flip, wp,   \
              (T *) y, (T *) probs, steps, chunk, batch, w32)
#define DL_LAUNCH_ROWS(CPL, RAG)                                                                                        \
    do {                                                                                                                \
        if (past) DL_LAUNCH_ROWS_AS(CPL, RAG, true);                                                                    \
        else DL_LAUNCH_ROWS_AS(CPL, RAG, false);                                                                        \
    } while (0)
        if (ncols <= 2 * DL_WAVE) {
            if (kind == Rows::whole) DL_LAUNCH_ROWS(2, false);
            else DL_LAUNCH_ROWS(2, true);
        } else {
            if (kind == Rows::whole) DL_LAUNCH_ROWS(4, false);
            else DL_LAUNCH_ROWS(4, true);
        }
#undef DL_LAUNCH_ROWS
#undef DL_LAUNCH_ROWS_AS
        return dl_launch_status();
    }
    const int64_t blocks = dl_ceil_div(nchunks, 4);
    if (blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
    constexpr int H = V >= 2 ? V / 2 : 1;
    // short rows: 8-byte vectors put a row on all 64 lanes instead of half of them
    const bool half = V >= 2 && ncols <= DL_WAVE / 2;
    const dim3 grid((unsigned) blocks, half ? 1 : col_tiles(ncols));
#define DL_LAUNCH_CHAIN_AS(VV, RAG, NT)                                                                                \
    DL_LAUNCH((forward_chain_kernel<T, VV, DL_TRAIN_CHUNK, GATES, RAG, NT>), grid, block, 0, s, xp, verts, neuron, flip, \
              wp, (T *) y, (T *) probs, nchunks, batch, w32)
#define DL_LAUNCH_CHAIN(VV, RAG)                                                                                       \
    do {                                                                                                               \
        if (past) DL_LAUNCH_CHAIN_AS(VV, RAG, true);                                                                   \
        else DL_LAUNCH_CHAIN_AS(VV, RAG, false);                                                                       \
    } while (0)
    if (half) {
        if (kind == Rows::whole) DL_LAUNCH_CHAIN(H, false);
        else DL_LAUNCH_CHAIN(H, true);
    } else {
        if (kind == Rows::whole) DL_LAUNCH_CHAIN(V, false);
        else DL_LAUNCH_CHAIN(V, true);
    }
#undef DL_LAUNCH_CHAIN
#undef DL_LAUNCH_CHAIN_AS
    return dl_launch_status();
}

template <typename T, bool LOGITS>
int forward_chain_lower_t(const void *lx, const int64_t *la, const int64_t *lb, const void *lw, void *lprobs,
                          const int32_t *verts, const int32_t *neuron, const uint8_t *flip, int64_t steps, const void *w,
                          void *y, void *probs, int64_t batch, bool any_rows, hipStream_t s) {
    constexpr int V = Vec16<T>::n;
    const Rows kind = rows_kind<T>(batch, lx, y);
    if (kind != Rows::whole && !(any_rows && kind == Rows::ragged)) return DL_ERR_TOO_LARGE;
    const int64_t nchunks = steps / DL_TRAIN_CHUNK, ncols = dl_ceil_div(batch, V);
    if (ncols > DL_FWD_ROWS_MIN) return DL_ERR_TOO_LARGE;        // rows of at most 2 KB
    const int64_t blocks = dl_ceil_div(nchunks, 4);
    if (blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
    // one wave takes every column tile of its chunk (at most two): the corner coefficients are formed once
#define DL_LAUNCH_LOWER(RAG)                                                                                            \
    DL_LAUNCH((forward_chain_lower_kernel<T, V, DL_TRAIN_CHUNK, LOGITS, RAG>), dim3((unsigned) blocks), dim3(DL_BLOCK), 0, \
              s, (const T *) lx, la, lb, (const T *) lw, (T *) lprobs, verts, neuron, flip, (const T *) w, (T *) y,      \
              (T *) probs, nchunks, batch)
    if (kind == Rows::whole) DL_LAUNCH_LOWER(false);
    else DL_LAUNCH_LOWER(true);
#undef DL_LAUNCH_LOWER
    return dl_launch_status();
}

template <typename T>
int backward_w_chain_t(const void *x, const int32_t *verts, const int32_t *neuron, const uint8_t *flip, int64_t steps,
                       const void *gy, const void *probs, void *gw, int64_t in_dim, int64_t batch, bool any_rows, hipStream_t s,
                       int64_t gdiv = 0, bool w32 = false) {
    constexpr int V = Vec16<T>::n;
    const Rows kind = rows_kind<T>(batch, x, gy);
    if (kind != Rows::whole && !(any_rows && kind == Rows::ragged)) return DL_ERR_TOO_LARGE;
    const int64_t nchunks = steps / DL_TRAIN_CHUNK, ncols = dl_ceil_div(batch, V);
    const int64_t blocks = dl_ceil_div(nchunks, 4);
    if (blocks > 0x7fffffffLL || ncols > 4 * DL_WAVE) return DL_ERR_TOO_LARGE;   // a lane holds at most 4 vectors of a row
    const bool past = gdiv == 0 && past_cache(DL_PAST_WEIGHTS, steps, in_dim, batch * (int64_t) sizeof(T));
#define DL_LAUNCH_W_CHAIN_AS(CPL, RAG, NT)                                                                             \
    DL_LAUNCH((backward_w_chain_kernel<T, V, CPL, DL_TRAIN_CHUNK, RAG, NT>), dim3((unsigned) blocks), dim3(DL_BLOCK),  \
              0, s, (const T *) x, verts, neuron, flip, (const T *) gy, (const T *) probs, (T *) gw, nchunks, batch, gdiv, w32)
#define DL_LAUNCH_W_CHAIN(CPL)                                                                                         \
    do {                                                                                                               \
        if (kind == Rows::whole && past) DL_LAUNCH_W_CHAIN_AS(CPL, false, true);                                       \
        else if (kind == Rows::whole) DL_LAUNCH_W_CHAIN_AS(CPL, false, false);                                         \
        else if (past) DL_LAUNCH_W_CHAIN_AS(CPL, true, true);                                                          \
        else DL_LAUNCH_W_CHAIN_AS(CPL, true, false);                                                                   \
    } while (0)
    if (ncols <= DL_WAVE) DL_LAUNCH_W_CHAIN(1);
    else if (ncols <= 2 * DL_WAVE) DL_LAUNCH_W_CHAIN(2);
    else DL_LAUNCH_W_CHAIN(4);
#undef DL_LAUNCH_W_CHAIN
#undef DL_LAUNCH_W_CHAIN_AS
    return dl_launch_status();
}

// Vertices (and overflow rows) up to which the one-pass backward finishes them in its own launch.  Each costs four row reads
// instead of a written and a read row; the launch that goes takes 4 to 5 us a layer (784 -> 4 x 64000, a captured step at
// batch 100: fp32 fused 187 -> 167 us with the pair's second launch gone too, half 226 -> 213).  (A vertex of many positions is
// one wave's serial work: the caller says DL_FIX_POSITIONS where there is none.)
constexpr int64_t DL_FIX_HERE = 64;

template <typename T> int64_t backward_partial_bytes(int64_t out_dim, int64_t batch) {
    constexpr int V = Vec16<T>::n;
    const int segments = row_segments(dl_ceil_div(batch, V));
    return segments > 1 ? (int64_t) segments * out_dim * 4 * (int64_t) sizeof(typename Acc<T>::type) : 0;
}

template <typename T>
int backward_chain_t(const void *x, const int32_t *verts, const int32_t *neuron, const uint8_t *flip, const int32_t *dst,
                     int64_t steps, const void *w, const void *gy, bool softmax_backward, const int32_t *fix_vertex,
                     const int32_t *fix_start, int64_t n_fix, int64_t overflow_rows, void *gw, void *gx, void *workspace,
                     int64_t in_dim, int64_t out_dim, int64_t batch, double scale, bool any_rows, bool fix_positions, hipStream_t s,
                     int64_t gdiv = 0, const LowerLayer<T> *lower = nullptr, bool w32 = false) {
    typedef typename Acc<T>::type C;
    constexpr int V = Vec16<T>::n;
    Rows kind = rows_kind<T>(batch, x, gy, gx, workspace);
    if (kind == Rows::whole && lower && !dl_aligned(lower->x, 16)) kind = Rows::ragged;
    if (kind != Rows::whole && !(any_rows && kind == Rows::ragged)) return DL_ERR_TOO_LARGE;
    if (!dl_aligned(workspace, 16)) return DL_ERR_TOO_LARGE;            // partial sums of whole C values lie at its start
    if (!x && (!lower || !lower->w)) return DL_ERR_INVALID_ARGUMENT;     // x may only be left out for recomputation
    const int64_t ncols = dl_ceil_div(batch, V);
    if (ncols > DL_ROWS_MAX_VECTORS) return DL_ERR_TOO_LARGE;
    const int segments = row_segments(ncols);
    // with `lower`: whole rows per wave only, and gx holds the n_fix rows that finish after the pass
    if (lower && (segments > 1 || w32)) return DL_ERR_TOO_LARGE;
    const LowerLayer<T> none = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    // workspace: [segments x out x 4 corner sums (only with several segments)] [overflow rows]
    const int64_t partial_bytes = backward_partial_bytes<T>(out_dim, batch);
    if ((partial_bytes > 0 || overflow_rows > 0) && workspace == nullptr) return DL_ERR_INVALID_ARGUMENT;
    C *partial = partial_bytes > 0 ? (C *) workspace : nullptr;
    C *overflow = (C *) ((char *) workspace + partial_bytes);
    const int chunk = ncols > 2 * DL_WAVE ? chain_chunk_long(steps * segments) : chain_chunk(steps * segments);
    const int64_t blocks = dl_ceil_div(dl_ceil_div(steps, chunk), 4), fix_blocks = dl_ceil_div(n_fix, 4);
    if (blocks > 0x7fffffffLL || fix_blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
    // a few vertices are finished by further workgroups of the same launch; many are cheaper through overflow rows
    const bool here = fix_positions && n_fix > 0 && n_fix <= DL_FIX_HERE && overflow_rows <= DL_FIX_HERE && blocks + fix_blocks <= 0x7fffffffLL;
    const FixHere fix = {fix_vertex, fix_start, here ? fix_start + n_fix + 1 : nullptr, here ? (int) n_fix : 0, (uint32_t) blocks};
    const dim3 grid((unsigned) (blocks + (here ? fix_blocks : 0)), (unsigned) segments), block(DL_BLOCK);
    const T *xp = (const T *) x, *wp = (const T *) w, *gp = (const T *) gy, *pp = softmax_backward ? wp : nullptr;
    constexpr int H = V >= 2 ? V / 2 : 1;
    const bool past = gdiv == 0 && past_cache(DL_PAST_BACKWARD, steps, in_dim, batch * (int64_t) sizeof(T));
#define DL_LAUNCH_BACKWARD_CHAIN_AS(VV, CPL, LOWER, RAG, NT)                                                             \
    DL_LAUNCH((backward_chain_kernel<T, VV, CPL, LOWER, RAG, NT>), grid, block, 0, s, xp, verts, neuron, flip, dst, wp, gp, \
              pp, (T *) gw, partial, (T *) gx, overflow, steps, chunk, in_dim, out_dim, batch, (C) scale, gdiv,         \
              LOWER ? *lower : none, fix, LOWER ? false : w32)
#define DL_LAUNCH_BACKWARD_CHAIN_RAG(VV, CPL, RAG, NT)                                                                   \
    do {                                                                                                                 \
        if (lower && !x) {                           /* (half has been refused: its rows are not recomputed) */          \
            if constexpr (sizeof(T) != 2) DL_LAUNCH_BACKWARD_CHAIN_AS(VV, CPL, 2, RAG, NT);                              \
        }                                                                                                                \
        else if (lower) DL_LAUNCH_BACKWARD_CHAIN_AS(VV, CPL, 1, RAG, NT);                                                \
        else DL_LAUNCH_BACKWARD_CHAIN_AS(VV, CPL, 0, RAG, NT);                                                           \
    } while (0)
#define DL_LAUNCH_BACKWARD_CHAIN(VV, CPL)                                                                                \
    do {                                                                                                                 \
        if (kind == Rows::whole && past) DL_LAUNCH_BACKWARD_CHAIN_RAG(VV, CPL, false, true);                             \
        else if (kind == Rows::whole) DL_LAUNCH_BACKWARD_CHAIN_RAG(VV, CPL, false, false);                               \
        else if (past) DL_LAUNCH_BACKWARD_CHAIN_RAG(VV, CPL, true, true);                                                \
        else DL_LAUNCH_BACKWARD_CHAIN_RAG(VV, CPL, true, false);                                                         \
    } while (0)
    if (V >= 2 && ncols <= DL_WAVE / 2)
        DL_LAUNCH_BACKWARD_CHAIN(H, 1);              // short rows: 8-byte vectors use all 64 lanes
    else if (ncols <= DL_WAVE)
        DL_LAUNCH_BACKWARD_CHAIN(V, 1);
    else if (ncols <= 2 * DL_WAVE)
        DL_LAUNCH_BACKWARD_CHAIN(V, 2);
    else
        DL_LAUNCH_BACKWARD_CHAIN(V, 4);
#undef DL_LAUNCH_BACKWARD_CHAIN_AS
#undef DL_LAUNCH_BACKWARD_CHAIN_RAG
#undef DL_LAUNCH_BACKWARD_CHAIN
    int st = dl_launch_status();
    if (st != DL_OK) return st;
    if (partial != nullptr) {
        const int64_t fin_blocks = dl_ceil_div(out_dim, 16);
        if (fin_blocks > 0x7fffffffLL) return DL_ERR_TOO_LARGE;
        DL_LAUNCH(backward_w_finish_kernel<T>, dim3((unsigned) fin_blocks), block, 0, s, (const C *) partial, pp, (T *) gw,
                  out_dim, segments, w32);
        st = dl_launch_status();
        if (st != DL_OK) return st;
    }
    if (n_fix == 0 || here) return DL_OK;
    const dim3 fix_grid((unsigned) fix_blocks, col_tiles(ncols));
    const C fix_scale = sizeof(T) == sizeof(C) ? (C) 1 : (C) scale;
    if (kind == Rows::whole)
        DL_LAUNCH((backward_fix_kernel<T, V, false>), fix_grid, block, 0, s, (const C *) overflow, fix_vertex, fix_start,
                  (T *) gx, n_fix, batch, fix_scale, lower != nullptr);
    else
        DL_LAUNCH((backward_fix_kernel<T, V, true>), fix_grid, block, 0, s, (const C *) overflow, fix_vertex, fix_start,
                  (T *) gx, n_fix, batch, fix_scale, lower != nullptr);
    st = dl_launch_status();
    if (st != DL_OK || !lower) return st;
    if (kind == Rows::whole)
        DL_LAUNCH((backward_w_rows_kernel<T, V, false>), dim3((unsigned) fix_blocks), block, 0, s, *lower, fix_vertex,
                  (const T *) gx, n_fix, batch);
    else
        DL_LAUNCH((backward_w_rows_kernel<T, V, true>), dim3((unsigned) fix_blocks), block, 0, s, *lower, fix_vertex,
                  (const T *) gx, n_fix, batch);
    return dl_launch_status();
}

// DL_F16_W32 / DL_F64_W32 (activations in half / double, gate weights and their gradients in fp32) -> the
// activations' dtype; returns whether the weights are fp32
bool weights_fp32(int &dtype) {
    if (dtype == DL_F16_W32) {
        dtype = DL_F16;
        return true;
    }
    if (dtype == DL_F64_W32) {
        dtype = DL_F64;
        return true;
    }
    return false;
}

// DL_GATES_OF_ARGMAX in a dtype code: taken out of it, and returned
bool gates_argmax(int &dtype) {
    const bool argmax = (dtype & DL_GATES_OF_ARGMAX) != 0;
    dtype &= ~DL_GATES_OF_ARGMAX;
    return argmax;
}

// DL_FIX_POSITIONS in a dtype code: taken out of it, and returned
bool takes_fix_positions(int &dtype) {
    const bool there = (dtype & DL_FIX_POSITIONS) != 0;
    dtype &= ~DL_FIX_POSITIONS;
    return there;
}

// DL_ROWS_ANY in a dtype code: taken out of it, and returned
bool takes_any_rows(int &dtype) {
    const bool any = (dtype & DL_ROWS_ANY) != 0;
    dtype &= ~DL_ROWS_ANY;
    return any;
}

}  // namespace

extern "C" int64_t dl_logic_backward_chained_workspace_bytes(int64_t overflow_rows, int64_t out_dim, int64_t batch,
                                                             int dtype) {
    if (overflow_rows < 0 || out_dim < 0 || batch < 0) return -DL_ERR_INVALID_ARGUMENT;
    takes_any_rows(dtype);
    takes_fix_positions(dtype);
    weights_fp32(dtype);
    switch (dtype) {
    case DL_F16: return backward_partial_bytes<__half>(out_dim, batch) + overflow_rows * batch * 4;    // parts in fp32
    case DL_F32: return backward_partial_bytes<float>(out_dim, batch) + overflow_rows * batch * 4;
    case DL_F64: return backward_partial_bytes<double>(out_dim, batch) + overflow_rows * batch * 8;
    default: return -DL_ERR_DTYPE;
    }
}

extern "C" int dl_logic_backward_chained(const void *x, const int32_t *verts, const int32_t *neuron, const uint8_t *flip,
                                         const int32_t *dst, int64_t steps, const void *w, const void *grad_y,
                                         int softmax_backward, const int32_t *fix_vertex, const int32_t *fix_start,
                                         int64_t n_fix, int64_t overflow_rows, void *grad_w, void *grad_x,
                                         void *workspace, int64_t in_dim, int64_t out_dim, int64_t batch, double scale,
                                         int dtype, void *stream) {
    const bool any = takes_any_rows(dtype), fp = takes_fix_positions(dtype), w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim <= 0 || out_dim <= 0 || batch <= 0 || steps < out_dim || n_fix < 0 || n_fix > in_dim || overflow_rows < 0)
        return DL_ERR_INVALID_ARGUMENT;
    if (!x || !verts || !neuron || !flip || !dst || !w || !grad_y || !grad_w || !grad_x) return DL_ERR_INVALID_ARGUMENT;
    if (n_fix > 0 && (!fix_vertex || !fix_start)) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    const bool sb = softmax_backward != 0;
    switch (dtype) {
    case DL_F16:
        return backward_chain_t<__half>(x, verts, neuron, flip, dst, steps, w, grad_y, sb, fix_vertex, fix_start, n_fix,
                                        overflow_rows, grad_w, grad_x, workspace, in_dim, out_dim, batch, scale, any, fp, s, 0, nullptr,
                                        w32);
    case DL_F32:
        return backward_chain_t<float>(x, verts, neuron, flip, dst, steps, w, grad_y, sb, fix_vertex, fix_start, n_fix,
                                       overflow_rows, grad_w, grad_x, workspace, in_dim, out_dim, batch, scale, any, fp, s);
    default:
        return backward_chain_t<double>(x, verts, neuron, flip, dst, steps, w, grad_y, sb, fix_vertex, fix_start, n_fix,
                                        overflow_rows, grad_w, grad_x, workspace, in_dim, out_dim, batch, scale, any, fp, s, 0, nullptr,
                                        w32);
    }
}

extern "C" int dl_logic_backward_chained_lower(const void *x, const int32_t *verts, const int32_t *neuron,
                                               const uint8_t *flip, const int32_t *dst, int64_t steps, const void *w,
                                               const void *grad_y, int softmax_backward, const int32_t *fix_vertex,
                                               const int32_t *fix_start, int64_t n_fix, int64_t overflow_rows,
                                               void *grad_w, void *fix_rows, void *workspace, const void *x_lower,
                                               const int64_t *a_lower, const int64_t *b_lower, const void *w_lower,
                                               int softmax_backward_lower, void *grad_w_lower, int64_t in_dim,
                                               int64_t out_dim, int64_t batch, double scale, int dtype, void *stream) {
    const bool any = takes_any_rows(dtype);
    const bool fp = takes_fix_positions(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim <= 0 || out_dim <= 0 || batch <= 0 || steps < out_dim || n_fix < 0 || n_fix > in_dim || overflow_rows < 0)
        return DL_ERR_INVALID_ARGUMENT;
    if (!verts || !neuron || !flip || !dst || !w || !grad_y || !grad_w || !x_lower || !a_lower || !b_lower || !grad_w_lower)
        return DL_ERR_INVALID_ARGUMENT;
    if ((softmax_backward_lower || !x) && !w_lower) return DL_ERR_INVALID_ARGUMENT;
    if (n_fix > 0 && (!fix_vertex || !fix_start || !fix_rows)) return DL_ERR_INVALID_ARGUMENT;
    // recomputing x needs the lower layer's probabilities exactly as its forward pass used them; the fp16 kernels
    // form them in fp32 and round only what they store
    if (!x && dtype == DL_F16) return DL_ERR_TOO_LARGE;
    hipStream_t s = (hipStream_t) stream;
    const bool sb = softmax_backward != 0;
    switch (dtype) {
    case DL_F16: {
        const LowerLayer<__half> low = {(const __half *) x_lower, a_lower, b_lower, (const __half *) w_lower,
                                        softmax_backward_lower ? (const __half *) w_lower : nullptr, (__half *) grad_w_lower};
        return backward_chain_t<__half>(x, verts, neuron, flip, dst, steps, w, grad_y, sb, fix_vertex, fix_start, n_fix,
                                        overflow_rows, grad_w, fix_rows, workspace, in_dim, out_dim, batch, scale, any, fp, s, 0, &low);
    }
    case DL_F32: {
        const LowerLayer<float> low = {(const float *) x_lower, a_lower, b_lower, (const float *) w_lower,
                                       softmax_backward_lower ? (const float *) w_lower : nullptr, (float *) grad_w_lower};
        return backward_chain_t<float>(x, verts, neuron, flip, dst, steps, w, grad_y, sb, fix_vertex, fix_start, n_fix,
                                       overflow_rows, grad_w, fix_rows, workspace, in_dim, out_dim, batch, scale, any, fp, s, 0, &low);
    }
    default: {
        const LowerLayer<double> low = {(const double *) x_lower, a_lower, b_lower, (const double *) w_lower,
                                        softmax_backward_lower ? (const double *) w_lower : nullptr, (double *) grad_w_lower};
        return backward_chain_t<double>(x, verts, neuron, flip, dst, steps, w, grad_y, sb, fix_vertex, fix_start, n_fix,
                                        overflow_rows, grad_w, fix_rows, workspace, in_dim, out_dim, batch, scale, any, fp, s, 0, &low);
    }
    }
}

extern "C" int dl_logic_forward_chained(const void *x, const int32_t *verts, const int32_t *neuron, const uint8_t *flip,
                                        int64_t steps, const void *w, void *y, void *probs, int64_t in_dim,
                                        int64_t out_dim, int64_t batch, int dtype, void *stream) {
    const bool any = takes_any_rows(dtype), argmax = gates_argmax(dtype), w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim < 0 || out_dim < 0 || batch <= 0 || steps < out_dim || steps % DL_TRAIN_CHUNK != 0)
        return DL_ERR_INVALID_ARGUMENT;
    if (argmax && probs) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim == 0) return DL_OK;
    if (!x || !verts || !neuron || !flip || !w || !y || in_dim == 0) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    if (probs) {
        switch (dtype) {
        case DL_F16: return forward_chain_t<__half, true>(x, verts, neuron, flip, steps, w, y, probs, in_dim, out_dim, batch, any, s, w32);
        case DL_F32: return forward_chain_t<float, true>(x, verts, neuron, flip, steps, w, y, probs, in_dim, out_dim, batch, any, s);
        default: return forward_chain_t<double, true>(x, verts, neuron, flip, steps, w, y, probs, in_dim, out_dim, batch, any, s, w32);
        }
    }
    if (argmax) {
        switch (dtype) {
        case DL_F16: return forward_chain_t<__half, GATES_ARGMAX>(x, verts, neuron, flip, steps, w, y, nullptr, in_dim, out_dim, batch, any, s, w32);
        case DL_F32: return forward_chain_t<float, GATES_ARGMAX>(x, verts, neuron, flip, steps, w, y, nullptr, in_dim, out_dim, batch, any, s);
        default: return forward_chain_t<double, GATES_ARGMAX>(x, verts, neuron, flip, steps, w, y, nullptr, in_dim, out_dim, batch, any, s, w32);
        }
    }
    switch (dtype) {
    case DL_F16: return forward_chain_t<__half, false>(x, verts, neuron, flip, steps, w, y, nullptr, in_dim, out_dim, batch, any, s, w32);
    case DL_F32: return forward_chain_t<float, false>(x, verts, neuron, flip, steps, w, y, nullptr, in_dim, out_dim, batch, any, s);
    default: return forward_chain_t<double, false>(x, verts, neuron, flip, steps, w, y, nullptr, in_dim, out_dim, batch, any, s, w32);
    }
}

extern "C" int dl_logic_forward_chained_lower(const void *x_lower, const int64_t *a_lower, const int64_t *b_lower,
                                              const void *w_lower, void *probs_lower, const int32_t *verts,
                                              const int32_t *neuron, const uint8_t *flip, int64_t steps, const void *w,
                                              void *y, void *probs, int64_t in_dim_lower, int64_t in_dim, int64_t out_dim,
                                              int64_t batch, int dtype, void *stream) {
    const bool any = takes_any_rows(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim_lower <= 0 || in_dim <= 0 || out_dim < 0 || batch <= 0 || steps < out_dim || steps % DL_TRAIN_CHUNK != 0)
        return DL_ERR_INVALID_ARGUMENT;
    if (out_dim == 0) return DL_OK;
    if (!x_lower || !a_lower || !b_lower || !w_lower || !verts || !neuron || !flip || !w || !y) return DL_ERR_INVALID_ARGUMENT;
    if ((probs == nullptr) != (probs_lower == nullptr)) return DL_ERR_INVALID_ARGUMENT;    // both layers on logits, or neither
    hipStream_t s = (hipStream_t) stream;
#define DL_FCL(TT, LG)                                                                                                  \
    forward_chain_lower_t<TT, LG>(x_lower, a_lower, b_lower, w_lower, probs_lower, verts, neuron, flip, steps, w, y, probs, \
                                  batch, any, s)
    if (probs) {
        switch (dtype) {
        case DL_F16: return DL_FCL(__half, true);
        case DL_F32: return DL_FCL(float, true);
        default: return DL_FCL(double, true);
        }
    }
    switch (dtype) {
    case DL_F16: return DL_FCL(__half, false);
    case DL_F32: return DL_FCL(float, false);
    default: return DL_FCL(double, false);
    }
#undef DL_FCL
}

extern "C" int dl_logic_backward_w_chained(const void *x, const int32_t *verts, const int32_t *neuron,
                                           const uint8_t *flip, int64_t steps, const void *grad_y, const void *probs,
                                           void *grad_w, int64_t in_dim, int64_t out_dim, int64_t batch, int dtype,
                                           void *stream) {
    const bool any = takes_any_rows(dtype), w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim < 0 || out_dim < 0 || batch <= 0 || steps < out_dim || steps % DL_TRAIN_CHUNK != 0)
        return DL_ERR_INVALID_ARGUMENT;
    if (out_dim == 0) return DL_OK;
    if (!x || !verts || !neuron || !flip || !grad_y || !grad_w || in_dim == 0) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    switch (dtype) {
    case DL_F16: return backward_w_chain_t<__half>(x, verts, neuron, flip, steps, grad_y, probs, grad_w, in_dim, batch, any, s, 0, w32);
    case DL_F32: return backward_w_chain_t<float>(x, verts, neuron, flip, steps, grad_y, probs, grad_w, in_dim, batch, any, s);
    default: return backward_w_chain_t<double>(x, verts, neuron, flip, steps, grad_y, probs, grad_w, in_dim, batch, any, s, 0, w32);
    }
}

extern "C" int dl_logic_forward(const void *x, const int64_t *a, const int64_t *b, const void *w, void *y,
                                int64_t in_dim, int64_t out_dim, int64_t batch, int dtype, void *stream) {
    const bool argmax = gates_argmax(dtype), w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim < 0 || out_dim < 0 || batch < 0) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim == 0 || batch == 0) return DL_OK;
    if (!x || !a || !b || !w || !y || in_dim == 0) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    if (argmax) {
        switch (dtype) {
        case DL_F16: return forward_t<__half, GATES_ARGMAX>(x, a, b, w, y, nullptr, out_dim, batch, s, w32);
        case DL_F32: return forward_t<float, GATES_ARGMAX>(x, a, b, w, y, nullptr, out_dim, batch, s);
        default: return forward_t<double, GATES_ARGMAX>(x, a, b, w, y, nullptr, out_dim, batch, s, w32);
        }
    }
    switch (dtype) {
    case DL_F16: return forward_t<__half, false>(x, a, b, w, y, nullptr, out_dim, batch, s, w32);
    case DL_F32: return forward_t<float, false>(x, a, b, w, y, nullptr, out_dim, batch, s);
    default: return forward_t<double, false>(x, a, b, w, y, nullptr, out_dim, batch, s, w32);
    }
}

extern "C" int dl_logic_forward_logits(const void *x, const int64_t *a, const int64_t *b, const void *logits, void *y,
                                       void *probs, int64_t in_dim, int64_t out_dim, int64_t batch, int dtype,
                                       void *stream) {
    const bool w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim < 0 || out_dim < 0 || batch <= 0) return DL_ERR_INVALID_ARGUMENT;   // probs are written by column tile 0
    if (out_dim == 0) return DL_OK;
    if (!x || !a || !b || !logits || !y || !probs || in_dim == 0) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    switch (dtype) {
    case DL_F16: return forward_t<__half, true>(x, a, b, logits, y, probs, out_dim, batch, s, w32);
    case DL_F32: return forward_t<float, true>(x, a, b, logits, y, probs, out_dim, batch, s);
    default: return forward_t<double, true>(x, a, b, logits, y, probs, out_dim, batch, s, w32);
    }
}

extern "C" int dl_logic_backward_w(const void *x, const int64_t *a, const int64_t *b, const void *grad_y,
                                   void *grad_w, int64_t in_dim, int64_t out_dim, int64_t batch, int dtype,
                                   void *stream) {
    const bool w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim < 0 || out_dim < 0 || batch < 0) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim == 0) return DL_OK;
    if (!a || !b || !grad_w || in_dim == 0) return DL_ERR_INVALID_ARGUMENT;
    if (batch > 0 && (!x || !grad_y)) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    switch (dtype) {
    case DL_F16: return backward_w_t<__half>(x, a, b, grad_y, nullptr, grad_w, out_dim, batch, s, 0, w32);
    case DL_F32: return backward_w_t<float>(x, a, b, grad_y, nullptr, grad_w, out_dim, batch, s);
    default: return backward_w_t<double>(x, a, b, grad_y, nullptr, grad_w, out_dim, batch, s, 0, w32);
    }
}

extern "C" int dl_logic_backward_logits(const void *x, const int64_t *a, const int64_t *b, const void *grad_y,
                                        const void *probs, void *grad_logits, int64_t in_dim, int64_t out_dim,
                                        int64_t batch, int dtype, void *stream) {
    const bool w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim < 0 || out_dim < 0 || batch < 0) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim == 0) return DL_OK;
    if (!a || !b || !probs || !grad_logits || in_dim == 0) return DL_ERR_INVALID_ARGUMENT;
    if (batch > 0 && (!x || !grad_y)) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    switch (dtype) {
    case DL_F16: return backward_w_t<__half>(x, a, b, grad_y, probs, grad_logits, out_dim, batch, s, 0, w32);
    case DL_F32: return backward_w_t<float>(x, a, b, grad_y, probs, grad_logits, out_dim, batch, s);
    default: return backward_w_t<double>(x, a, b, grad_y, probs, grad_logits, out_dim, batch, s, 0, w32);
    }
}

extern "C" int dl_logic_backward_x(const void *x, const int64_t *a, const int64_t *b, const void *w,
                                   const void *grad_y, const int64_t *start, const int64_t *idx, void *grad_x,
                                   int64_t in_dim, int64_t out_dim, int64_t batch, double scale, int dtype,
                                   void *stream) {
    const bool w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim < 0 || out_dim < 0 || batch < 0) return DL_ERR_INVALID_ARGUMENT;
    if (in_dim == 0 || batch == 0) return DL_OK;
    if (!x || !grad_x || !start) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim > 0 && (!a || !b || !w || !grad_y || !idx)) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    switch (dtype) {
    case DL_F16: return backward_x_t<__half>(x, a, b, w, grad_y, start, idx, grad_x, in_dim, batch, scale, s, 0, w32);
    case DL_F32: return backward_x_t<float>(x, a, b, w, grad_y, start, idx, grad_x, in_dim, batch, scale, s);
    default: return backward_x_t<double>(x, a, b, w, grad_y, start, idx, grad_x, in_dim, batch, scale, s, 0, w32);
    }
}

extern "C" int dl_logic_backward_both(const void *x, const int64_t *a, const int64_t *b, const void *w, const void *grad_y,
                                      int softmax_backward, const int64_t *start, const int64_t *idx, void *grad_w,
                                      void *grad_x, int64_t in_dim, int64_t out_dim, int64_t batch, int64_t k, double scale,
                                      int dtype, void *stream) {
    const bool w32 = weights_fp32(dtype);
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim <= 0 || out_dim <= 0 || batch <= 0 || k < 0) return DL_ERR_INVALID_ARGUMENT;
    if (k > 0 && out_dim % k != 0) return DL_ERR_NOT_DIVISIBLE;
    if (k > 0 && out_dim > 0xffffffffLL) return DL_ERR_TOO_LARGE;            // class of a neuron by 32-bit division
    if (!x || !a || !b || !w || !grad_y || !start || !idx || !grad_w || !grad_x) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    const bool sb = softmax_backward != 0;
    const int64_t gdiv = k > 0 ? out_dim / k : 0;
    switch (dtype) {
    case DL_F16:
        return backward_both_t<__half>(x, a, b, w, grad_y, sb, start, idx, grad_w, grad_x, in_dim, out_dim, batch, scale, s,
                                       gdiv, w32);
    case DL_F32:
        return backward_both_t<float>(x, a, b, w, grad_y, sb, start, idx, grad_w, grad_x, in_dim, out_dim, batch, scale, s,
                                      gdiv, w32);
    default:
        return backward_both_t<double>(x, a, b, w, grad_y, sb, start, idx, grad_w, grad_x, in_dim, out_dim, batch, scale, s,
                                       gdiv, w32);
    }
}

extern "C" int64_t dl_group_sum_workspace_bytes(int64_t out_dim, int64_t batch, int64_t k, int dtype) {
    if (out_dim < 0 || batch < 0 || k <= 0 || out_dim % k != 0) return 0;
    const int64_t elem = dtype == DL_F64 ? 8 : 4;
    return (int64_t) group_sum_splits(out_dim, batch, k) * k * batch * elem;
}

extern "C" int dl_group_sum_forward(const void *x, void *y, void *workspace, int64_t out_dim, int64_t batch, int64_t k,
                                    double tau, int dtype, void *stream) {
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (out_dim < 0 || batch < 0 || k <= 0 || tau == 0.0) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim % k != 0) return DL_ERR_NOT_DIVISIBLE;
    if (batch == 0) return DL_OK;
    if (!y || !workspace || (out_dim > 0 && !x)) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    const int splits = group_sum_splits(out_dim, batch, k);
    switch (dtype) {
    case DL_F16: return group_sum_forward_t<__half>(x, y, workspace, out_dim, batch, k, splits, tau, s);
    case DL_F32: return group_sum_forward_t<float>(x, y, workspace, out_dim, batch, k, splits, tau, s);
    default: return group_sum_forward_t<double>(x, y, workspace, out_dim, batch, k, splits, tau, s);
    }
}

extern "C" int dl_group_sum_backward(const void *grad_y, void *grad_x, int64_t out_dim, int64_t batch, int64_t k,
                                     double tau, int dtype, void *stream) {
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (out_dim < 0 || batch < 0 || k <= 0 || tau == 0.0) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim % k != 0) return DL_ERR_NOT_DIVISIBLE;
    if (batch == 0 || out_dim == 0) return DL_OK;
    if (!grad_y || !grad_x) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    switch (dtype) {
    case DL_F16: return group_sum_backward_t<__half>(grad_y, grad_x, out_dim, batch, k, tau, s);
    case DL_F32: return group_sum_backward_t<float>(grad_y, grad_x, out_dim, batch, k, tau, s);
    default: return group_sum_backward_t<double>(grad_y, grad_x, out_dim, batch, k, tau, s);
    }
}

// ---- the last LogicLayer fused with GroupSum (training mode) --------------------------------

extern "C" int dl_logic_forward_group_sum(const void *x, const int64_t *a, const int64_t *b, const void *w, void *probs,
                                          void *y, void *workspace, int64_t in_dim, int64_t out_dim, int64_t batch,
                                          int64_t k, double tau, int dtype, void *stream) {
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim <= 0 || out_dim <= 0 || batch <= 0 || k <= 0 || !(tau != 0.0)) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim % k != 0) return DL_ERR_NOT_DIVISIBLE;
    if (!x || !a || !b || !w || !y || !workspace) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    switch (dtype) {
    case DL_F16: return forward_group_sum_t<__half>(x, a, b, w, probs, y, workspace, out_dim, batch, k, tau, s);
    case DL_F32: return forward_group_sum_t<float>(x, a, b, w, probs, y, workspace, out_dim, batch, k, tau, s);
    default: return forward_group_sum_t<double>(x, a, b, w, probs, y, workspace, out_dim, batch, k, tau, s);
    }
}

static int grouped_args(int64_t in_dim, int64_t out_dim, int64_t batch, int64_t k, int dtype) {
    if (dtype != DL_F16 && dtype != DL_F32 && dtype != DL_F64) return DL_ERR_DTYPE;
    if (in_dim <= 0 || out_dim <= 0 || batch <= 0 || k <= 0) return DL_ERR_INVALID_ARGUMENT;
    if (out_dim % k != 0) return DL_ERR_NOT_DIVISIBLE;
    if (out_dim > 0xffffffffLL) return DL_ERR_TOO_LARGE;          // class of a neuron by 32-bit division
    return DL_OK;
}

extern "C" int dl_logic_backward_logits_grouped(const void *x, const int64_t *a, const int64_t *b, const void *grad_cls,
                                                const void *probs, void *grad_w, int64_t in_dim, int64_t out_dim,
                                                int64_t batch, int64_t k, int dtype, void *stream) {
    const int st = grouped_args(in_dim, out_dim, batch, k, dtype);
    if (st != DL_OK) return st;
    if (!x || !a || !b || !grad_cls || !grad_w) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    const int64_t per_class = out_dim / k;
    switch (dtype) {
    case DL_F16: return backward_w_t<__half>(x, a, b, grad_cls, probs, grad_w, out_dim, batch, s, per_class);
    case DL_F32: return backward_w_t<float>(x, a, b, grad_cls, probs, grad_w, out_dim, batch, s, per_class);
    default: return backward_w_t<double>(x, a, b, grad_cls, probs, grad_w, out_dim, batch, s, per_class);
    }
}

extern "C" int dl_logic_backward_x_grouped(const void *x, const int64_t *a, const int64_t *b, const void *w,
                                           const void *grad_cls, const int64_t *start, const int64_t *idx, void *grad_x,
                                           int64_t in_dim, int64_t out_dim, int64_t batch, int64_t k, double scale,
                                           int dtype, void *stream) {
    const int st = grouped_args(in_dim, out_dim, batch, k, dtype);
    if (st != DL_OK) return st;
    if (!x || !a || !b || !w || !grad_cls || !start || !idx || !grad_x) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    const int64_t per_class = out_dim / k;
    switch (dtype) {
    case DL_F16: return backward_x_t<__half>(x, a, b, w, grad_cls, start, idx, grad_x, in_dim, batch, scale, s, per_class);
    case DL_F32: return backward_x_t<float>(x, a, b, w, grad_cls, start, idx, grad_x, in_dim, batch, scale, s, per_class);
    default: return backward_x_t<double>(x, a, b, w, grad_cls, start, idx, grad_x, in_dim, batch, scale, s, per_class);
    }
}

extern "C" int dl_logic_backward_chained_grouped(const void *x, const int32_t *verts, const int32_t *neuron,
                                                 const uint8_t *flip, const int32_t *dst, int64_t steps, const void *w,
                                                 const void *grad_cls, int softmax_backward, const int32_t *fix_vertex,
                                                 const int32_t *fix_start, int64_t n_fix, int64_t overflow_rows,
                                                 void *grad_w, void *grad_x, void *workspace, int64_t in_dim,
                                                 int64_t out_dim, int64_t batch, int64_t k, double scale, int dtype,
                                                 void *stream) {
    const bool any = takes_any_rows(dtype);
    const bool fp = takes_fix_positions(dtype);
    const int st = grouped_args(in_dim, out_dim, batch, k, dtype);
    if (st != DL_OK) return st;
    if (steps < out_dim || n_fix < 0 || n_fix > in_dim || overflow_rows < 0) return DL_ERR_INVALID_ARGUMENT;
    if (!x || !verts || !neuron || !flip || !dst || !w || !grad_cls || !grad_w || !grad_x) return DL_ERR_INVALID_ARGUMENT;
    if (n_fix > 0 && (!fix_vertex || !fix_start)) return DL_ERR_INVALID_ARGUMENT;
    hipStream_t s = (hipStream_t) stream;
    const bool sb = softmax_backward != 0;
    const int64_t per_class = out_dim / k;
    switch (dtype) {
    case DL_F16:
        return backward_chain_t<__half>(x, verts, neuron, flip, dst, steps, w, grad_cls, sb, fix_vertex, fix_start, n_fix,
                                        overflow_rows, grad_w, grad_x, workspace, in_dim, out_dim, batch, scale, any, fp, s, per_class);
    case DL_F32:
        return backward_chain_t<float>(x, verts, neuron, flip, dst, steps, w, grad_cls, sb, fix_vertex, fix_start, n_fix,
                                       overflow_rows, grad_w, grad_x, workspace, in_dim, out_dim, batch, scale, any, fp, s, per_class);
    default:
        return backward_chain_t<double>(x, verts, neuron, flip, dst, steps, w, grad_cls, sb, fix_vertex, fix_start, n_fix,
                                        overflow_rows, grad_w, grad_x, workspace, in_dim, out_dim, batch, scale, any, fp, s, per_class);
    }
}

extern "C" int dl_version(void) { return 100; }

extern "C" const char *dl_status_string(int status) {
    switch (status) {
    case DL_OK: return "ok";
    case DL_ERR_INVALID_ARGUMENT: return "invalid argument (null pointer, negative size or misaligned buffer)";
    case DL_ERR_BIT_COUNT: return "`bit_count` has to be in { 8, 16, 32, 64 }";
    case DL_ERR_NOT_DIVISIBLE: return "in_dim has to be divisible by k";
    case DL_ERR_DTYPE: return "dtype has to be DL_F16, DL_F32 or DL_F64";
    case DL_ERR_LAUNCH: return "HIP refused the kernel launch";
    case DL_ERR_TOO_LARGE: return "size exceeds what this entry point supports";
    case DL_ERR_SCRATCH_LIMIT: return "the call needs more than the library's static scratch array (DL_STATIC_SCRATCH_BYTES)";
    case DL_ERR_CAPTURING: return "the first call on a device must be made outside a graph capture";
    default: return "unknown status";
    }
}

// ---- Adam over all of a model's weight tensors in one launch ---------------------------------
// Elementwise and bound by its 7 float streams (p, g, m, v read; p, m, v written).  The tensors'
// pointers and sizes travel in the kernel arguments; a block takes DL_ADAM_BLOCK_ELEMS consecutive
// elements of one tensor, found through the running block counts.  The step count lives on the
// device so that a captured launch advances it on every replay; a one-thread kernel advances it and
// derives the two bias-correction factors before the update runs.
#define DL_ADAM_MAX_TENSORS 48
#define DL_ADAM_BLOCK_ELEMS 4096

namespace {

struct AdamTensors {
    float *p[DL_ADAM_MAX_TENSORS];
    const float *g[DL_ADAM_MAX_TENSORS];
    float *m[DL_ADAM_MAX_TENSORS];
    float *v[DL_ADAM_MAX_TENSORS];
    int64_t numel[DL_ADAM_MAX_TENSORS];
    uint32_t first_block[DL_ADAM_MAX_TENSORS + 1];       // running sum of ceil(numel / DL_ADAM_BLOCK_ELEMS)
    int count;
};

// state[0]: updates done; state[1], state[2]: lr / (1 - beta1^step) and 1 / sqrt(1 - beta2^step) of the update
// under way, in double arithmetic (1 - 0.999^s cancels badly in float for small s)
__global__ void adam_advance_kernel(float *state, double lr, double beta1, double beta2) {
    const double s = (double) state[0] + 1.0;
    state[0] = (float) s;
    state[1] = (float) (lr / (1.0 - pow(beta1, s)));
    state[2] = (float) (1.0 / sqrt(1.0 - pow(beta2, s)));
}

__global__ __launch_bounds__(DL_BLOCK) void adam_kernel(AdamTensors t, const float *__restrict__ state, float beta2,
                                                        float one_minus_beta1, float one_minus_beta2, float eps,
                                                        float weight_decay) {
    // which tensor: scalar search over at most 48 entries
    int ti = 0;
    while (ti + 1 < t.count && blockIdx.x >= t.first_block[ti + 1]) ++ti;
    const int64_t base = (int64_t) (blockIdx.x - t.first_block[ti]) * DL_ADAM_BLOCK_ELEMS;
    const int64_t n = t.numel[ti];
    float *__restrict__ p = t.p[ti];
    const float *__restrict__ g = t.g[ti];
    float *__restrict__ m = t.m[ti];
    float *__restrict__ v = t.v[ti];

    const float step_size = state[1], inv_bc2_sqrt = state[2];

    auto update = [&](float &pi, float gi, float &mi, float &vi) {
        if (weight_decay != 0.0f) gi = fmaf(weight_decay, pi, gi);
        mi = fmaf(gi - mi, one_minus_beta1, mi);
        vi = fmaf(beta2, vi, one_minus_beta2 * gi * gi);
        pi -= step_size * mi / (sqrtf(vi) * inv_bc2_sqrt + eps);
    };
    const bool vec = ((reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(g) | reinterpret_cast<uintptr_t>(m) |
                       reinterpret_cast<uintptr_t>(v)) & 15) == 0;
#pragma unroll
    for (int r = 0; r < DL_ADAM_BLOCK_ELEMS / (4 * DL_BLOCK); ++r) {
        const int64_t i = base + ((int64_t) r * DL_BLOCK + threadIdx.x) * 4;
        if (i >= n) break;
        if (vec && i + 4 <= n) {
            float4 pv = *reinterpret_cast<const float4 *>(p + i), gv = *reinterpret_cast<const float4 *>(g + i);
            float4 mv = *reinterpret_cast<const float4 *>(m + i), vv = *reinterpret_cast<const float4 *>(v + i);
            update(pv.x, gv.x, mv.x, vv.x);
            update(pv.y, gv.y, mv.y, vv.y);
            update(pv.z, gv.z, mv.z, vv.z);
            update(pv.w, gv.w, mv.w, vv.w);
            *reinterpret_cast<float4 *>(p + i) = pv;
            *reinterpret_cast<float4 *>(m + i) = mv;
            *reinterpret_cast<float4 *>(v + i) = vv;
        } else {
            for (int64_t j = i; j < i + 4 && j < n; ++j) update(p[j], g[j], m[j], v[j]);
        }
    }
}

}  // namespace

extern "C" int dl_adam_max_tensors(void) { return DL_ADAM_MAX_TENSORS; }

extern "C" int dl_adam_step(int count, float *const *p, const float *const *g, float *const *m, float *const *v,
                            const int64_t *numel, float *state, double lr, double beta1, double beta2, double eps,
                            double weight_decay, void *stream) {
    if (count < 0 || !(lr >= 0.0) || !(beta1 >= 0.0 && beta1 < 1.0) || !(beta2 >= 0.0 && beta2 < 1.0) || !(eps >= 0.0) ||
        !(weight_decay >= 0.0))
        return DL_ERR_INVALID_ARGUMENT;
    if (count > DL_ADAM_MAX_TENSORS) return DL_ERR_TOO_LARGE;
    if (count == 0) return DL_OK;
    if (!p || !g || !m || !v || !numel || !state) return DL_ERR_INVALID_ARGUMENT;
    AdamTensors t;
    uint64_t blocks = 0;
    t.count = 0;
    for (int i = 0; i < count; ++i) {
        if (numel[i] < 0) return DL_ERR_INVALID_ARGUMENT;
        if (numel[i] == 0) continue;
        if (!p[i] || !g[i] || !m[i] || !v[i]) return DL_ERR_INVALID_ARGUMENT;
        const int k = t.count++;
        t.p[k] = p[i], t.g[k] = g[i], t.m[k] = m[i], t.v[k] = v[i], t.numel[k] = numel[i];
        t.first_block[k] = (uint32_t) blocks;
        blocks += (uint64_t) dl_ceil_div(numel[i], DL_ADAM_BLOCK_ELEMS);
        if (blocks > 0x7fffffffULL) return DL_ERR_TOO_LARGE;
    }
    hipStream_t s = (hipStream_t) stream;
    DL_LAUNCH(adam_advance_kernel, dim3(1), dim3(1), 0, s, state, lr, beta1, beta2);
    if (t.count > 0) {
        t.first_block[t.count] = (uint32_t) blocks;
        DL_LAUNCH(adam_kernel, dim3((unsigned) blocks), dim3(DL_BLOCK), 0, s, t, (const float *) state, (float) beta2,
                  (float) (1.0 - beta1), (float) (1.0 - beta2), (float) eps, (float) weight_decay);
    }
    return dl_launch_status();
}

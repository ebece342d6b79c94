// dense_mv.hip - y = W x on dense F32 / F16 / BF16 rows (ops.rs:87-98,
// 131-154, 600-623) for one or several columns.
//
// Weights widen exactly to fp32 and x stays fp32, so the products and sums
// are those of fp32 arithmetic for every kind.  Chains: one column, one per
// element of a piece over a wavefront's steps (56 products at most, F32 rows
// of 14336 elements on one wavefront), then trees; several, eight a step of
// up to 8 products, a tree over them, then one over the wavefront's steps.
// Rows may start at any element.  One column, two to four, and more are three
// summation orders; within each a column does not depend on the others.
//
// One column: dense_vec_kernel, 16-byte loads on the vector ALU.  Several:
// dense_mv_kernel on the fp32 matrix cores, one pass over the payload for up
// to 16 columns.  A workgroup takes 16 rows and up to 4 (v_mfma_f32_4x4x1,
// sixteen 4x4 blocks) or 16 columns (v_mfma_f32_16x16x4); its wavefronts take
// steps of the rows in turn and meet in LDS.  Lane l = 16 g + r holds the
// weights of row r for its quarter g of each step: 16-byte loads whose four
// lanes per row cover 64 consecutive bytes.  Both shapes take k-slot g from
// lane group g, so which element sits in which slot is free as long as x is
// read in the same order; for 4x4x1 the block of lane l is l / 4 = 4 g + r / 4,
// whose four rows are r and its neighbours and whose four x columns the same
// lanes hold.  x of a step is read once, contiguously, and turned into that
// order through the wavefront's own LDS (read from global memory in operand
// order its quarter-wavefronts touch four lines each: 8192x2560 bf16, 4
// columns, 16.0 against 10.6 us).
//
// What bounds it: the payload's bytes.  Per 16 rows x 128 elements a SIMD
// spends some 256 (4x4x1) or 1024 (16x16x4) cycles of matrix core, against
// 2000 cycles of a CU's share of HBM for a 16-bit payload; hence 4x4x1 up to
// 4 columns and the wide shape beyond.  Measured against the 2-byte loads and
// vector products that stood here: bf16 8192x2560, 1 / 4 / 6 columns 16.0 /
// 49.5 / 81 -> 8.4 / 9.8 / 11.4 us (42 MB: 5.0 / 4.3 / 3.7 TB/s), 4096x4096
// with 16 columns 131 -> 11.2, 32768x2047 with 16 (odd rows) 527 -> 43 us;
// fp32 4096x14336, one column, 77.5 -> 32.4 us.  Slower only on rows that do not
// fill a step: 100x100, 2 to 4 columns, 3.1 -> 4.1 us.
#include "common.hpp"

#include <algorithm>

namespace ouro {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
typedef uint32_t du32x4 __attribute__((ext_vector_type(4)));
typedef du32x4 du32x4_a4 __attribute__((aligned(4)));

template <bool WIDE> constexpr int kCols = WIDE ? 16 : 4;     // columns a workgroup
// elements of a row that a wavefront takes at a time
template <int KIND, bool WIDE> constexpr int kStep = WIDE || KIND == OURO_KIND_F32 ? 64 : 128;
// x of a step in LDS: a column's floats and 16 bytes, so that the 16-byte
// reads of neighbouring columns fall in distinct banks
template <int KIND, bool WIDE> constexpr int kXPitch = kStep<KIND, WIDE> + 4;
// 64 KiB of LDS hold x of 15 wavefronts at 16 columns
template <bool WIDE> constexpr int kMaxWaves = WIDE ? 15 : 16;
constexpr int kDenseRows = 16;
constexpr int kVecWaves = 8;  // one column: wavefronts a workgroup at most

struct DenseArgs {
    const uint8_t *w;
    const float *x;  // [k][in_len]
    float *y;        // [k][out_len]
    int out_len, in_len, k;
};

template <int KIND> constexpr int kElemBytes = KIND == OURO_KIND_F32 ? 4 : 2;

// 16 bytes of weights as fp32
template <int KIND>
__device__ __forceinline__ void widen(const du32x4 &p, float *w) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint32_t v = p[d];
        if constexpr (KIND == OURO_KIND_F32) {
            w[d] = __builtin_bit_cast(float, v);
        } else if constexpr (KIND == OURO_KIND_BF16) {
            w[2 * d] = __builtin_bit_cast(float, v << 16);
            w[2 * d + 1] = __builtin_bit_cast(float, v & 0xffff0000u);
        } else {
            w[2 * d] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(v)));
            w[2 * d + 1] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(v >> 16)));
        }
    }
}

// The 16-byte piece at p.  AL: any dword boundary; else rows may start at an
// odd 16-bit element, and the two dword-aligned loads that cover the piece are
// shifted into place (a 16-byte load off its dword boundary is slower: 1500x7001
// bf16 on the matrix cores 23.9 -> 15.2 us).  Every dword read holds at least one byte
// of the piece.
template <bool AL>
__device__ __forceinline__ du32x4 load_piece(const uint8_t *p) {
    if constexpr (AL) {
        return *reinterpret_cast<const du32x4_a4 *>(p);
    } else {
        const uint32_t s = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 3);
        const uint8_t *base = p - s;
        const du32x4 lo = *reinterpret_cast<const du32x4_a4 *>(base);
        const uint32_t e = *reinterpret_cast<const uint32_t *>(base + ((s + 15) & ~3u));
        du32x4 r;
        r.x = __builtin_amdgcn_alignbyte(lo.y, lo.x, s);
        r.y = __builtin_amdgcn_alignbyte(lo.z, lo.y, s);
        r.z = __builtin_amdgcn_alignbyte(lo.w, lo.z, s);
        r.w = __builtin_amdgcn_alignbyte(e, lo.w, s);
        return r;
    }
}

// Elements e .. of a row's last step, zeros from element n on.  A piece that
// passes the row's end is read as the row's last piece and shifted, one past
// it reads the first: no branches, so a step's loads go out together.
template <int KIND, bool AL>
__device__ __forceinline__ du32x4 last_piece(const uint8_t *row, long long e, int n) {
    constexpr int EB = kElemBytes<KIND>, PE = 16 / EB;
    if (n < PE) {  // uniform; a row shorter than a piece
        du32x4 r = {0u, 0u, 0u, 0u};
        for (int i = 0; i < n; ++i) {
            uint32_t v;
            if constexpr (EB == 4) v = reinterpret_cast<const uint32_t *>(row)[i];
            else v = static_cast<uint32_t>(reinterpret_cast<const uint16_t *>(row)[i]) << (16 * (i & 1));
            const int d = i * EB / 4;
            r.x |= d == 0 ? v : 0u;
            r.y |= d == 1 ? v : 0u;
            r.z |= d == 2 ? v : 0u;
            r.w |= d == 3 ? v : 0u;
        }
        return e == 0 ? r : du32x4{0u, 0u, 0u, 0u};
    }
    const int over = e + PE <= n ? 0 : e < n ? static_cast<int>(e + PE - n) : PE;  // elements past the end
    du32x4 v = load_piece<AL>(row + (over == PE ? 0 : e - over) * EB);
    const int bytes = over * EB;
    if (bytes & 8) v = du32x4{v.z, v.w, 0u, 0u};
    if (bytes & 4) v = du32x4{v.y, v.z, v.w, 0u};
    if constexpr (EB == 2) {
        const uint32_t s = bytes & 2;
        v = du32x4{__builtin_amdgcn_alignbyte(v.y, v.x, s), __builtin_amdgcn_alignbyte(v.z, v.y, s),
                   __builtin_amdgcn_alignbyte(v.w, v.z, s), __builtin_amdgcn_alignbyte(0u, v.w, s)};
    }
    return over == PE ? du32x4{0u, 0u, 0u, 0u} : v;
}

__device__ __forceinline__ f32x4 last_x(const float *x, long long e, int n) {
    return __builtin_bit_cast(f32x4, last_piece<OURO_KIND_F32, true>(reinterpret_cast<const uint8_t *>(x), e, n));
}

// A row's sum over the wavefronts, four short chains.
__device__ __forceinline__ float sum_waves(const float *p, int nw, int stride) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < nw; w += 4)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += w + i < nw ? p[(w + i) * stride] : 0.f;
    return (v[0] + v[1]) + (v[2] + v[3]);
}

// One column.  A workgroup takes R rows; its wavefronts take steps of 64
// pieces (512 16-bit or 256 32-bit elements) in turn, each lane one 16-byte
// piece of every row and its elements of x, one fp32 chain per element of the
// piece: 1 KiB contiguous per load.  Against the matrix-core kernel run with
// one column, a short matrix fills the chip sooner than with 16-row tiles
// (2048x2048 fp32 6.4 -> 4.0 us, 100x14336 bf16 16.1 -> 4.0 us).
template <int KIND, int R, bool AL>
__global__ __launch_bounds__(64 * kVecWaves) void dense_vec_kernel(DenseArgs a) {
    constexpr int EB = kElemBytes<KIND>, PE = 16 / EB, ST = 64 * PE;
    __shared__ float red[kVecWaves][R];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int row0 = blockIdx.x * R;
    const uint8_t *wr[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wr[r] = a.w + static_cast<long long>(min(row0 + r, a.out_len - 1)) * a.in_len * EB;
    const int full = a.in_len / ST, steps = (a.in_len - 1) / ST + 1;
    float acc[R][PE];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < PE; ++i) acc[r][i] = 0.f;
    for (int s = wave; s < steps; s += nw) {
        const long long e = static_cast<long long>(ST) * s + PE * lane;
        du32x4 raw[R];
        float xv[PE];
        if (s < full) {
#pragma unroll
            for (int r = 0; r < R; ++r) raw[r] = load_piece<AL>(wr[r] + e * EB);
#pragma unroll
            for (int q = 0; q < PE; q += 4) *reinterpret_cast<f32x4 *>(xv + q) = *reinterpret_cast<const f32x4_a4 *>(a.x + e + q);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) raw[r] = last_piece<KIND, AL>(wr[r], e, a.in_len);
#pragma unroll
            for (int q = 0; q < PE; q += 4) *reinterpret_cast<f32x4 *>(xv + q) = last_x(a.x, e + q, a.in_len);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float wv[PE];
            widen<KIND>(raw[r], wv);
#pragma unroll
            for (int i = 0; i < PE; ++i) acc[r][i] = __builtin_fmaf(wv[i], xv[i], acc[r][i]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        float v = (acc[r][0] + acc[r][1]) + (acc[r][2] + acc[r][3]);
        if constexpr (PE == 8) v += (acc[r][4] + acc[r][5]) + (acc[r][6] + acc[r][7]);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v += xor_shfl(v, off);
        if (nw == 1) {
            if (lane == 0 && row0 + r < a.out_len) a.y[row0 + r] = v;
        } else if (lane == 0) {
            red[wave][r] = v;
        }
    }
    if (nw == 1) return;
    __syncthreads();
    if (threadIdx.x < R && row0 + static_cast<int>(threadIdx.x) < a.out_len) {
        a.y[row0 + threadIdx.x] = sum_waves(&red[0][threadIdx.x], nw, R);
    }
}

// WIDE: 16 columns a workgroup, else 4.  LDS: each wavefront's step of x
// (min(columns, NC) rows of kXPitch floats), then the row sums.
template <int KIND, bool WIDE, bool AL>
__global__ __launch_bounds__(64 * kMaxWaves<WIDE>) void dense_mv_kernel(DenseArgs a) {
    constexpr int EB = kElemBytes<KIND>, PE = 16 / EB;  // elements a piece
    constexpr int NC = kCols<WIDE>, ST = kStep<KIND, WIDE>, XP = kXPitch<KIND, WIDE>;
    constexpr int NP = ST / 4 / PE;           // pieces a step
    constexpr int LC = ST / 4, CL = 64 / LC;  // lanes that load a column of x, columns a load
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * kDenseRows, c0 = blockIdx.y * NC;
    const int nc = min(NC, a.k - c0);
    const uint8_t *wr = a.w + static_cast<long long>(min(row0 + r, a.out_len - 1)) * a.in_len * EB;
    const float *xr = a.x + static_cast<long long>(c0) * a.in_len;
    float *xl = lds + wave * (min(NC, a.k) * XP);
    const float *xp = xl + min(lane & (NC - 1), nc - 1) * XP + PE * g;  // clamped columns are dropped
    const int xe = 4 * (lane % LC), xc = lane / LC;  // the lane's part of x: floats xe .. xe + 3 of columns xc + CL j
    const int full = a.in_len / ST, steps = (a.in_len - 1) / ST + 1;
    du32x4 raw[NP];
    f32x4 xs[NC / CL];
    auto load = [&](int s) {
        const long long s0 = static_cast<long long>(ST) * s, e0 = s0 + PE * g;  // piece p: elements e0 + 4 PE p ..
        if (s < full) {
#pragma unroll
            for (int p = 0; p < NP; ++p) raw[p] = load_piece<AL>(wr + (e0 + 4 * PE * p) * EB);
#pragma unroll
            for (int j = 0; j < NC / CL; ++j)
                if (CL * j < nc)
                    xs[j] = *reinterpret_cast<const f32x4_a4 *>(xr + static_cast<long long>(min(CL * j + xc, nc - 1)) * a.in_len + s0 + xe);
        } else {  // the row's last elements: zeros past its end on both sides
#pragma unroll
            for (int p = 0; p < NP; ++p) raw[p] = last_piece<KIND, AL>(wr, e0 + 4 * PE * p, a.in_len);
#pragma unroll
            for (int j = 0; j < NC / CL; ++j)
                if (CL * j < nc) xs[j] = last_x(xr + static_cast<long long>(min(CL * j + xc, nc - 1)) * a.in_len, s0 + xe, a.in_len);
        }
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (wave < steps) load(wave);
    for (int s = wave; s < steps; s += nw) {
        du32x4 cur[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) cur[p] = raw[p];
#pragma unroll
        for (int j = 0; j < NC / CL; ++j)
            if (CL * j < nc) *reinterpret_cast<f32x4 *>(xl + min(CL * j + xc, nc - 1) * XP + xe) = xs[j];
        __builtin_amdgcn_wave_barrier();  // xl is the wavefront's own: its LDS operations are in order
        if (s + nw < steps) load(s + nw);
        __builtin_amdgcn_sched_barrier(0);  // the next step's loads go out before this one's products
        f32x4 t[8] = {};
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            float wv[PE], xv[PE];
            widen<KIND>(cur[p], wv);
#pragma unroll
            for (int q = 0; q < PE; q += 4) *reinterpret_cast<f32x4 *>(xv + q) = *reinterpret_cast<const f32x4 *>(xp + 4 * PE * p + q);
#pragma unroll
            for (int i = 0; i < PE; ++i) {
                f32x4 &d = t[(PE * p + i) & 7];
                if constexpr (WIDE) d = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[i], wv[i], d, 0, 0, 0);
                else d = __builtin_amdgcn_mfma_f32_4x4x1f32(xv[i], wv[i], d, 0, 0, 0);
            }
        }
        __builtin_amdgcn_wave_barrier();
        acc += ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
    }
    // WIDE: lane 16 g + r holds columns 4 g .. 4 g + 3 of row r; else all four
    // columns of row r, one share per g
    if constexpr (!WIDE) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            acc[v] += xor_shfl(acc[v], 32);
            acc[v] += xor_shfl(acc[v], 16);
        }
    }
    __syncthreads();  // the sums take the place of x
    if (WIDE || g == 0) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = (WIDE ? 4 * g : 0) + v;
            if (c < nc) lds[(wave * nc + c) * kDenseRows + r] = acc[v];
        }
    }
    __syncthreads();
    for (int o = threadIdx.x; o < nc * kDenseRows; o += blockDim.x) {
        const int c = o / kDenseRows, row = row0 + o % kDenseRows;
        const float v = sum_waves(lds + o, nw, nc * kDenseRows);
        if (row < a.out_len) a.y[static_cast<long long>(c0 + c) * a.out_len + row] = v;
    }
}

template <int KIND, bool WIDE>
int launch_cols(const DenseArgs &a, bool al, hipStream_t s) {
    constexpr int NC = kCols<WIDE>;
    const dim3 grid((a.out_len - 1) / kDenseRows + 1, (a.k - 1) / NC + 1);
    const int steps = (a.in_len - 1) / kStep<KIND, WIDE> + 1;
    // about 16 wavefronts a CU over the rows, the steps spread evenly over a
    // workgroup's wavefronts; not by the column groups, so that a column's sum
    // is the same in any number of them
    int nw = static_cast<int>(std::min<unsigned>(std::min(kMaxWaves<WIDE>, steps), (4095 + grid.x) / grid.x));
    const int per = (steps + nw - 1) / nw;
    nw = (steps + per - 1) / per;
    const size_t lds = static_cast<size_t>(nw) * std::min(NC, a.k) * kXPitch<KIND, WIDE> * sizeof(float);
    const auto fn = al ? dense_mv_kernel<KIND, WIDE, true> : dense_mv_kernel<KIND, WIDE, KIND == OURO_KIND_F32>;
    hipLaunchKernelGGL(fn, grid, dim3(64 * nw), lds, s, a);
    return check_launch("dense_mv_kernel");
}

template <int KIND, int R>
int launch_vec(const DenseArgs &a, bool al, hipStream_t s) {
    const unsigned wgs = static_cast<unsigned>((a.out_len - 1) / R + 1);
    const int steps = (a.in_len - 1) / (1024 / kElemBytes<KIND>) + 1;
    int nw = static_cast<int>(std::min<unsigned>(std::min(kVecWaves, steps), (4096 + wgs - 1) / wgs));
    const int per = (steps + nw - 1) / nw;
    nw = (steps + per - 1) / per;
    const auto fn = al ? dense_vec_kernel<KIND, R, true> : dense_vec_kernel<KIND, R, KIND == OURO_KIND_F32>;
    hipLaunchKernelGGL(fn, dim3(wgs), dim3(64 * nw), 0, s, a);
    return check_launch("dense_vec_kernel");
}

template <int KIND>
int launch_kind(const DenseArgs &a, hipStream_t s) {
    // every row on a dword (fp32 always)
    const bool al = KIND == OURO_KIND_F32 || (a.in_len % 2 == 0 && reinterpret_cast<uintptr_t>(a.w) % 4 == 0);
    if (a.k == 1) return a.out_len >= 4096 ? launch_vec<KIND, 4>(a, al, s) : launch_vec<KIND, 1>(a, al, s);
    return a.k > kCols<false> ? launch_cols<KIND, true>(a, al, s) : launch_cols<KIND, false>(a, al, s);
}

}  // namespace

// y[c][row] for k columns of x on dense rows of any element-aligned payload;
// the caller has checked pointers, kind, sizes (each below 2^31) and alignment.
int dense_matmul(const void *payload, int kind, size_t out_len, size_t in_len, const float *x, size_t k, float *y,
                 void *stream) {
    const DenseArgs a{static_cast<const uint8_t *>(payload), x, y, static_cast<int>(out_len),
                      static_cast<int>(in_len), static_cast<int>(k)};
    const hipStream_t s = as_stream(stream);
    switch (kind) {
    case OURO_KIND_F32: return launch_kind<OURO_KIND_F32>(a, s);
    case OURO_KIND_F16: return launch_kind<OURO_KIND_F16>(a, s);
    default: return launch_kind<OURO_KIND_BF16>(a, s);
    }
}

}  // namespace ouro

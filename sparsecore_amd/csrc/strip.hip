// dW over strips (gfx950): the SIMD-order weight gradient for layers dense
// enough that a row holds several slots per block of X rows.
//
// dW[s] = dot(dY[i, :], X[col[s], :]) in the reference's SIMD order: 16 fma
// chains over n = 16 t + l, then its add tree
// (csrc/kernels/spmm_grad_avx2.cpp:112-258); the same bits as slk_sddmm.
//
// A strip is a quad of rows x one block of X rows x up to S of each row's slots
// there. A wave holds the quad's rows side by side, 16 lanes each, lane l of a
// row running chain l of every slot: one register per slot of the quad. X goes
// through LDS in windows of C rows x 64 columns, from a copy whose windows are
// laid out chain by chain (strip_layout_kernel: columns 16 t + l of chain l
// beside each other, padded to whole windows; 10 us for 25 MB). One 16-byte
// read per lane is then four steps of a chain, the 16 lanes of a row read 256
// contiguous bytes, conflict-free in any slot order, and staging is contiguous
// 16-byte direct loads at any N (4-byte loads that did the layout on the way
// cost 14 cycles of the load path each, more than the fmas). A slot's LDS
// offset comes by DPP from the lane that holds it. dY's window of a row is read
// once for all its slots of the strip, and each staged window serves the
// workgroup's 64·R rows: 15-25 bytes from the L2 per slot and window, against
// 50-64 for the segment kernel of sddmm.hip, whose quads of lanes take 8 slots
// per dY read. What bounds it is the LDS, a 16-byte read per four fmas, beside
// the vector unit: 73 TFLOP/s of slots and padding at the 560 reads per us of a CU,
// of which it reaches about two thirds (2304 x 768 at 30%, N = 8192: vector unit
// busy 57%, 24% of the waves' cycles waiting to issue to the LDS). Measured, layout
// included: that layer 365 -> 283 us, 1152 x 384 at 30% 171 -> 125, 4096^2 at 5%,
// N = 4096, 579 -> 405, 1537 x 1000 at 20%, N = 1777, 194 -> 52.
#include "common.hpp"
#include "dw_common.hpp"

#include <cmath>

namespace slk {
namespace {

constexpr uint32_t kBufWord3 = 0x00020000;  // gfx9 buffer resource dword 3
constexpr int kWin = 64;                    // columns of N per (part of a) window
constexpr int64_t kMaxBlocks = 2048;
constexpr int64_t kMaxRows = int64_t{4} * 256 * 65535;  // the fill's grid is 256 quads per row of blocks

constexpr int kWaves = 16;
constexpr int kMaxC = 256;                  // X rows per block
constexpr int kMaxParts = 288;              // rows x parts of a staged window: 72 KiB

__device__ __forceinline__ void lds_load16(const void* base, uint32_t bytes, uint32_t vo,
                                           uint32_t so, void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0),
                                          static_cast<int>(bytes), kBufWord3),
        (__attribute__((address_space(3))) void*)lds, 16, vo, so, 0, 0);
}

// lane I of each row of 16 lanes, in all 16
template <int I>
__device__ __forceinline__ int row_bcast(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + I, 0xf, 0xf, true);
}
// each row of 16 lanes rotated by I lanes
template <int I>
__device__ __forceinline__ float row_rotate(float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + I, 0xf, 0xf, true));
}

// LDS by its 32-bit address: an offset from a DPP move then takes one add (from
// a pointer to dynamic LDS the compiler adds the array's base apart)
__device__ __forceinline__ int lds_address(const void* p) {
    return static_cast<int>(
        reinterpret_cast<uint64_t>((const __attribute__((address_space(3))) char*)p));
}
__device__ __forceinline__ f32x4 lds_read16(int a) {
    return *(const __attribute__((address_space(3))) f32x4*)static_cast<uint32_t>(a);
}

// v computed here: without it the compiler moves a group's fmas, whose sums
// nothing else in the sweep reads, behind the branches that follow, and keeps
// their operands until then
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }

// XP[k][64 v + 4 l + t] = X[k][64 v + 16 t + l], 0 past N: a wave takes four
// windows of a row. The waves after `items` take a row of W each: its padding
// slots' zeros and, with dbias, its dY row's sum (beside the strips, each would
// hold a CU's whole LDS: 2304 rows at N = 8192 38 us more).
__global__ __launch_bounds__(256) void strip_layout_kernel(
    int64_t N, int64_t NP, int64_t quads, int64_t items, const float* __restrict__ X,
    float* __restrict__ XP, int64_t M, const int32_t* __restrict__ row_start,
    const int32_t* __restrict__ row_nnz, const int32_t* __restrict__ row_cap,
    const float* __restrict__ dY, float* __restrict__ dW, float* __restrict__ dbias) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t i = blockIdx.x * int64_t{4} + (threadIdx.x >> 6);
    if (i >= items) {
        zero_row_padding(row_start, row_nnz, row_cap, M, i - items, dW);
        if (dbias != nullptr) bias_row_sum(dY, M, N, i - items, dbias, N, 1);
        return;
    }
    const int64_t k = i / quads, n0 = (i - k * quads) * (4 * kWin) + (lane >> 4) * kWin;
    if (n0 >= NP) return;
    f32x4 v;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int64_t n = n0 + 16 * t + (lane & 15);
        v[t] = n < N ? X[k * N + n] : 0.0f;
    }
    *reinterpret_cast<f32x4*>(XP + k * NP + n0 + 4 * (lane & 15)) = v;
}

// 16 waves, R strips each, all in one block of C X rows (C a multiple of 16). A
// window has V parts of 64 columns: two halve the barriers, branches and offset
// adds per fma. AL: dY allows 16-byte loads.
template <int S, int R, int V, bool AL>
__global__ __launch_bounds__(kWaves * kWave, 4) void strip_dw_kernel(
    int64_t M, int64_t K, int64_t N, int64_t NP, int64_t first, const int32_t* __restrict__ order,
    const int32_t* __restrict__ row_start, const int32_t* __restrict__ col,
    const float* __restrict__ dY, const float* __restrict__ X, const float* __restrict__ XP,
    float* __restrict__ dW, const int2* __restrict__ items, const int32_t* __restrict__ rel,
    const int32_t* __restrict__ used, int32_t nb, int32_t C) {
    constexpr int NW = kWaves, kRowBytes = V * kWin * 4, kSteps = 4 * V;
    extern __shared__ __align__(1024) char smem[];  // two windows, then 1 KiB per wave for dY
    const int lane = threadIdx.x & (kWave - 1), l16 = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t grp = blockIdx.x;
    // groups in use in XCD-contiguous order: an XCD's mostly share a block
    const int64_t G = *used;
    if (grp >= G) return;  // block-uniform
    const int2* mine = items + xcd_logical_block(grp, G) * (NW * R) + w * R;
    const int64_t c0 = static_cast<int64_t>(mine[0].y >> 8) * C;

    int64_t row[R];
    int32_t s0[R], m[R], nmax[R], off[R][S / 16];
    const float* dyp[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int2 it = mine[k];
        const int64_t p = first + int64_t{4} * it.x + (lane >> 4);
        const bool ok = it.x >= 0 && p < M;
        row[k] = ok ? (order != nullptr ? order[p] : p) : 0;
        int32_t n = 0;
        s0[k] = 0;
        if (ok) {
            const int32_t* rr = rel + (int64_t{4} * it.x + (lane >> 4)) * (nb + 1) + (it.y >> 8);
            const int32_t lo = rr[0] + (it.y & 255) * S;
            n = rr[1] - lo;
            s0[k] = row_start[row[k]] + lo;
        }
        m[k] = n < 0 ? 0 : n > S ? S : n;
        nmax[k] = max(max(__builtin_amdgcn_readlane(m[k], 0), __builtin_amdgcn_readlane(m[k], 16)),
                      max(__builtin_amdgcn_readlane(m[k], 32), __builtin_amdgcn_readlane(m[k], 48)));
#pragma unroll
        for (int i = 0; i < S / 16; ++i) {
            const int s = 16 * i + l16;
            off[k][i] = s < m[k] ? static_cast<int32_t>(col[s0[k] + s] - c0) * kRowBytes : 0;
        }
        dyp[k] = dY + row[k] * N;
    }

    const int32_t last = static_cast<int32_t>(K - c0 < C ? K - c0 : C) - 1;
    const float* xb = XP + c0 * NP;
    const uint32_t rowb = static_cast<uint32_t>(4 * NP);
    const uint32_t xbytes = static_cast<uint32_t>(last + 1) * rowb;
    const int64_t n16 = N / 16;
    const int32_t nwin = static_cast<int32_t>(ceil_div(n16, int64_t{kSteps}));
    // a load stages 1 KiB, whole rows' windows; rows past K repeat the last
    constexpr int kPieceRows = 1024 / kRowBytes, kLanes = kWave / kPieceRows;
    constexpr int kPieces = (kMaxParts / V / kPieceRows + NW - 1) / NW;
    uint32_t xo[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
        const int32_t r = kPieceRows * (w + i * NW) + lane / kLanes;
        xo[i] = static_cast<uint32_t>(r < last ? r : last) * rowb + 16 * (lane % kLanes);
    }
    auto stage = [&](int buf, int32_t win) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int piece = w + i * NW;
            if (kPieceRows * piece < C)
                lds_load16(xb, xbytes, xo[i], static_cast<uint32_t>(win) * kRowBytes,
                           smem + buf * (C * kRowBytes) + piece * 1024);
        }
    };
    // dY's part v of window win, strip k: with AL 16 bytes a lane as they lie,
    // else the lane's four steps
    auto load_dy = [&](int32_t win, int v, int k) {
        const int64_t n0 = (static_cast<int64_t>(win) * V + v) * kWin;
        f32x4 d;
        if constexpr (AL) {
            const int64_t n = n0 + 4 * l16;
            d = *reinterpret_cast<const f32x4*>(dyp[k] + (n < N ? n : N - 4));
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int64_t n = n0 + 16 * t + l16;
                d[t] = dyp[k][n < N ? n : N - 1];
            }
        }
        return d;
    };
    // AL: lane l's steps 16 t + l through the wave's own LDS, row g's 16-byte
    // pieces rotated by 4 g so that the four rows' reads lie in distinct banks
    char* turn = smem + 2 * C * kRowBytes + w * 1024;
    const int g4 = lane >> 4;
    const int turn_w = g4 * 256 + ((l16 + 4 * g4) & 15) * 16;
    const int turn_r = g4 * 256 + (l16 & 3) * 4;
    auto steps_of = [&](f32x4 d) {
        if constexpr (AL) {
            *reinterpret_cast<f32x4*>(turn + turn_w) = d;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                d[t] = *reinterpret_cast<const float*>(
                    turn + turn_r + ((4 * t + (l16 >> 2) + 4 * g4) & 15) * 16);
        }
        return d;
    };

    float acc[R][S];
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
        for (int s = 0; s < S; ++s) acc[k][s] = 0.0f;
    f32x4 dn[R][V];  // each strip's dY of the window
    // window in buffer buf; with Tail only its first tn steps, else dY of
    // window next is loaded behind it
    auto sweep = [&](auto Tail, int buf, int tn, int32_t next) {
        const int lx = lds_address(smem) + buf * (C * kRowBytes) + l16 * 16;
        static_for<R>([&](auto J) {
            constexpr int k = decltype(J)::value;
            constexpr int kReads = 2;  // slots per group
            const int32_t n = nmax[k];
            f32x4 dy[V];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                dy[v] = steps_of(dn[k][v]);
                if constexpr (!decltype(Tail)::value) dn[k][v] = load_dy(next, v, k);
            }
            // slots in groups of kReads: a group's reads are issued before the
            // fmas of the one before it (past the last slot they read row 0)
            f32x4 x[2][kReads][V];
            auto reads = [&](auto Gc) {
                constexpr int g = decltype(Gc)::value;
                static_for<kReads>([&](auto I) {
                    constexpr int i = decltype(I)::value, s = kReads * g + i;
                    const int a = row_bcast<s % 16>(off[k][s / 16]) + lx;
#pragma unroll
                    for (int v = 0; v < V; ++v)
                        x[g & 1][i][v] = lds_read16(a + v * (kWin * 4));
                });
            };
            auto group = [&](auto self, auto Gc) {
                constexpr int g = decltype(Gc)::value;
                if (n > kReads * g) {
                    if constexpr (kReads * (g + 1) < S) reads(std::integral_constant<int, g + 1>{});
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int t = 0; t < kSteps; ++t)
#pragma unroll
                        for (int i = 0; i < kReads; ++i) {
                            float& a = acc[k][kReads * g + i];
                            const float f =
                                __builtin_fmaf(dy[t / 4][t % 4], x[g & 1][i][t / 4][t % 4], a);
                            if constexpr (decltype(Tail)::value) a = t < tn ? f : a;
                            else a = f;
                        }
#pragma unroll
                    for (int i = 0; i < kReads; ++i) pin(acc[k][kReads * g + i]);
                    if constexpr (kReads * (g + 1) < S)
                        self(self, std::integral_constant<int, g + 1>{});
                }
            };
            reads(std::integral_constant<int, 0>{});
            group(group, std::integral_constant<int, 0>{});
        });
    };
    if (nwin > 0) {
        stage(0, 0);
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int v = 0; v < V; ++v) dn[k][v] = load_dy(0, v, k);
    }
    const int32_t full = static_cast<int32_t>(n16 / kSteps);
    for (int32_t win = 0; win < full; ++win) {
        // this wave's loads are down, then every wave's
        __builtin_amdgcn_s_waitcnt(0);
        asm volatile("s_barrier" ::: "memory");
        const int32_t next = win + 1 < nwin ? win + 1 : win;
        stage((win & 1) ^ 1, next);  // every wave has read that buffer
        sweep(std::false_type{}, win & 1, kSteps, next);
    }
    __builtin_amdgcn_s_waitcnt(0);  // no direct load still writing LDS when the waves end
    if (nwin > full) {
        asm volatile("s_barrier" ::: "memory");
        sweep(std::true_type{}, full & 1, static_cast<int>(n16 - kSteps * static_cast<int64_t>(full)), 0);
    }

    // the add tree, in every lane of the row, with the 8-wide part of the tail
    // between its levels (lanes 8 .. 15 repeat lanes 0 .. 7)
    const int64_t j8 = 16 * n16;
    const bool has8 = N - j8 >= 8;
    const int64_t jt = has8 ? j8 + 8 : j8;
    static_for<R>([&](auto J) {
        constexpr int k = decltype(J)::value;
        const float d8 = has8 ? dyp[k][j8 + (l16 & 7)] : 0.0f;
        float res[S / 16];
        static_for<S>([&](auto Sc) {
            constexpr int s = decltype(Sc)::value;
            float a = acc[k][s];
            a = a + row_rotate<8>(a);
            if (has8) {
                const int64_t c = c0 + row_bcast<s % 16>(off[k][s / 16]) / kRowBytes;
                a = __builtin_fmaf(d8, X[c * N + j8 + (l16 & 7)], a);
            }
            a = a + row_rotate<4>(a);
            a = a + row_rotate<2>(a);
            a = a + row_rotate<1>(a);
            if constexpr (s % 16 == 0) res[s / 16] = a;
            else res[s / 16] = l16 == s % 16 ? a : res[s / 16];
        });
#pragma unroll
        for (int i = 0; i < S / 16; ++i)
            if (16 * i + l16 < m[k]) {
                const float* x = X + (c0 + off[k][i] / kRowBytes) * N;
                dW[s0[k] + 16 * i + l16] = running_sum(dyp[k] + jt, x + jt, N - jt, res[i]);
            }
    });
}

// ───────────────────────────── the build ────────────────────────────────────

// Per quad q: each row's first slot in every block (rel[q][r][0 .. nb],
// relative to row_start) and the strips per block (base[b][q]).
__global__ __launch_bounds__(256) void strip_count_kernel(
    int64_t M, int64_t first, int64_t nq, int32_t nb, int32_t C, int32_t S, const int32_t* __restrict__ order,
    const int32_t* __restrict__ row_start, const int32_t* __restrict__ row_nnz,
    const int32_t* __restrict__ col, int32_t* __restrict__ rel, int32_t* __restrict__ base) {
    extern __shared__ int32_t st[];  // [4][nb + 1]
    const int64_t q = blockIdx.x;
    const int r = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
    const int64_t p = first + 4 * q + r;
    const int64_t row = p < M ? (order != nullptr ? order[p] : p) : 0;
    int32_t* mine = st + r * (nb + 1);
    const int32_t s0 = p < M ? row_start[row] : 0, n = p < M ? row_nnz[row] : 0;
    int32_t before = -1;  // the block of the slot before this batch
    for (int32_t at = 0; at <= n; at += kWave) {
        const int32_t s = at + lane;
        const int32_t b = s < n ? col[s0 + s] / C : nb;
        int32_t pb = __shfl_up(b, 1);
        if (lane == 0) pb = before;
        if (s <= n)
            for (int32_t x = pb + 1; x <= b; ++x) mine[x] = s;
        before = __shfl(b, kWave - 1);
    }
    __syncthreads();
    for (int32_t i = threadIdx.x; i < 4 * (nb + 1); i += 256) rel[q * 4 * (nb + 1) + i] = st[i];
    for (int32_t b = threadIdx.x; b < nb; b += 256) {
        int32_t most = 0;
        for (int k = 0; k < 4; ++k)
            most = max(most, st[k * (nb + 1) + b + 1] - st[k * (nb + 1) + b]);
        base[b * nq + q] = (most + S - 1) / S;
    }
}

// base[b][.] to its exclusive scan, total[b] the sum: one workgroup per block.
__global__ __launch_bounds__(1024) void strip_scan_kernel(int64_t nq, int32_t* __restrict__ base,
                                                          int32_t* __restrict__ total) {
    __shared__ int32_t part[1024 / kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x >> 6;
    int32_t* mine = base + blockIdx.x * nq;
    int32_t carry = 0;
    for (int64_t at = 0; at < nq; at += 1024) {
        const int64_t i = at + threadIdx.x;
        const int32_t v = i < nq ? mine[i] : 0;
        int32_t scan = v;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int32_t t = __shfl_up(scan, o);
            if (lane >= o) scan += t;
        }
        __syncthreads();  // the last round's sums are read
        if (lane == kWave - 1) part[w] = scan;
        __syncthreads();
        int32_t add = carry;
        for (int k = 0; k < 1024 / kWave; ++k) {
            if (k < w) add += part[k];
            carry += part[k];
        }
        if (i < nq) mine[i] = add + scan - v;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

// The strips, block by block, each block padded to whole groups of `per`.
__global__ __launch_bounds__(256) void strip_fill_kernel(int64_t nq, int32_t nb, int32_t per,
                                                         const int32_t* __restrict__ base,
                                                         const int32_t* __restrict__ total,
                                                         int2* __restrict__ items,
                                                         int32_t* __restrict__ used) {
    __shared__ int32_t before;
    const int32_t b = blockIdx.x;
    if (threadIdx.x == 0) before = 0;
    __syncthreads();
    int32_t sum = 0;
    for (int32_t i = threadIdx.x; i < b; i += 256) sum += (total[i] + per - 1) / per;
    if (sum != 0) atomicAdd(&before, sum);
    __syncthreads();
    const int32_t mine = total[b], groups = (mine + per - 1) / per;
    int2* out = items + static_cast<int64_t>(before) * per;
    const int64_t q = blockIdx.y * int64_t{256} + threadIdx.x;
    if (q < nq) {
        const int32_t at = base[b * nq + q], end = q + 1 < nq ? base[b * nq + q + 1] : mine;
        for (int32_t j = at; j < end; ++j)
            out[j] = int2{static_cast<int32_t>(q), b << 8 | (j - at)};
    }
    if (blockIdx.y == 0) {
        for (int32_t j = mine + threadIdx.x; j < groups * per; j += 256) out[j] = int2{-1, b << 8};
        if (b == nb - 1 && threadIdx.x == 0) *used = before + groups;
    }
}

struct Extent {
    int64_t nq, nb, groups;
};
Extent strip_extent(const slk_csr* W, const slk_strips* T) {
    Extent e;
    e.nq = ceil_div(W->nrows - T->first, int64_t{4});
    e.nb = ceil_div(W->ncols, T->block);
    // strips: at most one per quad and block, and one per S slots of a row
    e.groups = (e.nq * e.nb + W->total_capacity / T->slots) / (kWaves * T->per_wave) + e.nb;
    return e;
}

// (whole windows of two parts)
int64_t padded_n(int64_t N) { return ceil_div(N, int64_t{2 * kWin}) * (2 * kWin); }

int check_strips(const slk_csr* W, const slk_strips* T, const char* who) {
    clear_error();
    if (int rc = validate_csr(W, who)) return rc;
    const std::string at = std::string(who) + ": ";
    if (T == nullptr) return fail(SLK_EINVAL, at + "NULL strips");
    if (T->first < 0 || T->first >= W->nrows || W->ncols <= 0)
        return fail(SLK_EINVAL, at + "no rows or columns");
    if (T->block < 16 || T->block > kMaxC || T->block % 16 != 0)
        return fail(SLK_EINVAL, at + "blocks are multiples of 16 up to 256 columns");
    if (ceil_div(W->ncols, T->block) > kMaxBlocks) return fail(SLK_EINVAL, at + "too many columns");
    if (W->nrows > kMaxRows) return fail(SLK_EINVAL, at + "too many rows");
    if ((T->first > 0 || T->ordered != 0) && W->row_order == nullptr)
        return fail(SLK_EINVAL, at + "no row order");
    if (T->slots < 1 || T->slots > 128 || T->per_wave < 1 || T->per_wave > 8)
        return fail(SLK_EINVAL, at + "bad strip size");
    if ((T->parts != 1 && T->parts != 2) || T->block * T->parts > kMaxParts)
        return fail(SLK_EINVAL, at + "blocks of two parts have at most 144 columns");
    return SLK_OK;
}

template <int S, int R, int V>
int launch_strips(const slk_csr* W, const slk_strips* T, const float* dY, const float* X,
                  const float* XP, int64_t N, float* dW, hipStream_t st) {
    const Extent e = strip_extent(W, T);
    if (e.groups > INT32_MAX) return fail(SLK_EINVAL, "sddmm_strips: problem too large");
    const bool al = N % 4 == 0 && reinterpret_cast<uintptr_t>(dY) % 16 == 0;
    const size_t lds = static_cast<size_t>(2 * T->block * V * kWin * 4 + kWaves * 1024);
    auto* kernel = al ? strip_dw_kernel<S, R, V, true> : strip_dw_kernel<S, R, V, false>;
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) !=
            hipSuccess)
        return fail(SLK_EDEVICE, "sddmm_strips: LDS refused");
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(e.groups)), dim3(kWaves * kWave), lds, st,
                       W->nrows, W->ncols, N, padded_n(N), T->first,
                       T->ordered ? W->row_order : nullptr, W->row_start, W->col_indices, dY, X, XP, dW,
                       reinterpret_cast<const int2*>(T->items), T->rel, T->used,
                       static_cast<int32_t>(e.nb), static_cast<int32_t>(T->block));
    return check_launch("sddmm_strips");
}

// Estimated microseconds at N columns of strips of T's sizes (a fit to layer
// shapes of 256 to 8192 rows, N 256 to 8192, 1% to 70%: rounds of
// workgroups, one per CU, x windows x (barrier and staging + strips x (dY +
// steps)), a step being one slot of each of a quad's rows, as many as the
// longest row has), or a negative number where a row's slots of a block would
// often not fit one strip.
double strip_cost(int64_t M, int64_t K, int64_t N, double density, const slk_strips& T) {
    const double mu = density * T.block, sd = std::sqrt(mu * (1.0 - density)) + 1e-9;
    const double p = 0.5 * std::erfc((T.slots + 0.5 - mu) / sd * 0.70710678);
    const double extra = 1.0 - std::pow(1.0 - p, 4.0);
    if (extra > 0.25) return -1.0;
    const double steps = std::fmin(mu + 1.03 * sd + 1.0, static_cast<double>(T.slots));
    const int64_t nb = ceil_div(K, T.block);
    const double per_block =
        std::ceil(ceil_div(M, int64_t{4}) * (1.0 + extra) / (kWaves * T.per_wave));
    const double rounds = std::ceil(per_block * nb / 256.0);
    const double windows = std::ceil(N / 64.0);
    const double step = T.parts == 2 ? 0.040 : 0.044;
    const double stage = T.block * (rounds > 1.0 ? 0.003 : 0.001);
    const double tail = N % kWin != 0 ? 8.0 : 0.0;  // the last window's and the scalars' columns
    return 8.0 + tail + (2.0 * K + M) * N * 4.0 / 4.5e6 +
           rounds * windows * (0.2 + stage + T.per_wave * (0.06 + step * steps));
}

// The same for slk_sddmm: what its kernels reach (slots x columns per ns), and
// the chain of windows that one workgroup or wave runs however small the matrix.
// Segment kernel: N % 4 == 0 and N >= 1024, from 100000 slots; 4-slot segments
// below 1/16. The rates are those of the shapes on which both sides are timed in
// profiles/schedule_choices.md (256 to 4096 rows, 384 to 4096 columns, 3% to 30%, N
// 256 to 8192): of 475 where strips are taken they lose by over 3% on six (10% at
// most: 768 x 4096 at 5%, N = 2048, 58 -> 65 us). From 1.5 million slots below 1/8 the segment kernel gains (4096^2 at 10%,
// N = 8192: 1254 us against 1402 in strips), as it does where rows hold over 40 of
// 70000 to 100000 slots on the per-slot kernels (1000 x 768 at 10%, N = 1024: 19
// against 23).
double sddmm_estimate(const slk_csr* W, int64_t N, double density) {
    const double slots = W->total_capacity / 1.2, work = slots * N * 1e-3;
    double rate = 3.9, chain = 0.0;
    if (N % 4 == 0 && N >= 1024 && slots >= 1e5) {
        if (density >= 0.0625) rate = 7.6 + 13.5 * density;
        else if (4.0 * W->ncols * N >= (1 << 27)) rate = 5.6;
        else rate = density >= 0.04 ? 5.2 : 4.5;
        if (slots >= 2e6) rate *= 1.3;
        else if (slots >= 1.5e6 && density < 0.125) rate *= 1.2;
        chain = 1.25 * N / 64.0;
    } else if (N % 4 == 0) {
        rate = N < 1024 ? 3.75 : slots >= 7e4 && slots >= 40.0 * W->nrows ? 5.0 : 4.3;
        chain = N / 150.0;
    }
    return 4.0 + std::fmax(work / rate * 1e-3, chain);
}

}  // namespace
}  // namespace slk

extern "C" int slk_strip_choose(const slk_csr* W, int64_t N, slk_strips* T, double* us) {
    using namespace slk;
    clear_error();
    if (int rc = validate_csr(W, "strip_choose")) return rc;
    if (T == nullptr || us == nullptr) return fail(SLK_EINVAL, "strip_choose: NULL output");
    *T = slk_strips{};
    *us = 0.0;
    if (W->nrows == 0 || W->nrows > kMaxRows || W->ncols == 0 || N < 1 || N > (int64_t{1} << 21))
        return SLK_OK;
    // rows of very different lengths pad each other (16384^2 Zipf(1.1) at 95%:
    // 5.34 ms against 5.29, at 99% 3.3 against 2.1), and dense rows run on the
    // matrix cores
    if (W->n_heavy_rows > 0 || W->n_dense_rows > 0) return SLK_OK;
    const double density =
        std::fmin(1.0, static_cast<double>(W->total_capacity) / (1.2 * W->nrows * W->ncols));
    static constexpr int kSizes[][2] = {{48, 1}, {32, 1}, {16, 1}, {16, 2}};
    for (int64_t c = 16; c <= kMaxC; c += 16)
        for (const auto& z : kSizes)
            for (int64_t v = 1; v <= 2 && c * v <= kMaxParts; ++v) {
                slk_strips t = {};
                t.block = c;
                t.slots = z[0];
                t.per_wave = z[1];
                t.parts = v;
                if (ceil_div(W->ncols, c) > kMaxBlocks) continue;
                const double u = strip_cost(W->nrows, W->ncols, N, density, t);
                if (u > 0.0 && (T->block == 0 || u < *us)) {
                    *T = t;
                    *us = u;
                }
            }
    // (the margin covers what both estimates missed on the measured shapes)
    if (*us >= 0.92 * sddmm_estimate(W, N, density)) *T = slk_strips{};
    return SLK_OK;
}

extern "C" int slk_strip_words(const slk_csr* W, const slk_strips* T, int64_t* words) {
    using namespace slk;
    if (int rc = check_strips(W, T, "strip_words")) return rc;
    if (words == nullptr) return fail(SLK_EINVAL, "strip_words: NULL output");
    const Extent e = strip_extent(W, T);
    words[0] = 2 * e.groups * kWaves * T->per_wave;  // items
    words[1] = e.nq * 4 * (e.nb + 1);                // rel
    words[2] = e.nb * e.nq + e.nb;                   // scratch: base, total
    return SLK_OK;
}

extern "C" int64_t slk_strip_layout_bytes(int64_t ncols, int64_t N) {
    return ncols > 0 && N > 0 ? 4 * ncols * slk::padded_n(N) : 0;
}

extern "C" int slk_strip_build(const slk_csr* W, const slk_strips* T, int32_t* items, int32_t* rel,
                               int32_t* used, int32_t* ws, void* stream) {
    using namespace slk;
    if (int rc = check_strips(W, T, "strip_build")) return rc;
    if (items == nullptr || rel == nullptr || used == nullptr || ws == nullptr)
        return fail(SLK_EINVAL, "strip_build: NULL output");
    const Extent e = strip_extent(W, T);
    hipStream_t st = as_stream(stream);
    int32_t* total = ws + e.nb * e.nq;
    hipLaunchKernelGGL(strip_count_kernel, dim3(static_cast<unsigned>(e.nq)), dim3(256),
                       static_cast<unsigned>(16 * (e.nb + 1)), st, W->nrows, T->first, e.nq,
                       static_cast<int32_t>(e.nb), static_cast<int32_t>(T->block),
                       static_cast<int32_t>(T->slots), T->ordered ? W->row_order : nullptr,
                       W->row_start, W->row_nnz, W->col_indices, rel, ws);
    if (int rc = check_launch("strip_build: count")) return rc;
    hipLaunchKernelGGL(strip_scan_kernel, dim3(static_cast<unsigned>(e.nb)), dim3(1024), 0, st,
                       e.nq, ws, total);
    if (int rc = check_launch("strip_build: scan")) return rc;
    hipLaunchKernelGGL(strip_fill_kernel,
                       dim3(static_cast<unsigned>(e.nb),
                            static_cast<unsigned>(ceil_div(e.nq, int64_t{256}))),
                       dim3(256), 0, st, e.nq, static_cast<int32_t>(e.nb),
                       static_cast<int32_t>(kWaves * T->per_wave), ws, total,
                       reinterpret_cast<int2*>(items), used);
    return check_launch("strip_build: fill");
}

extern "C" int slk_sddmm_strips(const slk_csr* W, const slk_strips* T, const float* dY,
                                const float* X, int64_t N, float* dW, float* dbias, void* ws,
                                int64_t ws_bytes, void* stream) {
    using namespace slk;
    if (int rc = check_strips(W, T, "sddmm_strips")) return rc;
    if (T->items == nullptr || T->rel == nullptr || T->used == nullptr)
        return fail(SLK_EINVAL, "sddmm_strips: incomplete strips");
    if (N < 1 || N > (int64_t{1} << 21)) return fail(SLK_EINVAL, "sddmm_strips: N outside [1, 2^21]");
    if (dY == nullptr || X == nullptr || dW == nullptr)
        return fail(SLK_EINVAL, "sddmm_strips: NULL operand");
    const int64_t need = slk_strip_layout_bytes(W->ncols, N);
    if (ws == nullptr || ws_bytes < need || reinterpret_cast<uintptr_t>(ws) % 16 != 0)
        return fail(SLK_EINVAL, "sddmm_strips: workspace of " + std::to_string(ws_bytes) +
                                    " bytes, needs " + std::to_string(need) + ", 16-byte aligned");
    hipStream_t st = as_stream(stream);
    float* XP = static_cast<float*>(ws);
    const int64_t quads = ceil_div(N, int64_t{4 * kWin}), items = W->ncols * quads;
    const int64_t lb = ceil_div(items + W->nrows, int64_t{4});
    if (lb > INT32_MAX) return fail(SLK_EINVAL, "sddmm_strips: problem too large");
    hipLaunchKernelGGL(strip_layout_kernel, dim3(static_cast<unsigned>(lb)), dim3(256), 0, st, N,
                       padded_n(N), quads, items, X, XP, W->nrows, W->row_start, W->row_nnz, W->row_capacity,
                       dY, dW, dbias);
    if (int rc = check_launch("sddmm_strips: layout")) return rc;
    switch (T->slots * 100 + T->per_wave * 10 + T->parts) {
        case 4811: return launch_strips<48, 1, 1>(W, T, dY, X, XP, N, dW, st);
        case 4812: return launch_strips<48, 1, 2>(W, T, dY, X, XP, N, dW, st);
        case 3211: return launch_strips<32, 1, 1>(W, T, dY, X, XP, N, dW, st);
        case 3212: return launch_strips<32, 1, 2>(W, T, dY, X, XP, N, dW, st);
        case 1611: return launch_strips<16, 1, 1>(W, T, dY, X, XP, N, dW, st);
        case 1612: return launch_strips<16, 1, 2>(W, T, dY, X, XP, N, dW, st);
        case 1621: return launch_strips<16, 2, 1>(W, T, dY, X, XP, N, dW, st);
        case 1622: return launch_strips<16, 2, 2>(W, T, dY, X, XP, N, dW, st);
        default: return fail(SLK_EINVAL, "sddmm_strips: no kernel for " + std::to_string(T->slots) +
                                             " slots x " + std::to_string(T->per_wave) + " strips x " +
                                             std::to_string(T->parts) + " parts");
    }
}

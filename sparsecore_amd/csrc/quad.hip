// SpMM over a stream of row quads (gfx950): Y = W·X for layers wide and dense
// enough that each staged X element serves several rows.
//
// Every output element is the row's fma chain in slot order from +0.0
// (csrc/kernels/spmm_avx2.cpp:123-262): the same bits as slk_spmm.
//
// The LDS kernel of spmm.hip gives a whole wave to one row at a time: each
// slot's column and value are broadcast by readlane, and its runs of a few
// slots per chunk cost branches and scalar work that outweigh the four fmas
// per lane (16384^2 at 5%: 121 cycles per SIMD for a slot's 512 columns, of
// which the fmas are 20). Here a wave holds four rows side by side, 16 lanes
// each. A stream built per topology lists, per quad of rows and chunk of X
// rows, windows of 16 slots of each of the four rows, one slot per lane (row r
// in lanes 16r .. 16r + 15): its X row's LDS offset and its value. Step i of a
// window broadcasts lane i of each 16-lane row to that row with DPP
// (row_newbcast): one add for the address, one or two 16-byte LDS reads (256
// contiguous bytes per row, conflict-free), one move for the value, and the
// fmas: no readlane, no per-slot scalar work, and a branch every two steps.
// Straight-line, that runs at 54 (64 columns a row) and 64 (128 columns)
// TFLOP/s. What bounds it is the vector unit's issue: 2304 x 768 at 30%, N = 8192,
// and the 16384^2 transpose at 5% keep it busy 74% and 73% of the cycles, with 8%
// and 1% of the waves' cycles waiting to issue to the LDS; 6 to 8 instructions
// per slot and 256 columns, padding included, of which the fmas are 4. Rows of a
// quad with fewer slots than its longest are padded with a zero X row and the value
// -0.0, which leaves every sum as it is (x + -0.0 = x for every x, NaN and
// both zeros included).
//
// Measured against slk_spmm, values kernel included: 2304 x 768 at 20%, N =
// 8192, 238 -> 190 us; 768 x 3072 at 30%, N = 4096, 286 -> 196; 4096^2 at 10%,
// N = 4096, 566 -> 462 (30 TFLOP/s of useful slots; about a third of the
// steps are padding, the rest of the gap is the windows and chunk barriers);
// 3072 x 768 at 10%, N = 1001, 87 -> 37 us (no 16-byte lanes: the other path
// is the gather kernel).
#include "common.hpp"

namespace slk {
namespace {

constexpr uint32_t kBufWord3 = 0x00020000;  // gfx9 buffer resource dword 3
constexpr int kWaves = 16;
constexpr int kChunkBytes = 64 * 1024;  // one X chunk's buffer; its last KiB is the zero row
constexpr int kZeroOff = kChunkBytes - 1024;
constexpr int kAhead = 3;               // windows in flight per wave
constexpr int kWinBytes = 512;          // 64 offsets, 64 values
constexpr int kQuadLds = 2 * kChunkBytes + kWaves * (kAhead + 1) * kWinBytes;  // all 160 KiB
constexpr int64_t kMaxChunks = 2048;

// X rows per chunk for H 64-column halves of a row
__host__ __device__ constexpr int chunk_rows(int h) { return kZeroOff / (256 * h); }

__device__ __forceinline__ void lds_load16(const void* base, uint32_t bytes, uint32_t vo,
                                           void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0),
                                          static_cast<int>(bytes), kBufWord3),
        (__attribute__((address_space(3))) void*)lds, 16, vo, 0, 0, 0);
}
__device__ __forceinline__ void lds_load4(const void* base, uint32_t bytes, uint32_t vo,
                                          uint32_t so, void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0),
                                          static_cast<int>(bytes), kBufWord3),
        (__attribute__((address_space(3))) void*)lds, 4, vo, so, 0, 0);
}

// at most N vector-memory operations of this wave outstanding
template <int N>
__device__ __forceinline__ void vm_le() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// lane I of each row of 16 lanes, in all 16
template <int I>
__device__ __forceinline__ int row_bcast(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + I, 0xf, 0xf, true);
}

// ───────────────────────────── the kernel ───────────────────────────────────
//
// A workgroup of 16 waves owns 64·RW rows x 64·H columns of Y: wave w's quad j
// is quad (row block)·16·RW + 16 j + w, its sums RW·H·4 registers. X goes
// through LDS in chunks of chunk_rows(H) rows, double-buffered, by direct
// loads; a wave's windows go through a ring of four in LDS, three in flight, by
// direct loads too, so that nothing in the loop waits for a register load
// behind the next chunk's staging. The quads' window counts and starts for
// this chunk and the next sit in the lanes of two registers, so that the
// prefetch can run past the chunk's end. AL: X, Y and N allow 16-byte accesses.
template <int RW, int H, bool AL>
__global__ __launch_bounds__(kWaves * kWave, 4) void quad_spmm_kernel(
    int64_t M, int64_t K, int64_t N, int64_t nq, int64_t nrowblk,
    const int32_t* __restrict__ qstart, const uint8_t* __restrict__ qcount,
    const uint32_t* __restrict__ qoff, const float* __restrict__ qval,
    const float* __restrict__ X, const float* __restrict__ bias, float* __restrict__ Y) {
    constexpr int KC = chunk_rows(H), kRowBytes = 256 * H, kCols = 64 * H;
    static_assert(RW >= kAhead, "the prefetch stays within the next chunk");
    __shared__ __align__(1024) char smem[kQuadLds];
    const int lane = threadIdx.x & (kWave - 1), l16 = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    char* ring = smem + 2 * kChunkBytes + w * ((kAhead + 1) * kWinBytes);
    const int64_t lb = xcd_logical_block(blockIdx.x, gridDim.x);
    const int64_t tile = lb / nrowblk, rb = lb - tile * nrowblk;
    const int64_t n0 = tile * kCols;
    const int64_t q0 = rb * (kWaves * RW) + w;  // the wave's quad j: q0 + 16 j
    const int32_t nch = static_cast<int32_t>(ceil_div(K, int64_t{KC}));
    const uint32_t rowb = static_cast<uint32_t>(4 * N);

    if (threadIdx.x < 2 * kWave)  // the zero row behind each chunk buffer
        *reinterpret_cast<f32x4*>(smem + (threadIdx.x >> 6) * kChunkBytes + kZeroOff + lane * 16) =
            f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // chunk ch into buffer buf (rows past K repeat the last, columns past N the
    // last four: no slot reads the former, no lane stores the latter)
    auto stage = [&](int buf, int32_t ch) {
        char* xb = smem + buf * kChunkBytes;
        const int64_t k0 = static_cast<int64_t>(ch) * KC;
        const int32_t last = static_cast<int32_t>(K - k0 < KC ? K - k0 : KC) - 1;
        const float* src = X + k0 * N;
        const uint32_t bytes = static_cast<uint32_t>(last + 1) * rowb;
        if constexpr (AL) {
            constexpr int kLanes = kRowBytes / 16, kPieces = kZeroOff / 1024;
            const int64_t n = n0 + 4 * (lane % kLanes);
            const uint32_t vo = static_cast<uint32_t>((n < N ? n : N - 4) * 4);
#pragma unroll
            for (int i = 0; i < (kPieces + kWaves - 1) / kWaves; ++i) {
                const int p = w + i * kWaves;
                if (p < kPieces) {
                    const int r = p * (kWave / kLanes) + lane / kLanes;
                    lds_load16(src, bytes, vo + static_cast<uint32_t>(r < last ? r : last) * rowb,
                               xb + p * 1024);
                }
            }
        } else {
            constexpr int kPieces = kZeroOff / 256;
#pragma unroll 4
            for (int i = 0; i < (kPieces + kWaves - 1) / kWaves; ++i) {
                const int p = w + i * kWaves;
                if (p < kPieces) {
                    const int r = p / H;
                    const int64_t n = n0 + (p % H) * kWave + lane;
                    lds_load4(src, bytes, static_cast<uint32_t>((n < N ? n : N - 1) * 4),
                              static_cast<uint32_t>(r < last ? r : last) * rowb, xb + p * 256);
                }
            }
        }
    };

    // lane j < RW: quad j in chunk ch; lane RW + j: in chunk ch + 1
    auto describe = [&](int32_t ch, int32_t& start, int32_t& count) {
        const int64_t q = q0 + static_cast<int64_t>(lane % RW) * kWaves;
        const int64_t c = ch + lane / RW;
        const bool ok = lane < 2 * RW && q < nq && c < nch;
        start = ok ? qstart[c * nq + q] : 0;
        count = ok ? qcount[c * nq + q] : 0;
    };
    auto windows = [](int32_t n) { return n > 16 ? (n + 15) >> 4 : 1; };
    int32_t vs, vn, next_s, next_n;
    describe(0, vs, vn);
    int32_t ij = 0, iw = 0, fi = 0, f = 0;  // next window to load: quad ij's iw-th; ring indices
    auto load_window = [&] {
        const int64_t at =
            static_cast<int64_t>(__builtin_amdgcn_readlane(vs, ij) + iw) * kWave;
        char* dst = ring + (fi & kAhead) * kWinBytes;
        lds_load4(qoff + at, 256, lane * 4, 0, dst);
        lds_load4(qval + at, 256, lane * 4, 0, dst + 256);
        ++fi;
        ++iw;
        const bool done = iw >= windows(__builtin_amdgcn_readlane(vn, ij));
        ij += done ? 1 : 0;
        iw = done ? 0 : iw;
    };

    f32x4 acc[RW][H];
#pragma unroll
    for (int j = 0; j < RW; ++j)
#pragma unroll
        for (int h = 0; h < H; ++h) acc[j][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    stage(0, 0);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) load_window();
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    // (past the last chunk the last one is staged again, into the free buffer)
    for (int32_t ch = 0; ch < nch; ++ch) {
        const int b = ch & 1;
        describe(ch + 1, next_s, next_n);
        stage(b ^ 1, ch + 1 < nch ? ch + 1 : nch - 1);
        const int lx = b * kChunkBytes + l16 * 16;
        static_for<RW>([&](auto J) {
            constexpr int j = decltype(J)::value;
            const int32_t n = __builtin_amdgcn_readlane(vn, j);
            const int32_t nw = windows(n);
            for (int32_t iwin = 0; iwin < nw; ++iwin) {
                vm_le<2 * (kAhead - 1)>();  // window f is in LDS: two loads per later one
                const char* src = ring + (f & kAhead) * kWinBytes;
                const int off = *reinterpret_cast<const int*>(src + lane * 4);
                const int val = *reinterpret_cast<const int*>(src + 256 + lane * 4);
                load_window();  // into the slot of window f - 1, read before
                ++f;
                const int32_t m = n - 16 * iwin;
                f32x4 x[4][H];
                auto reads = [&](auto S) {
                    constexpr int s0 = decltype(S)::value;
                    static_for<4>([&](auto I) {
                        constexpr int i = decltype(I)::value;
                        const int a = row_bcast<s0 + i>(off) + lx;
#pragma unroll
                        for (int h = 0; h < H; ++h)
                            x[i][h] = *reinterpret_cast<const f32x4*>(smem + a + h * 256);
                    });
                    __builtin_amdgcn_sched_barrier(0);
                };
                auto fmas = [&](auto S, auto I0) {
                    constexpr int s0 = decltype(S)::value, i0 = decltype(I0)::value;
                    static_for<2>([&](auto I) {
                        constexpr int i = i0 + decltype(I)::value;
                        const float v = __int_as_float(row_bcast<s0 + i>(val));
#pragma unroll
                        for (int h = 0; h < H; ++h)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                acc[j][h][e] = __builtin_fmaf(v, x[i][h][e], acc[j][h][e]);
                    });
                };
                using C0 = std::integral_constant<int, 0>;
                using C2 = std::integral_constant<int, 2>;
                using C4 = std::integral_constant<int, 4>;
                using C8 = std::integral_constant<int, 8>;
                using C12 = std::integral_constant<int, 12>;
                // (nested, so that the sums meet at one place only)
                if (m > 0) {
                    reads(C0{});
                    fmas(C0{}, C0{});
                    if (m > 2) {
                        fmas(C0{}, C2{});
                        if (m > 4) {
                            reads(C4{});
                            fmas(C4{}, C0{});
                            if (m > 6) {
                                fmas(C4{}, C2{});
                                if (m > 8) {
                                    reads(C8{});
                                    fmas(C8{}, C0{});
                                    if (m > 10) {
                                        fmas(C8{}, C2{});
                                        if (m > 12) {
                                            reads(C12{});
                                            fmas(C12{}, C0{});
                                            if (m > 14) fmas(C12{}, C2{});
                                        }
                                    }
                                }
                            }
                        }
                    }
                }
            }
        });
        // This wave's loads of the next chunk are down: at least RW windows'
        // loads, two each, were issued after them, and kAhead of those may fly
        // on. Then the barrier (a bare one: __syncthreads() waits for all).
        vm_le<2 * kAhead>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        vs = next_s;
        vn = next_n;
        ij -= RW;
    }
    __builtin_amdgcn_s_waitcnt(0);  // no direct load still writing LDS when the waves end
#pragma unroll
    for (int j = 0; j < RW; ++j) {
        const int64_t row = (q0 + static_cast<int64_t>(j) * kWaves) * 4 + (lane >> 4);
        if (row >= M) continue;
        const float bb = bias != nullptr ? bias[row] : 0.0f;
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const int64_t n = n0 + h * 64 + 4 * l16;
            f32x4 a = acc[j][h];
            if (bias != nullptr) {
#pragma unroll
                for (int e = 0; e < 4; ++e) a[e] = a[e] + bb;
            }
            if constexpr (AL) {
                if (n < N) *reinterpret_cast<f32x4*>(Y + row * N + n) = a;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) Y[row * N + n + e] = a[e];
            }
        }
    }
}

// val[i] = values[slot[i]], -0.0 where no slot is; *used windows
__global__ __launch_bounds__(256) void quad_values_kernel(const int32_t* __restrict__ used,
                                                          const int32_t* __restrict__ slot,
                                                          const float* __restrict__ values,
                                                          float* __restrict__ val) {
    const int64_t n = static_cast<int64_t>(*used) * (kWave / 4);
    for (int64_t i = blockIdx.x * int64_t{256} + threadIdx.x; i < n; i += gridDim.x * int64_t{256}) {
        typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
        const i32x4 s = reinterpret_cast<const i32x4*>(slot)[i];
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = s[e] >= 0 ? values[s[e]] : -0.0f;
        reinterpret_cast<f32x4*>(val)[i] = v;
    }
}

// ───────────────────────────── the build ────────────────────────────────────

// Per quad: each row's first slot in every chunk (rel[q][r][0 .. nch],
// relative to row_start), the chunk counts (the longest of the four rows),
// the chunks' window starts relative to the quad's, the quad's windows.
template <int KC>
__global__ __launch_bounds__(256) void quad_count_kernel(
    int64_t M, int64_t nq, int32_t nch, const int32_t* __restrict__ row_start,
    const int32_t* __restrict__ row_nnz, const int32_t* __restrict__ col,
    int32_t* __restrict__ rel, int32_t* __restrict__ qstart, uint8_t* __restrict__ qcount,
    int32_t* __restrict__ total) {
    extern __shared__ int32_t st[];  // [4][nch + 1]
    const int64_t q = blockIdx.x;
    const int r = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
    const int64_t row = 4 * q + r;
    int32_t* mine = st + r * (nch + 1);
    const int32_t s0 = row < M ? row_start[row] : 0, n = row < M ? row_nnz[row] : 0;
    int32_t before = -1;  // the chunk of the slot before this batch
    for (int32_t base = 0; base <= n; base += kWave) {
        const int32_t s = base + lane;
        const int32_t c = s < n ? col[s0 + s] / KC : nch;
        int32_t p = __shfl_up(c, 1);
        if (lane == 0) p = before;
        if (s <= n)
            for (int32_t x = p + 1; x <= c; ++x) mine[x] = s;
        before = __shfl(c, kWave - 1);
    }
    __syncthreads();
    for (int32_t i = threadIdx.x; i < 4 * (nch + 1); i += 256)
        rel[q * 4 * (nch + 1) + i] = st[i];
    if (r != 0) return;
    int32_t sum = 0;
    for (int32_t base = 0; base < nch; base += kWave) {
        const int32_t ch = base + lane;
        int32_t most = 0;
        if (ch < nch)
            for (int k = 0; k < 4; ++k)
                most = max(most, st[k * (nch + 1) + ch + 1] - st[k * (nch + 1) + ch]);
        const int32_t nw = ch < nch ? (most > 16 ? (most + 15) >> 4 : 1) : 0;
        int32_t scan = nw;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int32_t t = __shfl_up(scan, o);
            if (lane >= o) scan += t;
        }
        if (ch < nch) {
            qstart[static_cast<int64_t>(ch) * nq + q] = sum + scan - nw;
            qcount[static_cast<int64_t>(ch) * nq + q] = static_cast<uint8_t>(most);
        }
        sum += __shfl(scan, kWave - 1);
    }
    if (lane == 0) total[q] = sum;
}

// total[0 .. nq) to its exclusive scan, total[nq] the sum: one workgroup.
__global__ __launch_bounds__(1024) void quad_scan_kernel(int64_t nq, int32_t* __restrict__ total) {
    __shared__ int32_t part[1024 / kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x >> 6;
    int32_t carry = 0;
    for (int64_t base = 0; base < nq; base += 1024) {
        const int64_t i = base + threadIdx.x;
        const int32_t v = i < nq ? total[i] : 0;
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
        if (i < nq) total[i] = add + scan - v;
    }
    if (threadIdx.x == 0) total[nq] = carry;
}

// The windows: lane 16 r + i of a window holds slot 16·(window) + i of row r's
// run in the chunk. With perm (a transpose's slot map) the stored slot is
// perm[slot], so that the values come from the transposed matrix's own.
template <int KC>
__global__ __launch_bounds__(256) void quad_fill_kernel(
    int64_t M, int64_t nq, int32_t nch, const int32_t* __restrict__ row_start,
    const int32_t* __restrict__ col, const int64_t* __restrict__ perm,
    const int32_t* __restrict__ rel, const int32_t* __restrict__ total,
    int32_t* __restrict__ qstart, const uint8_t* __restrict__ qcount, uint32_t* __restrict__ qoff,
    int32_t* __restrict__ qslot, int64_t n_windows, int32_t row_bytes) {
    const int64_t q = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1), r = lane >> 4, l16 = lane & 15;
    const int64_t row = 4 * q + r;
    const int32_t s0 = row < M ? row_start[row] : 0;
    const int32_t base = total[q];
    const int32_t* mine = rel + (q * 4 + r) * (nch + 1);
    for (int32_t ch = threadIdx.x >> 6; ch < nch; ch += 4) {
        const int64_t at = static_cast<int64_t>(ch) * nq + q;
        const int32_t first = qstart[at] + base, n = qcount[at];
        const int32_t nw = n > 16 ? (n + 15) >> 4 : 1;
        const int32_t lo = mine[ch], hi = mine[ch + 1];
        for (int32_t iw = 0; iw < nw && first + iw < n_windows; ++iw) {
            const int32_t s = lo + 16 * iw + l16;
            const int64_t i = static_cast<int64_t>(first + iw) * kWave + lane;
            uint32_t off = kZeroOff;
            int32_t slot = -1;
            if (s < hi) {
                slot = s0 + s;
                off = static_cast<uint32_t>(col[slot] - ch * KC) * static_cast<uint32_t>(row_bytes);
                if (perm != nullptr) slot = static_cast<int32_t>(perm[slot]);
            }
            qoff[i] = off;
            qslot[i] = slot;
        }
        if (lane == 0) qstart[at] = first;
    }
}

bool halves_ok(int64_t h) { return h == 1 || h == 2; }

template <int RW, int H, bool AL>
int launch_quad(const slk_csr* W, const slk_quads* Q, const float* val, const float* X, int64_t N,
                const float* bias, float* Y, hipStream_t st) {
    const int64_t nq = ceil_div(W->nrows, int64_t{4});
    const int64_t nrowblk = ceil_div(nq, int64_t{kWaves} * RW);
    const int64_t blocks = nrowblk * ceil_div(N, int64_t{64} * H);
    if (blocks > INT32_MAX) return fail(SLK_EINVAL, "spmm_quad: problem too large for one launch");
    hipLaunchKernelGGL((quad_spmm_kernel<RW, H, AL>), dim3(static_cast<unsigned>(blocks)),
                       dim3(kWaves * kWave), 0, st, W->nrows, W->ncols, N, nq, nrowblk,
                       Q->start, Q->count, Q->offset, val, X, bias, Y);
    return check_launch("spmm_quad");
}

template <int H, bool AL>
int launch_quad_rw(int rw, const slk_csr* W, const slk_quads* Q, const float* val, const float* X,
                   int64_t N, const float* bias, float* Y, hipStream_t st) {
    switch (rw) {
        case 3: return launch_quad<3, H, AL>(W, Q, val, X, N, bias, Y, st);
        case 4: return launch_quad<4, H, AL>(W, Q, val, X, N, bias, Y, st);
        case 6: return launch_quad<6, H, AL>(W, Q, val, X, N, bias, Y, st);
        case 8: return launch_quad<8, H, AL>(W, Q, val, X, N, bias, Y, st);
        case 9:
            if constexpr (H == 1) return launch_quad<9, H, AL>(W, Q, val, X, N, bias, Y, st);
            break;
        case 16:
            if constexpr (H == 1) return launch_quad<16, H, AL>(W, Q, val, X, N, bias, Y, st);
            break;
        default: break;
    }
    return fail(SLK_EINVAL, "spmm_quad: no kernel for " + std::to_string(rw) + " quads per wave");
}

// Estimated microseconds: rounds of workgroups (one per CU, by its LDS) x X
// chunks x (staging and barrier + quads x (window + steps)), a step being one
// slot of each of the quad's rows, as many per chunk as its longest row has
// (about one standard deviation above the mean). The constants are a fit to layer
// shapes of 37 to 16384 rows, 50 to 4096 columns, N 41 to 16384 and 1% to 60%; of
// the 524 shapes on which both sides are timed in profiles/schedule_choices.md
// quads lose on two by over 3% (4% at most).
double quad_cost(int64_t M, int64_t K, int64_t N, double density, int h, int rw) {
    const double mu = density * chunk_rows(h);
    const double steps = mu + 1.03 * __builtin_sqrt(mu) + 1.0;
    const int64_t blocks =
        ceil_div(ceil_div(M, int64_t{4}), int64_t{kWaves} * rw) * ceil_div(N, int64_t{64} * h);
    const double rounds = static_cast<double>(ceil_div(blocks, int64_t{256}));
    const double chunks = static_cast<double>(ceil_div(K, int64_t{chunk_rows(h)}));
    const double fixed = N % 4 == 0 ? 40.0 : 90.0;
    return 6.0 + 0.038 * rounds * chunks * (fixed + rw * (4.0 + steps * (h == 2 ? 1.7 : 1.0)));
}

double capacity_density(const slk_csr* W) {
    return static_cast<double>(W->total_capacity) / (1.2 * W->nrows * W->ncols);
}

// The quads per wave with the least estimate (SLK_TUNE_QUAD_RW overrides).
int quad_rw(const slk_csr* W, int h, int64_t N, double* cost = nullptr) {
    int best = 0;
    double least = 0.0;
    for (const int rw : {3, 4, 6, 8, 9, 16}) {
        if (h == 2 && rw > 8) continue;
        const double c = quad_cost(W->nrows, W->ncols, N, capacity_density(W), h, rw);
        if (best == 0 || c < least) {
            best = rw;
            least = c;
        }
    }
    if (cost != nullptr) *cost = least;
    if (const int64_t t = tuning(SLK_TUNE_QUAD_RW); t > 0) best = static_cast<int>(t);
    return best;
}

}  // namespace
}  // namespace slk

extern "C" int64_t slk_quad_windows(const slk_csr* W, int64_t halves) {
    using namespace slk;
    if (W == nullptr || !halves_ok(halves) || W->nrows <= 0 || W->ncols <= 0) return 0;
    // per quad and chunk ceil(longest / 16), at least one; the longest of four
    // rows is at most their sum
    const int64_t nq = ceil_div(W->nrows, int64_t{4});
    return W->total_capacity / 16 + nq * ceil_div(W->ncols, int64_t{chunk_rows(static_cast<int>(halves))});
}

extern "C" int64_t slk_quad_chunks(int64_t ncols, int64_t halves) {
    using namespace slk;
    if (ncols <= 0 || !halves_ok(halves)) return 0;
    return ceil_div(ncols, int64_t{chunk_rows(static_cast<int>(halves))});
}

extern "C" int64_t slk_quad_halves(const slk_csr* W, int64_t N) {
    using namespace slk;
    if (W == nullptr || W->nrows <= 0 || W->ncols <= 0 || N < 4 || N > (int64_t{1} << 22)) return 0;
    // rows of very different lengths would pad each other, and rows dense
    // enough for the matrix cores are faster there
    if (W->n_heavy_rows > 0 || W->n_dense_rows > 0) return 0;
    for (const int k : {SLK_TUNE_SPMM_KERNEL, SLK_TUNE_SPMM_H, SLK_TUNE_SPMM_RW, SLK_TUNE_SPMM_SPLIT,
                        SLK_TUNE_SPMM_VEC, SLK_TUNE_SPMM_BIN, SLK_TUNE_SPMM_G, SLK_TUNE_DENSE_ROWS})
        if (tuning(k) >= 0) return 0;
    double least = 0.0;
    int best = 0;
    for (const int h : {1, 2}) {
        if (slk_quad_chunks(W->ncols, h) > kMaxChunks || slk_quad_windows(W, h) > INT32_MAX) continue;
        double c;
        quad_rw(W, h, N, &c);
        if (best == 0 || c < least) {
            least = c;
            best = h;
        }
    }
    return best != 0 && least < 0.9 * spmm_estimate(W, N) ? best : 0;
}

namespace slk {
namespace {

// What every part of the build checks; the quads and chunks.
int quad_extent(const slk_csr* W, int64_t halves, int64_t ws_words, const char* who, int64_t* nq,
                int64_t* nch) {
    clear_error();
    if (int rc = validate_csr(W, who)) return rc;
    const std::string at = std::string(who) + ": ";
    if (!halves_ok(halves)) return fail(SLK_EINVAL, at + "halves must be 1 or 2");
    if (W->nrows == 0 || W->ncols == 0) return fail(SLK_EINVAL, at + "empty matrix");
    *nq = ceil_div(W->nrows, int64_t{4});
    *nch = slk_quad_chunks(W->ncols, halves);
    if (*nch > kMaxChunks) return fail(SLK_EINVAL, at + "too many columns");
    if (*nq > INT32_MAX || slk_quad_windows(W, halves) > INT32_MAX)  // (their scan is 32-bit)
        return fail(SLK_EINVAL, at + "too many windows");
    const int64_t need = *nq * 4 * (*nch + 1);
    if (ws_words < need)
        return fail(SLK_EINVAL, at + "workspace of " + std::to_string(ws_words) + " words, needs " +
                                    std::to_string(need));
    return SLK_OK;
}

}  // namespace
}  // namespace slk

extern "C" int slk_quad_count(const slk_csr* W, int64_t halves, int32_t* ws, int64_t ws_words,
                              int32_t* start, uint8_t* count, int32_t* used, void* stream) {
    using namespace slk;
    int64_t nq = 0, nch = 0;
    if (int rc = quad_extent(W, halves, ws_words, "quad_build", &nq, &nch)) return rc;
    if (ws == nullptr || start == nullptr || count == nullptr || used == nullptr)
        return fail(SLK_EINVAL, "quad_build: NULL output");
    hipStream_t st = as_stream(stream);
    auto* kernel = halves == 2 ? quad_count_kernel<chunk_rows(2)> : quad_count_kernel<chunk_rows(1)>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(nq)), dim3(256),
                       static_cast<unsigned>(16 * (nch + 1)), st, W->nrows, nq,
                       static_cast<int32_t>(nch), W->row_start, W->row_nnz, W->col_indices, ws,
                       start, count, used);
    if (int rc = check_launch("quad_build: count")) return rc;
    hipLaunchKernelGGL(quad_scan_kernel, dim3(1), dim3(1024), 0, st, nq, used);
    return check_launch("quad_build: scan");
}

extern "C" int slk_quad_fill(const slk_csr* W, const int64_t* perm, int64_t halves, int32_t* ws,
                             int64_t ws_words, int32_t* start, uint8_t* count, uint32_t* offset,
                             int32_t* slot, int64_t n_windows, int32_t* used, void* stream) {
    using namespace slk;
    int64_t nq = 0, nch = 0;
    if (int rc = quad_extent(W, halves, ws_words, "quad_build", &nq, &nch)) return rc;
    if (n_windows < 1) return fail(SLK_EINVAL, "quad_build: no windows");
    if (ws == nullptr || start == nullptr || count == nullptr || offset == nullptr ||
        slot == nullptr || used == nullptr)
        return fail(SLK_EINVAL, "quad_build: NULL output");
    auto* kernel = halves == 2 ? quad_fill_kernel<chunk_rows(2)> : quad_fill_kernel<chunk_rows(1)>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(nq)), dim3(256), 0, as_stream(stream),
                       W->nrows, nq, static_cast<int32_t>(nch), W->row_start, W->col_indices, perm,
                       ws, used, start, count, offset, slot, n_windows,
                       static_cast<int32_t>(256 * halves));
    return check_launch("quad_build: fill");
}

extern "C" int slk_quad_build(const slk_csr* W, const int64_t* perm, int64_t halves, int32_t* ws,
                              int64_t ws_words, int32_t* start, uint8_t* count, uint32_t* offset,
                              int32_t* slot, int64_t n_windows, int32_t* used, void* stream) {
    using namespace slk;
    int64_t nq = 0, nch = 0;
    if (int rc = quad_extent(W, halves, ws_words, "quad_build", &nq, &nch)) return rc;
    if (n_windows < slk_quad_windows(W, halves))
        return fail(SLK_EINVAL, "quad_build: workspace of " + std::to_string(n_windows) +
                                    " windows, needs " +
                                    std::to_string(slk_quad_windows(W, halves)));
    if (offset == nullptr || slot == nullptr) return fail(SLK_EINVAL, "quad_build: NULL output");
    if (int rc = slk_quad_count(W, halves, ws, ws_words, start, count, used, stream)) return rc;
    return slk_quad_fill(W, perm, halves, ws, ws_words, start, count, offset, slot, n_windows, used,
                         stream);
}

extern "C" int slk_spmm_quad(const slk_csr* W, const slk_quads* Q, const float* values,
                             float* val_ws, const float* X, int64_t K, int64_t N,
                             const float* bias, float* Y, void* stream) {
    using namespace slk;
    clear_error();
    if (int rc = validate_csr(W, "spmm_quad")) return rc;
    if (Q == nullptr || !halves_ok(Q->halves) || Q->start == nullptr || Q->count == nullptr ||
        Q->offset == nullptr || Q->slot == nullptr || Q->used == nullptr || Q->n_windows < 1)
        return fail(SLK_EINVAL, "spmm_quad: incomplete quad stream");
    if (W->ncols != K)
        return fail(SLK_EINVAL, "spmm_quad: shape mismatch. W has ncols=" +
                                    std::to_string(W->ncols) + " but X has shape[0]=" +
                                    std::to_string(K));
    if (W->nrows == 0 || N == 0) return SLK_OK;
    // a chunk of X in one buffer resource: 252 rows of 4 N bytes below 2^32
    if (N < 4 || N > (int64_t{1} << 22)) return fail(SLK_EINVAL, "spmm_quad: N outside [4, 2^22]");
    if (K == 0 || X == nullptr || Y == nullptr || values == nullptr || val_ws == nullptr)
        return fail(SLK_EINVAL, "spmm_quad: NULL or empty operand");
    hipStream_t st = as_stream(stream);
    const int64_t groups = Q->n_windows * (kWave / 4);
    const int64_t vb = groups < 256 * 2048 ? ceil_div(groups, int64_t{256}) : 2048;
    hipLaunchKernelGGL(quad_values_kernel, dim3(static_cast<unsigned>(vb)), dim3(256), 0, st,
                       Q->used + ceil_div(W->nrows, int64_t{4}), Q->slot, values, val_ws);
    if (int rc = check_launch("spmm_quad: values")) return rc;
    const bool al = N % 4 == 0 && (reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Y)) % 16 == 0;
    const int h = static_cast<int>(Q->halves), rw = quad_rw(W, h, N);
    if (h == 2) return al ? launch_quad_rw<2, true>(rw, W, Q, val_ws, X, N, bias, Y, st)
                          : launch_quad_rw<2, false>(rw, W, Q, val_ws, X, N, bias, Y, st);
    return al ? launch_quad_rw<1, true>(rw, W, Q, val_ws, X, N, bias, Y, st)
              : launch_quad_rw<1, false>(rw, W, Q, val_ws, X, N, bias, Y, st);
}

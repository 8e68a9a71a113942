// Planning and launches of the prefill-shaped quantized matmul (qmm_kernel.hpp):
// tile shape and split of K, split reduction, row pieces of weights beyond the
// buffer offsets, routed experts, and re-packing of the other code widths.
#include <mutex>

#include "qmm_kernel.hpp"

namespace eq {

// y = bf16(sum over splits of the partial tiles), splits summed in order.
// y[m, n] (row stride ldy) = bf16(sum over splits of ws[split, m, n]), the
// partials dense [splits, M, N] f32; four outputs per thread (vec: y 8-byte
// aligned and N, ldy multiples of 4, so the four stay in one row).
template <typename XT = BF16T>
__global__ __launch_bounds__(256) void qmm_split_reduce(uint16_t* __restrict__ y, const float* __restrict__ ws,
                                                         int64_t mn, int64_t n, int64_t ldy, int splits, bool vec) {
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    const int64_t i = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
    if (i >= mn) return;
    if (vec && i + 4 <= mn) {
        f32x4_t v = *reinterpret_cast<const f32x4_t*>(ws + i);
        for (int s = 1; s < splits; s++) {
            const f32x4_t u = *reinterpret_cast<const f32x4_t*>(ws + int64_t(s) * mn + i);
            v = f32x4_t{v[0] + u[0], v[1] + u[1], v[2] + u[2], v[3] + u[3]};
        }
        const int64_t row = i / n, col = i - row * n;
        typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<u16x4*>(y + row * ldy + col) =
            u16x4{QmmAct<XT>::out(v[0]), QmmAct<XT>::out(v[1]), QmmAct<XT>::out(v[2]), QmmAct<XT>::out(v[3])};
    } else {
        for (int64_t e = i; e < mn && e < i + 4; e++) {
            float v = ws[e];
            for (int s = 1; s < splits; s++) v += ws[int64_t(s) * mn + e];
            const int64_t row = e / n;
            y[row * ldy + (e - row * n)] = QmmAct<XT>::out(v);
        }
    }
}

// Compute units of the current device.
static int qmm_cu_count() {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) return 256;
    return v;
}

// The types of a launch: code bits, group size, scale (EQ_DTYPE_U8: MXFP4) and activation types.
struct QmmTypes {
    int bits, gs, scale_dtype, x_dtype;
    int64_t param_bytes() const { return scale_dtype == EQ_DTYPE_U8 ? 1 : 2; }
};

static bool qmm_run(int tm, int tn, const QmmTypes& t, const QmmArgs& a, int workgroups, hipStream_t st) {
    const bool pw = qmm_param_words(t.gs, a.K, a.cps, a.s, a.b);
    if (tn == 2) return qmm_run_t42(t.bits, t.gs, t.scale_dtype, t.x_dtype, pw, a, workgroups, st);
    if (tm == 2) return qmm_run_t21(t.bits, t.gs, t.scale_dtype, t.x_dtype, pw, a, workgroups, st);
    if (tm == 3) return qmm_run_t31(t.bits, t.gs, t.scale_dtype, t.x_dtype, pw, a, workgroups, st);
    return qmm_run_t41(t.bits, t.gs, t.scale_dtype, t.x_dtype, pw, a, workgroups, st);
}

// One launch (plus the split reduction): every buffer below 2^31 bytes.
static bool launch_qmm_piece(const QmmTypes& t, uint16_t* y, int ldy, const uint16_t* x, const uint32_t* w, const void* s,
                             const void* b, int M, int N, int K, bool may_split, const WsSource* src, hipStream_t st) {
    QmmArgs a{};
    a.y = y, a.x = x, a.w = w, a.s = static_cast<const uint16_t*>(s), a.b = static_cast<const uint16_t*>(b);
    a.M = M, a.N = N, a.K = K, a.ldy = ldy;
    const QmmPlan plan = qmm_plan(M, N, K, t.gs, t.bits, may_split, qmm_cu_count());
    a.mtiles = plan.mtiles, a.ntiles = plan.ntiles;
    const int tiles = a.mtiles * a.ntiles, nchunks = K / kBK;
    int splits = plan.splits;
    if (splits > 1) {
        // whole words of parameters per split, so that its windows stay 4-byte aligned
        const int unit = t.gs == 128 ? 4 : 2;
        a.cps = ((nchunks + splits - 1) / splits + unit - 1) / unit * unit;
        splits = (nchunks + a.cps - 1) / a.cps;  // no empty split
        // a fixed scratch region may hold fewer splits than planned
        const size_t per_split = size_t(M) * size_t(N) * 4u;
        if (src && splits > 1 && size_t(splits) * per_split > src->cap) {
            const int fit = int(src->cap / per_split);
            if (fit >= 2) {
                a.cps = ((nchunks + fit - 1) / fit + unit - 1) / unit * unit;
                splits = (nchunks + a.cps - 1) / a.cps;
            } else {
                splits = 1;
            }
        }
        if (splits > 1) {
            a.ws = static_cast<float*>(ws_acquire(src, size_t(splits) * per_split, st));
            if (!a.ws && !src) {
                // The library workspace cannot grow (the stream is capturing,
                // or the allocation failed).  Running unsplit would be a
                // different plan with a different summation order than the
                // same call made eagerly, so the call fails instead.
                set_error("quantized_matmul (qmm): the split-K plan needs " +
                          std::to_string(size_t(splits) * per_split) +
                          " bytes of workspace on this stream, which cannot grow while the stream is capturing "
                          "(make one call of this shape on the stream before capturing)");
                note_refusal();
                return false;
            }
            if (!a.ws) splits = 1;
        }
    }
    a.splits = splits;
    if (splits == 1) a.cps = nchunks;
    if (!qmm_run(plan.tm, plan.tn, t, a, tiles * splits, st)) return false;
    if (splits == 1) return true;
    const int64_t mn = int64_t(M) * N;
    const dim3 grid(unsigned((mn / 4 + 255) / 256 + 1)), block(256);
    const bool vec = aligned(y, 8) && N % 4 == 0 && ldy % 4 == 0;
    if (t.x_dtype == EQ_DTYPE_BF16) qmm_split_reduce<BF16T><<<grid, block, 0, st>>>(y, a.ws, mn, N, ldy, splits, vec);
    else qmm_split_reduce<F16T><<<grid, block, 0, st>>>(y, a.ws, mn, N, ldy, splits, vec);
    return true;
}

// Buffer offsets in the kernel are 32-bit: a weight matrix of 2^31 bytes or
// more runs in row pieces (multiples of the 256-column tile), an activation
// matrix that large in row pieces (multiples of the 128-row tile).
// y's row stride is ldy (N when negative); split K only when y is one whole
// piece of stride N.
static void launch_qmm_t(const QmmTypes& t, uint16_t* y, const uint16_t* x, const uint32_t* w, const void* s, const void* b,
                         int M, int N, int K, const WsSource* src, hipStream_t st, int ldy = -1) {
    if (ldy < 0) ldy = N;
    const int64_t limit = (int64_t(1) << 31) - 1;
    const int64_t row_bytes = int64_t(K) * t.bits / 8;
    const int64_t G = K / t.gs, PB = t.param_bytes();
    int64_t n_piece = limit / row_bytes / kBN * kBN;
    int64_t m_piece = limit / (int64_t(K) * 2) / kBM * kBM;
    n_piece = n_piece < kBN ? kBN : n_piece;
    m_piece = m_piece < kBM ? kBM : m_piece;
    const bool whole = n_piece >= N && m_piece >= M;
    for (int64_t m0 = 0; m0 < M; m0 += m_piece) {
        const int mc = int(M - m0 < m_piece ? M - m0 : m_piece);
        for (int64_t n0 = 0; n0 < N; n0 += n_piece) {
            const int nc = int(N - n0 < n_piece ? N - n0 : n_piece);
            const char* sp = static_cast<const char*>(s) + n0 * G * PB;
            const char* bp = b ? static_cast<const char*>(b) + n0 * G * PB : nullptr;
            // (only a whole problem splits K, so a refusal comes before any launch)
            if (!launch_qmm_piece(t, y + m0 * ldy + n0, ldy, x + m0 * K, w + n0 * (row_bytes / 4), sp, bp, mc, nc, K, whole, src,
                                  st))
                return;
        }
    }
}

// Group sizes with kernel variants.
static bool qmm_gs_ok(int gs) { return gs == 16 || gs == 32 || gs == 64 || gs == 128; }

// ------------------------------------------------------- grouped (experts)

// First index i of a[0, n) with a[i] >= v (a sorted ascending; for unsorted
// input the result is still in [0, n]).
__device__ __forceinline__ int lower_bound_i32(const int32_t* __restrict__ a, int n, int v) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Prepares a grouped launch.  Workgroup 0: sorted expert indices -> the tile
// list; expert e owns rows [lower_bound(e), lower_bound(e + 1)) and takes
// ceil(rows / bm) entries {e, first, rows, bm t}, experts in passes of 1024
// with a block scan of the entry counts; entries at or past `cap` are dropped,
// and out[cap] receives how many there are.  The indices are searched
// in LDS where they fit (from memory a search is a chain of a dozen trips).
// The other workgroups meanwhile clear y (rows of no expert stay zero), n bf16
// values, n a multiple of 4, y 8-byte aligned.
constexpr int kGroupIds = 8192;
__global__ __launch_bounds__(1024) void qmm_group_prepare(int4* __restrict__ out, const int32_t* __restrict__ rhs,
                                                          int batch, int experts, int cap, int bm,
                                                          uint16_t* __restrict__ y, int64_t n) {
    if (blockIdx.x > 0) {
        const int64_t stride = int64_t(gridDim.x - 1) * 4096;
        for (int64_t i = (int64_t(blockIdx.x - 1) * 1024 + threadIdx.x) * 4; i < n; i += stride)
            *reinterpret_cast<uint2*>(y + i) = make_uint2(0, 0);
        return;
    }
    __shared__ int32_t ids[kGroupIds];
    __shared__ int scan[1024];
    __shared__ int carry;
    const int tid = threadIdx.x;
    const bool local = batch <= kGroupIds;
    if (local)
        for (int i = tid; i < batch; i += 1024) ids[i] = rhs[i];
    if (tid == 0) carry = 0;
    __syncthreads();
    const int32_t* search = local ? ids : rhs;
    for (int e0 = 0; e0 < experts; e0 += 1024) {
        const int e = e0 + tid;
        int first = 0, rows = 0;
        if (e < experts) {
            first = lower_bound_i32(search, batch, e);
            const int end = lower_bound_i32(search, batch, e + 1);
            rows = end > first ? end - first : 0;
        }
        const int nt = (rows + bm - 1) / bm;
        scan[tid] = nt;
        __syncthreads();
        for (int o = 1; o < 1024 && o < experts - e0; o <<= 1) {  // inclusive scan
            const int v = tid >= o ? scan[tid - o] : 0;
            __syncthreads();
            scan[tid] += v;
            __syncthreads();
        }
        const int base = carry + scan[tid] - nt;
        for (int t = 0; t < nt; t++)
            if (base + t < cap) out[base + t] = make_int4(e, first, rows, t * bm);
        const int last = experts - e0 < 1024 ? experts - e0 - 1 : 1023;
        __syncthreads();
        if (tid == last) carry += scan[last];
        __syncthreads();
    }
    if (tid == 0) out[cap] = make_int4(carry < cap ? carry : cap, 0, 0, 0);
}

// xg[b] = x[lhs[b]] (K bf16 per row, 16-byte copies); an out-of-range index
// gives a zero row.  One workgroup per row.
__global__ __launch_bounds__(256) void qmm_gather_rows(uint16_t* __restrict__ xg, const uint16_t* __restrict__ x,
                                                       const int32_t* __restrict__ lhs, int64_t x_batches, int K) {
    const int64_t b = blockIdx.x;
    const int64_t src = lhs ? int64_t(lhs[b]) : (x_batches == 1 ? 0 : b);
    uint4* dst = reinterpret_cast<uint4*>(xg + b * K);
    const bool ok = src >= 0 && src < x_batches;
    const uint4* from = reinterpret_cast<const uint4*>(x + (ok ? src : 0) * K);
    for (int i = threadIdx.x; i < K / 8; i += 256) dst[i] = ok ? from[i] : make_uint4(0, 0, 0, 0);
}

static bool launch_qmm_grouped_t(const QmmTypes& t, uint16_t* y, const uint16_t* x, const uint32_t* w, const void* s, const void* b,
                                 const int32_t* lhs, const int32_t* rhs, int batch, int64_t x_batches, int experts,
                                 int N, int K, hipStream_t st, const WsSource* src = nullptr) {
    // Tiles by the mean number of rows per expert: 64 x 128 up to 64 rows (two such
    // workgroups of 4-bit codes share a CU), 128 x 256 above; with 8-bit codes (one
    // to a CU) and at group size 16 (more work per code) up to 40.  Time of the 64
    // x 128 tiles over that of the 128 x 256 ones, geometric mean of six banks of 8 to
    // 128 experts: 4-bit group 64 at 40 / 56 / 64 / 80 rows 0.75 / 0.90 / 0.98 /
    // 1.07, group 32 0.78 / 0.94 / 1.02 at 64, group 16 0.78 / 1.01 / 1.11; 8-bit
    // group 64 at 40 / 48 / 64 rows 0.87 / 1.09 / 1.19.  Routes on few of the experts
    // fill the tiles they take, at these means and above (128 experts of 768 x 2048,
    // 16 rows in the mean, all on two: 20 / 33 us; 64 rows: 47 / 42).
    const int mean = batch / (experts > 0 ? experts : 1);
    const bool small = mean <= (t.bits == 4 && t.gs >= 32 ? 64 : 40);
    const int tm = small ? 2 : 4, tn = small ? 1 : 2, bm = 32 * tm;
    const int cap = experts + (batch + bm - 1) / bm;  // sum over experts of ceil(rows / bm)
    // one launch with 32-bit offsets: each expert's codes below 2^31 bytes, and
    // the rows of x, which are otherwise gathered first
    if (int64_t(N) * K * t.bits / 8 >= (int64_t(1) << 31) || int64_t(batch) * K * 2 >= (int64_t(1) << 31)) return false;
    const bool direct = x_batches * int64_t(K) * 2 < (int64_t(1) << 31);
    const size_t xg_bytes = direct ? 0 : (size_t(batch) * size_t(K) * 2u + 255u) & ~size_t(255);
    void* ws = ws_acquire(src, xg_bytes + size_t(cap + 1) * sizeof(int4), st);
    if (!ws) return false;
    uint16_t* xg = reinterpret_cast<uint16_t*>(ws);
    int4* list = reinterpret_cast<int4*>(reinterpret_cast<char*>(ws) + xg_bytes);
    const int64_t yn = int64_t(batch) * N;
    qmm_group_prepare<<<dim3(1 + unsigned(yn / 4096 < 1024 ? yn / 4096 + 1 : 1024)), dim3(1024), 0, st>>>(
        list, rhs, batch, experts, cap, bm, y, yn);
    if (!direct) qmm_gather_rows<<<dim3(unsigned(batch)), dim3(256), 0, st>>>(xg, x, lhs, x_batches, K);
    QmmArgs a{};
    a.y = y, a.x = direct ? x : xg, a.w = w, a.s = static_cast<const uint16_t*>(s), a.b = static_cast<const uint16_t*>(b);
    a.M = batch, a.N = N, a.K = K, a.ldy = N;
    a.mtiles = cap, a.ntiles = (N + 128 * tn - 1) / (128 * tn), a.splits = 1, a.cps = K / kBK;
    a.groups = list;
    a.lhs = direct ? lhs : nullptr, a.x_rows = direct ? int(x_batches) : batch;
    return qmm_run(tm, tn, t, a, (a.mtiles * a.ntiles + 7) / 8 * 8, st);  // (an eighth for each XCD, rounded up)
}

bool launch_qmm_grouped(int bits, int gs, int scale_dtype, uint16_t* y, const uint16_t* x, const uint32_t* w,
                        const void* s, const void* b, const int32_t* lhs, const int32_t* rhs, int batch,
                        int64_t x_batches, int experts, int N, int K, hipStream_t st, const WsSource* src) {
    if ((bits != 4 && bits != 8) || !qmm_gs_ok(gs) || (scale_dtype != EQ_DTYPE_BF16 && scale_dtype != EQ_DTYPE_F16))
        return false;
    return launch_qmm_grouped_t({bits, gs, scale_dtype, EQ_DTYPE_BF16}, y, x, w, s, b, lhs, rhs, batch, x_batches, experts,
                                N, K, st, src);
}

bool launch_qmm_mfma_mxfp4(uint16_t* y, const uint16_t* x, const uint32_t* w, const uint8_t* s, int M, int N, int K,
                           const WsSource* ws, hipStream_t st) {
    launch_qmm_t({4, 32, EQ_DTYPE_U8, EQ_DTYPE_BF16}, y, x, w, s, nullptr, M, N, K, ws, st);
    return true;
}

bool launch_qmm_grouped_mxfp4(uint16_t* y, const uint16_t* x, const uint32_t* w, const uint8_t* s,
                              const int32_t* lhs, const int32_t* rhs, int batch, int64_t x_batches, int experts, int N,
                              int K, hipStream_t st) {
    return launch_qmm_grouped_t({4, 32, EQ_DTYPE_U8, EQ_DTYPE_BF16}, y, x, w, s, nullptr, lhs, rhs, batch, x_batches,
                                experts, N, K, st);
}

// ------------------------------------------- prefill at 2, 3, 5 and 6 bits
//
// The codes of these widths are an LSB-first bit stream (a 32-code unit of a
// row is exactly BITS words).  For M > 16 they are re-packed, a slice of
// weight rows at a time, to one byte per code in the stream's workspace and
// multiplied by the 8-bit matrix-core kernel with the same scales and biases
// and group size: the code values, and so the products, are unchanged.

// One thread per 32-code unit: BITS words in, 8 words (32 byte codes) out.
template <int BITS>
__global__ __launch_bounds__(256) void qmm_codes_to_bytes(const uint32_t* __restrict__ w, uint4* __restrict__ out,
                                                          int64_t units) {
    const int64_t u = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (u >= units) return;
    uint32_t in[BITS];
#pragma unroll
    for (int i = 0; i < BITS; i++) in[i] = w[u * BITS + i];
    uint32_t o[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
        uint32_t v = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int bit = (4 * q + e) * BITS, wd = bit >> 5, sh = bit & 31;
            uint32_t c = in[wd] >> sh;
            if (sh + BITS > 32) c |= in[wd + 1] << (32 - sh);
            v |= (c & ((1u << BITS) - 1u)) << (8 * e);
        }
        o[q] = v;
    }
    out[2 * u] = make_uint4(o[0], o[1], o[2], o[3]);
    out[2 * u + 1] = make_uint4(o[4], o[5], o[6], o[7]);
}

static bool launch_qmm_odd_t(const QmmTypes& t, uint16_t* y, const uint16_t* x, const uint32_t* w, const void* s,
                             const void* b, int M, int N, int K, const WsSource* src, hipStream_t st, int ldy = -1) {
    const int bits = t.bits, gs = t.gs;
    const QmmTypes bytes{8, gs, t.scale_dtype, t.x_dtype};
    if (ldy < 0) ldy = N;
    // rows per slice: their byte codes within 64 MiB, a multiple of the 256-column tile
    int64_t nc = (int64_t(64) << 20) / K / kBN * kBN;
    nc = nc < kBN ? kBN : nc;
    nc = nc > N ? N : nc;
    const size_t code_bytes = (size_t(nc) * size_t(K) + 255) & ~size_t(255);
    // room after the codes for the split-K partials of a slice the planner would split
    const int splits = qmm_plan(M, int(nc), K, gs, 8, true, qmm_cu_count()).splits;
    const size_t part_bytes = splits > 1 ? size_t(splits) * size_t(M) * size_t(nc) * 4u : 0;
    size_t want = code_bytes + part_bytes;
    char* base = static_cast<char*>(ws_acquire(src, want, st));
    if (!base && !src) {
        // the library workspace cannot grow (capture): fail rather than run
        // another plan than the same call made eagerly
        set_error("quantized_matmul (qmm, " + std::to_string(bits) + "-bit): the plan needs " + std::to_string(want) +
                  " bytes of workspace on this stream, which cannot grow while the stream is capturing "
                  "(make one call of this shape on the stream before capturing)");
        note_refusal();
        return true;
    }
    if (!base) base = static_cast<char*>(ws_acquire(src, want = code_bytes, st));
    if (!base) return false;
    const size_t cap = src ? src->cap : want;
    WsSource rest{base + code_bytes, cap > code_bytes ? cap - code_bytes : 0, nullptr};
    const int64_t G = K / gs;
    constexpr int64_t PB = 2;
    for (int64_t n0 = 0; n0 < N; n0 += nc) {
        const int ncs = int(N - n0 < nc ? N - n0 : nc);
        const int64_t units = int64_t(ncs) * (K / 32);
        const dim3 grid(unsigned((units + 255) / 256));
        const uint32_t* wr = w + n0 * (int64_t(K) * bits / 32);
        uint4* codes = reinterpret_cast<uint4*>(base);
        switch (bits) {
        case 2: qmm_codes_to_bytes<2><<<grid, 256, 0, st>>>(wr, codes, units); break;
        case 3: qmm_codes_to_bytes<3><<<grid, 256, 0, st>>>(wr, codes, units); break;
        case 5: qmm_codes_to_bytes<5><<<grid, 256, 0, st>>>(wr, codes, units); break;
        default: qmm_codes_to_bytes<6><<<grid, 256, 0, st>>>(wr, codes, units); break;
        }
        const char* sp = static_cast<const char*>(s) + n0 * G * PB;
        const char* bp = b ? static_cast<const char*>(b) + n0 * G * PB : nullptr;
        const uint32_t* w8 = reinterpret_cast<const uint32_t*>(base);
        const WsSource* parts = rest.cap > 0 ? &rest : nullptr;
        if (!parts) {
            // no room for partials: a fixed region of exactly the codes, no split
            static const WsSource none{nullptr, 0, nullptr};
            parts = &none;
        }
        launch_qmm_t(bytes, y + n0, x, w8, sp, bp, M, ncs, K, parts, st, ldy);
    }
    return true;
}

bool launch_qmm_mfma(int bits, int gs, int scale_dtype, uint16_t* y, const uint16_t* x, const uint32_t* w,
                     const void* s, const void* b, int M, int N, int K, const WsSource* ws, hipStream_t st,
                     int ldy, int x_dtype) {
    if (!qmm_gs_ok(gs) || (scale_dtype != EQ_DTYPE_BF16 && scale_dtype != EQ_DTYPE_F16) ||
        (x_dtype != EQ_DTYPE_BF16 && x_dtype != EQ_DTYPE_F16))
        return false;
    const QmmTypes t{bits, gs, scale_dtype, x_dtype};
    if (bits == 4 || bits == 8) {
        launch_qmm_t(t, y, x, w, s, b, M, N, K, ws, st, ldy);
        return true;
    }
    if (bits == 2 || bits == 3 || bits == 5 || bits == 6)
        return launch_qmm_odd_t(t, y, x, w, s, b, M, N, K, ws, st, ldy);
    return false;
}

}  // namespace eq

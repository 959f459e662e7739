// fp16 linears of the Llama family (w_qkv / wo / w1w3 / w2 of an unquantised checkpoint, lm_head) on the kernels of gemm_stream.h: the weight stream for
// decode-sized forwards, tiles by DMA for prompts.
//
// Replaces: LlamaLinear::Forward -> gemm::Gemm::Run for fp16 weights (src/turbomind/models/llama/LlamaLinear.cu:140-216), the gated-SiLU epilogue
// (kernels/gemm/epilogue.h:159-176,428-446).  Same arithmetic as gemm_kernel<WT = 1> (gemm_w4a16.hip): fp32 accumulation, one rounding of the result;
// the image is the one linear_weight_prepare_f16 makes ([k / 128][n / 16][4] blocks of one KB).
//
// Weights from HBM, MI355X, here | gemm_kernel: 8 rows (2048, 4096) 7.2 | 13.0 us, (8192, 2048) 14.1 | 43.7, (2048, 16384) gated 15.7 | 17.2; 64 rows (14336,
// 4096) 33 | 101; 2664 rows (2048, 16384) gated 215 | 501; 8192 rows (4096, 28672) gated 1702 | 5390 us (1.13 PFLOP/s), (14336, 4096) 810 | 2159 (1.19).
#include "gemm_rows.h"
#include "tm_kernels.h"
#include <algorithm>

namespace tmk {

struct F16Item {
    int64_t x_off, w_off;
    int     M;
};

struct F16Epi {
    int gated;  // columns alternate (gate_j, up_j): out[m][j] = silu(acc[m][2 j]) * acc[m][2 j + 1]
    int vec;    // rows of y start on 8 bytes

    static constexpr bool kPairs = false, kTileRuns = false;
    static constexpr int  kReads = 0;
    __device__ __forceinline__ const int* row_offsets() const
    {
        return nullptr;
    }
    __device__ __forceinline__ int items() const
    {
        return 1;
    }
    __device__ __forceinline__ F16Item item(int, int M, int) const
    {
        return {0, 0, M};
    }
    __device__ __forceinline__ unsigned touch(const StreamArgs&, const F16Item&, int, int) const  // (nothing is read)
    {
        return 0;
    }
    template<int NT>
    __device__ __forceinline__ void rows(const StreamArgs& a, const F16Item&, int m, int n, const floatx4 (&acc)[NT]) const
    {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int c = n + 16 * j;
            if (c >= a.N) {  // (N is a multiple of 16)
                continue;
            }
            const floatx4 v = acc[j];
            if (gated) {
                const float s0 = silu_f32(v[0]);
                const float s1 = silu_f32(v[2]);
                half_t*     y  = (half_t*)a.y + (size_t)m * a.ldy + (c >> 1);
                if (vec) {
                    *(half2_t*)y = half2_t{(half_t)(s0 * v[1]), (half_t)(s1 * v[3])};
                }
                else {
                    y[0] = (half_t)(s0 * v[1]), y[1] = (half_t)(s1 * v[3]);
                }
            }
            else {
                half_t* y = (half_t*)a.y + (size_t)m * a.ldy + c;
                if (vec) {
                    *(half4_t*)y = half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
                }
                else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        y[e] = (half_t)v[e];
                    }
                }
            }
        }
    }
};

// The same for a decode step's [q | k | v] product: queries and keys are rotated, keys and values go to the cache (kv_rope_store_kernel's arithmetic: the product's fp16
// rounding first, then fp16 multiplications and additions on pairs), which a launch behind the product did.  8 sequences, 16 + 2 x 8 heads of 128, (2048, 4096): 5.4 +
// 3.0 us, now 5.8
struct F16EpiKv: F16Epi {
    F16KvSink kv;

    template<int NT>
    __device__ __forceinline__ void rows(const StreamArgs& a, const F16Item&, int m, int n, const floatx4 (&acc)[NT]) const
    {
        const int      pos = kv.k_len[m] - 1;
        const KvLayout L   = kv.cache.layout;
        const int      blk = pos / L.block_len, ti = pos - blk * L.block_len;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int c = n + 16 * j, head = c >> 7, d = c & 127, kh = head - kv.q_heads;
            if (c >= a.N) {
                continue;
            }
            half4_t h = {(half_t)acc[j][0], (half_t)acc[j][1], (half_t)acc[j][2], (half_t)acc[j][3]};
            if (kh < L.kv_heads && kv.cos_sin) {
                const half4_t cs = *(const half4_t*)(kv.cos_sin + (size_t)min(pos, kv.max_pos - 1) * 64 + (d >> 1));
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    const half_t x0 = h[e], x1 = h[e + 1];
                    const half_t a0 = cs[e] * x0, a1 = cs[e + 1] * x1, b0 = cs[e] * x1, b1 = cs[e + 1] * x0;
                    h[e]     = a0 - a1;
                    h[e + 1] = b0 + b1;
                }
            }
            if (kh < 0) {
                *(half4_t*)((half_t*)a.y + (size_t)m * a.ldy + c) = h;
                continue;
            }
            char* block = global_ptr(kv.cache.block_ptrs[kv.cache.cu_block_nums[m] + blk]) + kv.cache.layer_offset;
            *(half4_t*)(block + (kh < L.kv_heads ? L.k_data(kh, ti) : L.v_data(kh - L.kv_heads, ti)) + d * 2) = h;
        }
    }
};

// The same for a product that closes a residual block: y += h(acc), in fp16 (residual_rmsnorm's addition)
struct F16EpiAdd: F16Epi {
    __device__ __forceinline__ unsigned touch(const StreamArgs& a, const F16Item&, int m, int n) const
    {
        return ((const unsigned short*)a.y)[(size_t)m * a.ldy + n];
    }
    template<int NT>
    __device__ __forceinline__ void rows(const StreamArgs& a, const F16Item&, int m, int n, const floatx4 (&acc)[NT]) const
    {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int c = n + 16 * j;
            if (c < a.N) {
                half4_t* y = (half4_t*)((half_t*)a.y + (size_t)m * a.ldy + c);
                *y         = *y + half4_t{(half_t)acc[j][0], (half_t)acc[j][1], (half_t)acc[j][2], (half_t)acc[j][3]};
            }
        }
    }
};

// Where gemm_kernel is still the better one: its workgroups of 64 rows x 128 columns take the weights straight into registers and read x half as often as 64
// columns do, so it wins where about one round of them keeps the CUs busy.  us, gemm_kernel | here, weights from HBM:
//   up to 64 rows, 193 ... 256 workgroups: (K, N) = (4096, 28672) gated 8 rows 35.4 | 34.7, 32 rows 35.5 | 38.5, 64 rows 40 | 44, (5120, 27648) gated 8 rows
//     43.6 | 44.1, 64 rows 48 | 55, (4096, 32000) 64 rows 42 | 47; not (4096, 24576) 32 rows 34 | 32, (4096, 20480) 64 rows 37 | 31, (2048, 16384) gated 21 | 15,
//     nor (4096, 36864) 32 rows 65 | 55, (4096, 8192) gated 27 | 16
//   41 ... 64 rows of wider outputs, where their last round is at least three quarters full or one of many: K = 4096, 64 rows, 256 workgroups 42.6 | 46.1, 448 77 | 87, 512
//     84 | 93, 723 127 | 137, 1002 179 | 192, 1188 218 | 232; not 288 68 | 58, 384 73 | 68, 576 113 | 111, nor K = 2048 640 63 | 61; nor 32 rows, 384 71 | 62, 1002 170 | 166
//   more rows, one round of them where 64 x 64 tiles take two: (2048, 16384) gated, 128 rows 20.9 | 26, (4096, 6144) 192 rows 30 | 42, (4096, 4096) 320 rows 29 |
//     39, (14336, 4096) 320 rows 92 | 130; not where one round of tiles is enough, (4096, 4096) 256 rows 29 | 23, nor where it takes two, 640 rows 58 | 45
bool f16_stream_supported(const LinearWeight& w, int M)
{
    const int  rb = (M + 63) / 64, t64 = (w.N + 63) / 64 * rb, t128 = (w.N + 127) / 128 * rb;
    const bool full    = t128 % 256 == 0 || t128 % 256 >= 192 || t128 > 1024;
    const bool general = M <= 64 ? t128 > 192 && (M > 40 ? full : t128 <= 256) : t64 > 256 && t128 <= 256;
    return w.type == 1 && w.packed && (size_t)w.K * w.N * 2 < ((size_t)1 << 31) && !general;  // (byte offsets inside the image are 32 bits)
}

int f16_stream_splits(const LinearWeight& w, int M)
{
    const StreamPlan p = stream_plan(w.K / 32, w.N, M, 1, false, 2, false, ~(size_t)0, 1 << 30, 0, true);
    return p.skinny ? p.splits : 1;
}

template<int MT, class Epi>
static int launch_skinny(const StreamArgs& a, const Epi& epi, const StreamPlan& p, hipStream_t st)
{
    const dim3 grid((a.tiles + p.cw - 1) / p.cw, a.row_blocks, p.splits);
    if (p.narrow) {
        if (MT <= 2 && stream_narrow_waves(a) == 16) {
            stream_narrow_kernel<half_t, Epi, MT, 1, MT <= 2 ? 16 : 8><<<dim3(a.tiles, a.row_blocks), 1024, 0, st>>>(a, epi);
        }
        else {
            stream_narrow_kernel<half_t, Epi, MT, 1, 8><<<dim3(a.tiles, a.row_blocks), 512, 0, st>>>(a, epi);
        }
    }
    else if (p.cw == 6) {
        stream_skinny_kernel<half_t, Epi, MT, 1, 6, 1><<<grid, 384, 0, st>>>(a, epi);
    }
    else {
        stream_skinny_kernel<half_t, Epi, MT, 1, 4, 1><<<grid, 256, 0, st>>>(a, epi);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<class K>
static int launch_tiles(K kernel, const StreamArgs& a, const F16Epi& epi, int bm, int bn, hipStream_t st)
{
    const int lds = stream_tile_bufs(bm, bn) * (bm + bn) * 64;
    if (const int rc = ensure_dynamic_lds((const void*)kernel, lds)) {
        return rc;
    }
    kernel<<<dim3((unsigned)((a.M + bm - 1) / bm) * (unsigned)(((a.col1 ? a.col1 : a.tiles * 16) - a.col0 + bn - 1) / bn)), 256, lds, st>>>(a, epi);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

static int launch_tile_shape(const StreamArgs& a, const F16Epi& epi, int tile, hipStream_t st)
{
    return tile == 0 ? launch_tiles(stream_tile256_kernel<half_t, F16Epi>, a, epi, 256, 256, st) :
           tile == 1 ? launch_tiles(stream_tile_kernel<half_t, F16Epi, 256, 128, 2, 2>, a, epi, 256, 128, st) :
           tile == 2 ? launch_tiles(stream_tile_kernel<half_t, F16Epi, 128, 128, 2, 2>, a, epi, 128, 128, st) :
                       launch_tiles(stream_tile_kernel<half_t, F16Epi, 64, 64, 2, 2>, a, epi, 64, 64, st);
}

// splits: slices of k the caller's workspace holds slabs for (1: none).  With slices, fp32 slabs [slices][M][N] are left in the workspace and *slabs says
// how many (defer, or no arrival counters), or they meet inside the launch (tickets)
int launch_f16_stream(const LinearWeight& w, const half_t* x, int ldx, half_t* y, int ldy, int M, bool gated, int splits, float* workspace,
                      unsigned* tickets, int ticket_count, bool defer, int* slabs, hipStream_t st, const F16KvSink* kv, bool* kv_done,
                      bool add)
{
    TM_REQUIRE(f16_stream_supported(w, M), "fp16 linear: image");
    const bool       slice = splits > 1 && workspace;
    const StreamPlan p     = stream_plan(w.K / 32, w.N, M, 1, false, 2, false, slice ? ~(size_t)0 : 0, slice ? 1 << 30 : 0, 0, true, 0, true);
    StreamArgs       a{};
    a.x = (const char*)x, a.ldx = (int64_t)ldx * 2;
    a.w = (const char*)w.packed, a.tiles = w.N / 16, a.steps = w.K / 32;
    a.w_tile = 4096, a.w_quad = (int64_t)a.tiles * 4096;
    a.y = y, a.ldy = ldy, a.M = M, a.N = w.N;
    const F16Epi epi{gated ? 1 : 0, gated ? (ldy % 2 == 0 && (uintptr_t)y % 4 == 0) : (ldy % 4 == 0 && (uintptr_t)y % 8 == 0)};
    *slabs = 1;
    if (p.skinny) {
        TM_REQUIRE(p.splits <= std::max(1, splits), "fp16 linear: slices of k");
        a.split_steps = p.split_steps;
        a.row_blocks  = p.row_blocks;
        if (p.splits > 1) {
            a.slabs   = workspace;
            a.tickets = defer || (a.tiles + p.cw - 1) / p.cw * p.row_blocks > ticket_count ? nullptr : tickets;
            *slabs    = a.tickets ? 1 : p.splits;
        }
        // (results that leave as slabs are rounded, rotated and stored by the launches behind this one)
        if (kv && !gated && *slabs == 1 && ldy % 4 == 0 && (uintptr_t)y % 8 == 0) {
            const F16EpiKv ek{epi, *kv};
            *kv_done = true;
            return p.mt == 1 ? launch_skinny<1>(a, ek, p, st) : p.mt == 2 ? launch_skinny<2>(a, ek, p, st) : launch_skinny<4>(a, ek, p, st);
        }
        if (add) {
            TM_REQUIRE(*slabs == 1 && !gated && ldy % 4 == 0 && (uintptr_t)y % 8 == 0, "fp16 linear: a residual addition");
            const F16EpiAdd ea{epi};
            return p.mt == 1 ? launch_skinny<1>(a, ea, p, st) : p.mt == 2 ? launch_skinny<2>(a, ea, p, st) : launch_skinny<4>(a, ea, p, st);
        }
        return p.mt == 1 ? launch_skinny<1>(a, epi, p, st) : p.mt == 2 ? launch_skinny<2>(a, epi, p, st) : launch_skinny<4>(a, epi, p, st);
    }
    TM_REQUIRE(!add, "fp16 linear: a residual addition");
    if (p.cut > 0) {
        StreamArgs rest = a;
        rest.col0       = p.cut;
        a.col1          = p.cut;
        if (const int rc = launch_tile_shape(a, epi, p.tile, st)) {
            return rc;
        }
        return launch_tile_shape(rest, epi, p.tile2, st);
    }
    return launch_tile_shape(a, epi, p.tile, st);
}

// ---- few rows that come with their norm ------------------------------------------------------------------------------------------------
template<int RPW, int P, int CW, int KP, int R, class Epi>
static int launch_rows(const StreamArgs& a, const Epi& epi, const half_t* resid, const half_t* norm_w, float eps, int team, hipStream_t st)
{
    const auto kernel = stream_rows_kernel<half_t, Epi, NormRows<RPW, P>, CW, KP, R>;
    const int  lds    = stream_rows_lds(a.M, a.steps, CW, KP);
    if (const int rc = ensure_dynamic_lds((const void*)kernel, lds)) {
        return rc;
    }
    kernel<<<dim3((a.tiles + CW - 1) / CW), CW * KP * 64, lds, st>>>(a, epi, NormRows<RPW, P>{resid, norm_w, eps, team});
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

bool f16_norm_rows_supported(const LinearWeight& w, int M)
{
    return w.type == 1 && w.packed && (size_t)w.K * w.N * 2 < ((size_t)1 << 31) && w.K % 512 == 0 && M >= 1 && (M <= 8 ? w.K <= 4096 : M <= 16 && w.K <= 2048);
}

// Beyond 512 column tiles a workgroup takes four, whatever their number: where the fullest CU then streams longer than memory takes for all of them, and than a plan of four or six
// tiles would leave it, by more than a norm launch is worth, the launch stays.  us a layer, launch | norm in the product, 8 rows (12 and 16 alike): (2048, 16896) 44.8 | 47.3, (2048, 22016)
// 48.7 | 49.6, (2560, 19456) 53.2 | 56.8, (1536, 17920) 41.4 | 43.2, (4096, 19456) 76.3 | 82.0; (2048, 24576) 50.9 | 50.8, one row 50.5 | 48.3; (2048, 16384) 43.6 | 42.2
bool f16_norm_rows_pays(const LinearWeight& w)
{
    const int tiles = w.N / 16;
    auto      us    = [&](int cw) { return ((tiles + cw - 1) / cw + 255) / 256 * cw * (w.K * 32 / 33e3); };  // a CU's load path: 33 KB a microsecond
    return tiles <= 512 || us(4) <= std::max(tiles * (w.K * 32 / 6e6), std::min(us(4), us(6))) + 0.75;
}

template<int CW, int KP, int R, class Epi>
static int launch_rows_of(const StreamArgs& a, const Epi& epi, const half_t* resid, const half_t* norm_w, float eps, hipStream_t st)
{
    const int waves = CW * KP;
    int       teams = 1;
    while (teams < waves && teams < a.M) {
        teams *= 2;
    }
    const int team = waves / teams, p = (a.steps / 16 + team - 1) / team, rpw = (a.M + teams - 1) / teams;
    TM_REQUIRE(rpw == 1 ? p <= 8 : rpw == 2 && p <= 4, "fp16 linear with its norm: rows");
    return rpw == 2 ? launch_rows<2, 4, CW, KP, R>(a, epi, resid, norm_w, eps, team, st) :
           p <= 1   ? launch_rows<1, 1, CW, KP, R>(a, epi, resid, norm_w, eps, team, st) :
           p <= 2   ? launch_rows<1, 2, CW, KP, R>(a, epi, resid, norm_w, eps, team, st) :
           p <= 4   ? launch_rows<1, 4, CW, KP, R>(a, epi, resid, norm_w, eps, team, st) :
                      launch_rows<1, 8, CW, KP, R>(a, epi, resid, norm_w, eps, team, st);
}

// us with the norm in the product | as a launch of its own ahead of the better of the other kernels (graph replays, weights from HBM): K = 2048, 8 rows, N = 2048 6.4 |
// 8.5, 4096 7.0 | 9.1, 6144 8.6 | 11.2, 10240 11.3 | 12.7, 16384 13.7 | 15.5, 28672 21.3 | 22.8; one row, 16384 13.1 | 14.8; 16 rows, 4096 8.1 | 9.8, 16384 14.8 | 15.7;
// K = 1024, 8 rows, 4096 6.2 | 7.7; K = 4096, 8 rows, 4096 10.5 | 11.4, 16384 24.1 | 24.3; one row 22.5 | 24.4.  One column tile a workgroup is best while one round of them
// fills the CUs (8 rows, K = 2048, N = 4096: 7.0, two tiles 8.2), two up to 512 tiles (N = 8192: 10.1 and 9.3, four 10.8); beyond, four waves that
// take a column tile each where their rows leave them time for it (one row, N = 16384: 13.1, eight waves 13.6; 16 rows: 15.6 and 14.8)
template<class Epi>
static int launch_norm_rows(const StreamArgs& a, const Epi& epi, const half_t* resid, const half_t* norm_w, float eps, hipStream_t st)
{
    if (a.tiles <= 256) {
        return launch_rows_of<1, 8, 8>(a, epi, resid, norm_w, eps, st);
    }
    if (a.tiles <= 512) {
        return launch_rows_of<2, 4, 8>(a, epi, resid, norm_w, eps, st);
    }
    return a.M <= 4 ? launch_rows_of<4, 1, 16>(a, epi, resid, norm_w, eps, st) : launch_rows_of<4, 2, 8>(a, epi, resid, norm_w, eps, st);
}

int launch_f16_norm_rows(const LinearWeight& w, const half_t* resid, const half_t* norm_w, float eps, half_t* y, int ldy, int M, bool gated, hipStream_t st,
                         const F16KvSink* kv)
{
    TM_REQUIRE(f16_norm_rows_supported(w, M) && resid && norm_w && y, "fp16 linear with its norm");
    TM_REQUIRE(!kv || (!gated && ldy % 4 == 0 && (uintptr_t)y % 8 == 0), "fp16 linear with its norm: cache store");
    StreamArgs a{};
    a.w = (const char*)w.packed, a.tiles = w.N / 16, a.steps = w.K / 32;
    a.w_tile = 4096, a.w_quad = (int64_t)a.tiles * 4096;
    a.y = y, a.ldy = ldy, a.M = M, a.N = w.N;
    const F16Epi epi{gated ? 1 : 0, gated ? (ldy % 2 == 0 && (uintptr_t)y % 4 == 0) : (ldy % 4 == 0 && (uintptr_t)y % 8 == 0)};
    return kv ? launch_norm_rows(a, F16EpiKv{epi, *kv}, resid, norm_w, eps, st) : launch_norm_rows(a, epi, resid, norm_w, eps, st);
}

void stream_plan_report(int kind, int K, int N, int M, bool scratch, int* plan)
{
    const int items = kind >> 8 & 0xfff, item_rows = kind >> 20;
    kind &= 0xff;
    LinearWeight w{};
    w.type = 1, w.K = K, w.N = N, w.packed = &w;  // (as loaded)
    if (kind == 2 && !f16_stream_supported(w, M)) {
        std::fill(plan, plan + 5, 0);
        return;
    }
    const size_t     ws = scratch ? (kind == 2 ? ~(size_t)0 : kStreamWsBytes) : 0;
    const int        tickets = scratch ? (kind == 2 ? 1 << 30 : kStreamTickets) : 0;
    const StreamPlan p = kind == 2 ? stream_plan(K / 32, N, M, 1, false, 2, false, ws, tickets, 0, true, 0, true) :
                                     stream_plan((K + 31) / 32, (N + 127) / 128 * 128, M, std::max(items, 1), items > 0, kind == 1 ? 4 : 2, false, ws, tickets, 0, false,
                                                 item_rows, true);
    const int out[5] = {p.skinny ? (p.narrow ? 1 : 2) : 3 + p.tile, p.skinny ? (p.narrow ? 1 : p.cw) : 0, p.skinny ? p.mt : 0, p.skinny ? p.splits : 1, p.skinny ? 0 : p.cut};
    std::copy(out, out + 5, plan);
}

}  // namespace tmk

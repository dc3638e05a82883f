// block_linear.hip -- the linear layers of many rows (prompts, and decode steps of more
// than 32 sequences) as tiled matrix-core products with the operations after each layer
// fused in: q|k|v + bias + rotary + the K/V rows' place in the paged pool, projection +
// residual, gate|up + SwiGLU.  The reference runs each of these as cuBLAS GEMMs followed
// by one kernel per elementwise op (qwen_serve.cu:90-124, qwen_kernels.cu:46-122).
//
// y[M, N] = A[M, K] W[N, K]^T, fp16 operands, fp32 accumulation.  A workgroup computes a
// BM x BN tile with KG groups of four waves; group g takes the 64-wide k blocks g, g + KG,
// ..., and the groups are summed through LDS at the end (a 700-row layer has too few
// tiles to fill the chip, and a K of 4864 is a chain of 76 blocks: four groups run it in
// 19 steps).  Waves 2 x 2 over the tile, 32x32x16 MFMAs with the weights as the row
// operand, so a lane holds four consecutive outputs of one row.  Blocks come in as whole
// 128-byte lines (8 rows per wave load) into registers two steps ahead and lie in LDS
// row-major with 16-byte chunks XOR-permuted by the row, double-buffered, one barrier per
// step.  Rows past M and columns past N read as zero through the descriptors; every
// output goes through an fp16 tile in LDS, so the epilogue works on 16-byte vectors.
//
// Every output rounds where the op-by-op path stores fp16 (the product, then bias,
// rotary, residual, activation): results equal that path up to fp32 summation order.
//
// Workgroups are dealt so that the row tiles of a column tile run on one XCD one after
// the other: a weight tile enters one L2, the activations every one.
#include "internal.hpp"
#include "kvc_abi.h"

#include <climits>
#include <cmath>

namespace kvc {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

constexpr int kBlkK = 64;           // k per block: one 128-byte line per row
constexpr int kOobOfs = 0x7FFFFFF0;  // past every descriptor: loads return 0

enum BlockEpi { kBlkStore = 0, kBlkResidual = 1, kBlkQkv = 2, kBlkSwiglu = 3 };

struct BlockParams {
    const _Float16* a;     // [M, K]
    const _Float16* w;     // [N, K] (SwiGLU: [2 I, K], gate rows then up rows)
    int M, N, K;           // N: output columns (SwiGLU: I)
    int mt, nt;            // row and column tiles
    _Float16* out;         // store: y; residual: x (+=); swiglu: act; qkv: q
    const _Float16* bias;  // qkv
    _Float16* k_out;       // qkv: rows [M, kv_cols], or the pool (slots given)
    _Float16* v_out;
    const int* pos;        // qkv: rotary position of each row, or nullptr: pos_base + row
    const int* slots;      // qkv: pool slot of each row (phys * block + in), or nullptr; < 0: not written
    int pos_base, q_cols, kv_cols, head_dim, block;
    float log2_theta;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, 0x00020000);
}
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

template <int BM, int BN, int KG, int EPI, int PD>
__global__ __launch_bounds__(KG * 256) void block_kernel(BlockParams p) {
    constexpr int MT = BM / 64, NT = BN / 64;              // 32-wide MFMA tiles per wave
    constexpr int kRowsTile = BM + BN;                     // A rows, then W rows
    constexpr int kGroupBytes = kRowsTile * kBlkK * 2;
    constexpr int kStage = KG * kGroupBytes;
    constexpr int NL = kRowsTile / 32;                     // 8-row wave loads per wave and block
    constexpr int LDT = BN + 8;                            // row stride of the output tile
    constexpr int kRedBytes = (KG - 1) * BM * BN * 4;
    __shared__ __attribute__((aligned(16))) char s_buf[2 * kStage];
    static_assert(kRedBytes + BM * LDT * 2 <= 2 * kStage, "reduction and output tile fit the buffers");

    const int lane = threadIdx.x & 63;
    const int wave = uniform(threadIdx.x >> 6);
    const int g = wave >> 2, wv = wave & 3;
    const int wm = wv & 1, wn = wv >> 1;
    const int l32 = lane & 31, h = lane >> 5;
    // column tiles n = xcd + 8 j; on an XCD the row tiles of one follow each other
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int tm = idx % p.mt, tn = (idx / p.mt) * 8 + xcd;
    if (tn >= p.nt) return;
    const int m0 = tm * BM;
    const int n0 = tn * (EPI == kBlkSwiglu ? BN / 2 : BN);
    const int kbytes = p.K * 2;
    const int steps = (p.K + KG * kBlkK - 1) / (KG * kBlkK);

    // wave loads i of this wave: 8 rows starting at row 8 (wv + 4 i) of the A|W tile
    const int lrow = lane >> 3, lch = lane & 7;
    const __amdgpu_buffer_rsrc_t ra = rsrc(p.a + (size_t)m0 * p.K, min(p.M - m0, BM) * kbytes);
    __amdgpu_buffer_rsrc_t rw[2];
    if constexpr (EPI == kBlkSwiglu) {
        const int cols = min(p.N - n0, BN / 2) * kbytes;
        rw[0] = rsrc(p.w + (size_t)n0 * p.K, cols);
        rw[1] = rsrc(p.w + (size_t)(p.N + n0) * p.K, cols);
    } else {
        rw[0] = rw[1] = rsrc(p.w + (size_t)n0 * p.K, min(p.N - n0, BN) * kbytes);
    }
    u4 rg[PD][NL];  // blocks in flight
    // wave load i of block s (a wave load lies wholly in A or in one half of W)
    auto load = [&](int s, int i) -> u4 {
        const int k = (s * KG + g) * kBlkK + lch * 8;
        const int r = 8 * (wv + 4 * i);
        const int ro = (r < BM ? r : EPI == kBlkSwiglu ? (r - BM) % (BN / 2) : r - BM) + lrow;
        const __amdgpu_buffer_rsrc_t rs = 8 * 4 * i < BM ? ra : (r - BM < BN / 2 ? rw[0] : rw[1]);
        int o = k < p.K ? ro * kbytes + k * 2 : kOobOfs;
        asm("" : "+v"(o));
        return __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0);
    };
    auto store = [&](int half, int i, u4 v) {  // (row & 7 == lrow)
        *reinterpret_cast<u4*>(s_buf + half * kStage + g * kGroupBytes + (8 * (wv + 4 * i) + lrow) * 128 + ((lch ^ lrow) << 4)) = v;
    };
    f16v acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[n][m][i] = 0.f;
    int ka[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) ka[d] = l32 * 128 + (((2 * d + h) ^ (l32 & 7)) << 4);
    // one block: between the MFMAs of its four k steps, a quarter of the next block's LDS
    // writes and of a further block's loads each (all at once they hold every wave up in
    // the same queue before any wave's MFMAs start)
    auto step = [&](int s, u4 (&r_)[NL]) {
        const int half = s & 1;
        const char* ba = s_buf + half * kStage + g * kGroupBytes + wm * (BM / 2) * 128;
        const char* bw = s_buf + half * kStage + g * kGroupBytes + (BM + wn * (BN / 2)) * 128;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            h8 af[MT], wf[NT];
#pragma unroll
            for (int m = 0; m < MT; ++m) af[m] = *reinterpret_cast<const h8*>(ba + ka[d] + m * 32 * 128);
#pragma unroll
            for (int n = 0; n < NT; ++n) wf[n] = *reinterpret_cast<const h8*>(bw + ka[d] + n * 32 * 128);
#pragma unroll
            for (int i = d * NL / 4; i < (d + 1) * NL / 4; ++i) {
                store(half ^ 1, i, r_[i]);
                r_[i] = load(s + 1 + PD, i);  // (blocks past K read nothing)
            }
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[n], af[m], acc[n][m], 0, 0, 0);
        }
    };
#pragma unroll
    for (int u = 0; u < PD; ++u)
#pragma unroll
        for (int i = 0; i < NL; ++i) rg[u][i] = load(u, i);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        store(0, i, rg[0][i]);
        rg[0][i] = load(PD, i);
    }
    for (int s = 0; s < steps; s += PD) {
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            if (s + u >= steps) break;
            __syncthreads();
            step(s + u, rg[(u + 1) % PD]);
        }
    }
    __syncthreads();
    // acc[n][m][i]: output column wn BN/2 + 32 n + 8 (i / 4) + 4 h + i % 4 of row wm BM/2 + 32 m + l32
    if constexpr (KG > 1) {
        f4* red = reinterpret_cast<f4*>(s_buf);
        auto slot = [&](int gg, int n, int m, int b) {
            return red + ((((gg - 1) * 4 + wv) * NT * MT + n * MT + m) * 4 + b) * 64 + lane;
        };
        if (g > 0) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        *slot(g, n, m, b) = f4{acc[n][m][4 * b], acc[n][m][4 * b + 1], acc[n][m][4 * b + 2], acc[n][m][4 * b + 3]};
        }
        __syncthreads();
        if (g == 0) {
#pragma unroll
            for (int gg = 1; gg < KG; ++gg)
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            const f4 x = *slot(gg, n, m, b);
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[n][m][4 * b + r] += x[r];
                        }
        }
    }
    _Float16* tile = reinterpret_cast<_Float16*>(s_buf + kRedBytes);
    if (g == 0) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    h4 o;
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] = (_Float16)acc[n][m][4 * b + r];
                    *reinterpret_cast<h4*>(tile + (wm * (BM / 2) + 32 * m + l32) * LDT + wn * (BN / 2) + 32 * n + 8 * b + 4 * h) = o;
                }
    }
    __syncthreads();
    auto at = [&](int r, int c) { return *reinterpret_cast<const h8*>(tile + r * LDT + c); };

    if constexpr (EPI == kBlkStore || EPI == kBlkResidual) {
        for (int i = threadIdx.x; i < BM * (BN / 8); i += KG * 256) {
            const int r = i / (BN / 8), c = i % (BN / 8) * 8;
            if (m0 + r >= p.M || n0 + c >= p.N) continue;
            h8* o = reinterpret_cast<h8*>(p.out + (size_t)(m0 + r) * p.N + n0 + c);
            h8 v = at(r, c);
            if constexpr (EPI == kBlkResidual) {
                const h8 x = *o;
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = (_Float16)((float)x[e] + (float)v[e]);
            }
            *o = v;
        }
    } else if constexpr (EPI == kBlkSwiglu) {
        for (int i = threadIdx.x; i < BM * (BN / 16); i += KG * 256) {
            const int r = i / (BN / 16), c = i % (BN / 16) * 8;
            if (m0 + r >= p.M || n0 + c >= p.N) continue;
            const h8 gt = at(r, c), up = at(r, BN / 2 + c);
            h8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float gf = (float)gt[e];
                o[e] = (_Float16)(gf / (1.0f + expf(-gf)) * (float)up[e]);
            }
            *reinterpret_cast<h8*>(p.out + (size_t)(m0 + r) * p.N + n0 + c) = o;
        }
    } else {
        // items: row x eight rotary pairs (t, t + D/2) of a head; a tile holds whole heads
        const int D = p.head_dim, hd = D / 2;
        for (int i = threadIdx.x; i < BM * (BN / 16); i += KG * 256) {
            const int r = i / (BN / 16), j = i % (BN / 16) * 8;  // j: pair column in the tile
            const int head = j / hd, t = j - head * hd;
            const int c = head * D + t, col = n0 + c;
            const int row = m0 + r;
            if (row >= p.M || col >= p.N) continue;
            h8 y0 = at(r, c), y1 = at(r, c + hd);
            const h8 b0 = *reinterpret_cast<const h8*>(p.bias + col), b1 = *reinterpret_cast<const h8*>(p.bias + col + hd);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                y0[e] = (_Float16)((float)y0[e] + (float)b0[e]);
                y1[e] = (_Float16)((float)y1[e] + (float)b1[e]);
            }
            if (col < p.q_cols + p.kv_cols) {  // rotary on q and k (qwen_kernels.cu:64-79)
                const float ps = (float)(p.pos ? p.pos[row] : p.pos_base + row);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float inv = exp2f(-p.log2_theta * (2.0f * (float)(t + e) / (float)D));
                    float sn, co;
                    sincosf(ps * inv, &sn, &co);
                    const float x1 = (float)y0[e], x2 = (float)y1[e];
                    y0[e] = (_Float16)(x1 * co - x2 * sn);
                    y1[e] = (_Float16)(x2 * co + x1 * sn);
                }
            }
            _Float16* o;
            if (col < p.q_cols) {
                o = p.out + (size_t)row * p.q_cols + col;
            } else {
                const bool isk = col < p.q_cols + p.kv_cols;
                const int kc = col - p.q_cols - (isk ? 0 : p.kv_cols);
                o = isk ? p.k_out : p.v_out;
                if (p.slots) {
                    const int slot = p.slots[row];
                    if (slot < 0) continue;
                    const int phys = slot / p.block, in = slot - phys * p.block, kh = kc / D;
                    o += (((size_t)phys * (p.kv_cols / D) + kh) * p.block + in) * D + (kc - kh * D);
                } else {
                    o += (size_t)row * p.kv_cols + kc;
                }
            }
            *reinterpret_cast<h8*>(o) = y0;
            *reinterpret_cast<h8*>(o + hd) = y1;
        }
    }
}

template <int BM, int BN, int KG, int EPI, int PD>
int launch_block(BlockParams& p, hipStream_t st) {
    const int bn = EPI == kBlkSwiglu ? BN / 2 : BN;
    p.mt = (p.M + BM - 1) / BM;
    p.nt = (p.N + bn - 1) / bn;
    const long long grid = (long long)((p.nt + 7) / 8) * 8 * p.mt;
    if (grid > INT_MAX) return set_error(KVC_ERR_ARG, "linear: grid too large");
    hipLaunchKernelGGL((block_kernel<BM, BN, KG, EPI, PD>), dim3((unsigned)grid), dim3(KG * 256), 0, st, p);
    return hip_check(hipGetLastError(), "block linear launch");
}

// Tiles of 128 x 128 once they give nearly a workgroup per CU, else of 64 x 64 (700 rows,
// q|k|v 9.6 and 16 us; gate|up, 456 tiles of 128, 30.6 and 23.5).  K groups: two for small
// tiles (16 rows, o_proj 5.9 us, 6.2 with one, 7.0 with four), four for a long K with few
// tiles (700 rows, K 4864, 19.5 us; 26.0 with one); large tiles of the residual layers run
// two as well (4096 rows, K 4864 52.6 us, 55.2 with one; K 896 16.4 and 14.6).  Two blocks
// in flight were as good as three or four.  What bounds a step: LDS traffic and the loads'
// issue (64 B per cycle) of tiles this small, about as long as the MFMAs each; 700 rows of
// gate|up 520 TFLOP/s.  Before (rocBLAS and a kernel per op, 700 rows): q|k|v with bias and
// rotary 46 us -> 10, o_proj and residual 15 -> 6.5, gate|up and SwiGLU 36 -> 23.5, down and
// residual 29 -> 20.
template <int EPI>
int launch_block_shape(BlockParams& p, hipStream_t st) {
    auto tiles = [&](int t) {
        const int bn = EPI == kBlkSwiglu ? t / 2 : t;
        return (long long)((p.M + t - 1) / t) * ((p.N + bn - 1) / bn);
    };
    const bool longk = p.K >= 2048;
    if (tiles(128) >= 200 || (EPI == kBlkQkv && p.head_dim > 64))  // (a q|k|v tile holds whole heads)
        return EPI == kBlkResidual || longk ? launch_block<128, 128, 2, EPI, 2>(p, st)
                                            : launch_block<128, 128, 1, EPI, 1>(p, st);
    return longk && tiles(64) < 300 ? launch_block<64, 64, 4, EPI, 2>(p, st) : launch_block<64, 64, 2, EPI, 2>(p, st);
}

bool al16(const void* p) { return p && ((uintptr_t)p & 15u) == 0; }

int check_block(int M, int N, int K, const void* x, const void* w) {
    if (M < 0 || N <= 0 || K <= 0 || N % 8 || K % 8) return set_error(KVC_ERR_ARG, "block linear: M >= 0, N and K multiples of 8");
    if ((long long)K * 256 >= INT_MAX) return set_error(KVC_ERR_UNSUPPORTED, "block linear: K too large");
    if (M > 0 && (!al16(x) || !al16(w))) return set_error(KVC_ERR_ARG, "block linear: x and w must be 16-byte aligned");
    return KVC_OK;
}

}  // namespace
}  // namespace kvc

using namespace kvc;

extern "C" {

int kvc_block_linear(void* y, const void* x, const void* w, int M, int N, int K, int residual, kvc_stream_t st) {
    int rc = check_block(M, N, K, x, w);
    if (rc || M == 0) return rc;
    if (!al16(y) || y == x) return set_error(KVC_ERR_ARG, "block linear: y must be 16-byte aligned and not x");
    BlockParams p{};
    p.a = (const _Float16*)x; p.w = (const _Float16*)w; p.M = M; p.N = N; p.K = K; p.out = (_Float16*)y;
    return residual ? launch_block_shape<kBlkResidual>(p, (hipStream_t)st)
                    : launch_block_shape<kBlkStore>(p, (hipStream_t)st);
}

int kvc_block_qkv(void* q, void* k, void* v, const void* x, const void* w_qkv, const void* b_qkv, const int* pos,
                  int pos_base, const int* slots, int M, int H, int Hq, int Hkv, int D, int BLOCK, float theta,
                  kvc_stream_t st) {
    if (Hq <= 0 || Hkv <= 0 || (D != 32 && D != 64 && D != 128) || !(theta > 1.f))
        return set_error(KVC_ERR_ARG, "block qkv: heads > 0, D 32, 64 or 128, theta > 1");
    int rc = check_block(M, (Hq + 2 * Hkv) * D, H, x, w_qkv);
    if (rc || M == 0) return rc;
    if (slots && BLOCK <= 0) return set_error(KVC_ERR_ARG, "block qkv: slots need BLOCK > 0");
    if (!al16(q) || !al16(k) || !al16(v) || !al16(b_qkv))
        return set_error(KVC_ERR_ARG, "block qkv: null or misaligned pointer");
    BlockParams p{};
    p.a = (const _Float16*)x; p.w = (const _Float16*)w_qkv; p.M = M; p.N = (Hq + 2 * Hkv) * D; p.K = H;
    p.out = (_Float16*)q; p.k_out = (_Float16*)k; p.v_out = (_Float16*)v; p.bias = (const _Float16*)b_qkv;
    p.pos = pos; p.pos_base = pos_base; p.slots = slots; p.block = BLOCK;
    p.q_cols = Hq * D; p.kv_cols = Hkv * D; p.head_dim = D; p.log2_theta = log2f(theta);
    return launch_block_shape<kBlkQkv>(p, (hipStream_t)st);
}

int kvc_block_swiglu(void* act, const void* x, const void* w_gate_up, int M, int I, int H, kvc_stream_t st) {
    int rc = check_block(M, I, H, x, w_gate_up);
    if (rc || M == 0) return rc;
    if (!al16(act)) return set_error(KVC_ERR_ARG, "block swiglu: act must be 16-byte aligned");
    BlockParams p{};
    p.a = (const _Float16*)x; p.w = (const _Float16*)w_gate_up; p.M = M; p.N = I; p.K = H; p.out = (_Float16*)act;
    return launch_block_shape<kBlkSwiglu>(p, (hipStream_t)st);
}

}  // extern "C"

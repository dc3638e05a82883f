// prompt_mfma.hpp -- prompt (prefill) attention on the matrix cores (fp16 K/V, head_dim 64/128).
//
// Included by decode_kernels.hpp inside namespace kvc::{anonymous}; uses its helpers.
//
// qk_paged_causal_attn (qwen_kernels.cu:146-181): query i of one sequence at position
// base + i attends to keys 0 .. base + i of the paged pools.  Two kernels share the
// arithmetic of a 32-key x 32-query tile:
//
//   QK^T  : S^T[32 keys][32 queries] = K Q^T with v_mfma_f32_32x32x16_f16, so a lane
//           holds 16 scores of ONE query (column l % 32): the row maximum and sum need one
//           exchange with lane l ^ 32, and the rescale factor is a per-lane scalar.
//   softmax: fp32 online (reference, sum, acc) in log2 units; O is rescaled only when some
//           query of the wave met a new maximum.  head_dim 128: then every query takes the
//           tile's own maximum as its reference (at most 2^8 below its running maximum), since
//           a probability of exactly 1 loses nothing to its rounding to fp16, and the fewer
//           maxima the key streams have between them, the larger the error (1000 queries
//           behind 6000 keys, against 64 bits: running maxima of two streams 2.83e-4, of the
//           four of the 16-query units before 2.80e-4, this 2.69e-4; 100 behind 1500 2.66e-4,
//           2.61e-4, 2.53e-4).  At head_dim 64 running maxima are no further off than those
//           units were (2.45e-4 and 2.47e-4 at 2048 queries), and this cost 3% there.
//   PV    : O^T[32 dims][32 queries] += V^T P^T.  The lane's own probabilities are in the
//           B operand layout up to the order of the keys, and V^T is read back in that
//           order with the transposing LDS read, so P never leaves its registers.
//
// prompt_kernel: a workgroup of 8 waves takes 32 * QG consecutive queries of one head, QG
// groups of 32 queries times KS = 8 / QG key streams.  Keys come in sets of 128, stream ks
// of a set taking its KT = 128 / KS keys; wave w brings rows 16w .. 16w+15 of a set (one
// block id, whole rows, 1 KiB per wave load, rows past the end read as zero through the
// descriptor) into registers while the set before is computed, then into the other half
// of the LDS buffer; one barrier per set.  The larger QG, the fewer times a key is loaded.
// prompt_stream_kernel: 32 queries, eight key streams of their own, no barrier.
//
// LDS: K rows as 16-byte chunks XOR-permuted by the row, V rows as 32-byte segments
// permuted by the row, so that neither operand read meets a bank twice.
//
// What bounds them: the vector instructions of the softmax (about 60 per tile, 33 more
// with a rescale, 600 cycles) beside 256 cycles of MFMA; at 8192 queries of 14 heads, D 64,
// vector and matrix instructions together fill 83% of the cycles (196 us, 610 TFLOP/s); at
// 2048 queries the longest tiles and the start and end of each workgroup (about 4 us).
// Before (16 queries of a head per unit, each key loaded per unit): 2048 queries 37 -> 22
// us, 1000 queries of 32 heads, D 128, behind 6000 keys 515 -> 140 us, 700 queries 10.3 ->
// 8.2 us.

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

// Inf and NaN in V behind the causal edge.  A key that a query does not see has probability
// 0, and 0 x Inf is NaN, so in the tiles of the edge the elements of V that are not finite
// are staged as 0 (clear_nonfinite) and a workgroup that met one adds them, in its epilogue,
// to the queries that see their key (add_nonfinite).
__device__ __forceinline__ bool nonfinite(unsigned half_bits) { return (half_bits & 0x7C00u) == 0x7C00u; }

// Whether the wave's v hold Inf or NaN.
template <int NV>
__device__ __forceinline__ bool any_nonfinite(const u32x4 (&v)[NV]) {
    const f16x2 zero = {(_Float16)0.f, (_Float16)0.f};
    f16x2 c[4] = {zero, zero, zero, zero};  // + x * 0: stays 0 unless some x is Inf or NaN
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const unsigned x = v[i][e];
            c[e] = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, x), zero, c[e]);
        }
    const f16x2 t = (c[0] + c[1]) + (c[2] + c[3]);
    return __any(!(t[0] == zero[0] && t[1] == zero[1]));
}

template <int NV>
__device__ __forceinline__ void clear_nonfinite(u32x4 (&v)[NV]) {
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            v[i][e] &= (nonfinite(v[i][e]) ? 0u : 0xFFFFu) | (nonfinite(v[i][e] >> 16) ? 0u : 0xFFFF0000u);
}

// acc += the elements d0 .. d0 + 3 of V that are Inf or NaN, of keys [first, last].
template <int D>
__device__ __forceinline__ f32x4 add_nonfinite(f32x4 acc, const char* vb, const int* table, int bsh, int Hkv, int hk,
                                            int first, int last, int d0) {
    for (int j = first; j <= last; ++j) {
        const size_t row = ((size_t)(unsigned)(table[j >> bsh] * Hkv + hk) << bsh) + (j & ((1 << bsh) - 1));
        const f16x4 v = *reinterpret_cast<const f16x4*>(vb + (row * D + d0) * 2);
        const u16x4 bits = __builtin_bit_cast(u16x4, v);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (nonfinite(bits[r])) acc[r] += (float)v[r];
    }
    return acc;
}

template <int D, int QG>
__global__ __launch_bounds__(8 * kWave) void prompt_kernel(DecodeParams p) {
    constexpr int W = 8;
    constexpr int ROW = D * 2;              // bytes per K/V row
    constexpr int KS = W / QG;              // key streams
    constexpr int kPromptSet = 16 * W;      // keys per LDS set (each wave loads 16 rows)
    constexpr int KT = kPromptSet / KS;     // keys per stream and set (64 or 32)
    constexpr int NS = KT / 32;             // 32-key subtiles
    constexpr int KD = D / 16;              // MFMA k steps over the head dimension
    constexpr int DT = D / 32;              // 32-dim output tiles
    constexpr int VL = 16 * ROW / 1024;     // wave loads per 16-row subtile
    constexpr int kSetBytes = kPromptSet * ROW;
    __shared__ __attribute__((aligned(16))) char s_kv[2][2][kSetBytes];  // [half][K / V]
    __shared__ float s_ml[KS][QG][32][2];
    __shared__ int s_bad[W];
    static_assert(KS * QG * 32 * D * 4 <= 2 * 2 * kSetBytes, "partials fit the tile buffers");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = uniform(threadIdx.x >> 6);
    const int qg = wave % QG, ks = wave / QG;
    const int l32 = lane & 31, h = lane >> 5;

    // KV heads fastest: consecutive workgroups go to the XCDs in turn, so the query tiles
    // of a KV head meet in few L2s; longest prefixes first
    int unit = blockIdx.x;
    const int hi = unit % p.Hq;  unit /= p.Hq;
    const int hk = hi % p.Hkv, qh = hk * p.group + hi / p.Hkv;
    const int ntq = (p.N + 32 * QG - 1) / (32 * QG);
    const int q0 = (ntq - 1 - unit) * 32 * QG;
    const int base = p.fixed_len;
    const int lmax = base + min(q0 + 32 * QG, p.N);  // keys of the tile's last query
    const int nsets = (lmax + kPromptSet - 1) / kPromptSet;
    const int nfull = min(nsets, (base + q0 + 1) / kPromptSet);  // sets that every query of the tile sees whole
    bool bad = false;  // this wave cleared elements of V in the sets after those
    const int qw = q0 + 32 * qg;                     // the wave's first query
    const int qlast = base + qw + l32;               // last key this column sees

    const int bsh = __builtin_ctz((unsigned)p.block), bmask = p.block - 1;
    const unsigned blk_bytes = (unsigned)p.block * ROW;
    const char* kb = static_cast<const char*>(p.k);
    const char* vb = static_cast<const char*>(p.v);
    // rows 16 wave .. +15 of set s; their block ids are held one set per lane, 64 sets at a
    // time (read per set they were scalar loads, whose wait also holds up the LDS reads)
    auto first_tok = [&](int s) { return s * kPromptSet + 16 * wave; };
    int ids = 0;
    auto load_ids = [&](int s) { ids = p.table_all[min(first_tok(s + lane), lmax - 1) >> bsh]; };
    u32x4 rk[VL], rv[VL];
    size_t i_off = 0;
    int i_bytes = 0;
    auto issue_k = [&](int s) {
        const int t = first_tok(s);
        const int id = __builtin_amdgcn_readlane(ids, s & (kWave - 1));
        int rows = max(lmax - t, 0);
        asm("" : "+s"(rows));
        i_bytes = min(rows, 16) * ROW;
        i_off = (size_t)(unsigned)(id * p.Hkv + hk) * blk_bytes + (unsigned)((t & bmask) * ROW);
        const __amdgpu_buffer_rsrc_t kr = tile_rsrc(kb + i_off, i_bytes);
#pragma unroll
        for (int i = 0; i < VL; ++i) rk[i] = buffer_load16(kr, i * 1024 + lane * 16);
    };
    auto issue_v = [&]() {  // of the rows issue_k located
        const __amdgpu_buffer_rsrc_t vr = tile_rsrc(vb + i_off, i_bytes);
#pragma unroll
        for (int i = 0; i < VL; ++i) rv[i] = buffer_load16(vr, i * 1024 + lane * 16);
    };
    auto kchunk = [](int r, int ch) { return ch ^ (r & 7); };
    auto vseg = [](int r, int seg) { return seg ^ (D == 64 ? (r >> 1) & 3 : r & 7); };
    auto store = [&](int half, bool edge) {
        if (edge && any_nonfinite(rv)) {
            clear_nonfinite(rv);
            bad = true;
        }
#pragma unroll
        for (int i = 0; i < VL; ++i) {
            const int off = i * 1024 + lane * 16;
            const int r = 16 * wave + off / ROW, cb = off % ROW;
            *reinterpret_cast<u32x4*>(s_kv[half][0] + r * ROW + kchunk(r, cb >> 4) * 16) = rk[i];
            *reinterpret_cast<u32x4*>(s_kv[half][1] + r * ROW + vseg(r, cb >> 5) * 32 + (cb & 31)) = rv[i];
        }
    };

    load_ids(0);
    issue_k(0);
    issue_v();
    // q as the B operand: lane l holds query qw + l % 32, dims 16 d + 8 (l / 32) .. +7
    // (queries past N read as zero through the descriptor)
    f16x8v qb[KD];
    {
        const __amdgpu_buffer_rsrc_t qr = tile_rsrc(p.q, p.N * p.Hq * ROW);
        const int qoff = ((qw + l32) * p.Hq + qh) * ROW + h * 16;
#pragma unroll
        for (int d = 0; d < KD; ++d) qb[d] = __builtin_bit_cast(f16x8v, buffer_load16(qr, qoff + d * 32));
    }
    // scores use |scale|: a negative scale negates q instead (exact in fp16)
    const float sl2 = fabsf(p.scale_log2);
    if (p.scale_log2 < 0.f) {
#pragma unroll
        for (int d = 0; d < KD; ++d) qb[d] = -qb[d];
    }
    float m = -FLT_MAX, l = 0.f;  // of this column; l of the lane's own keys only
    float top = -FLT_MAX;         // its running maximum (m: the reference of l and O; D 64: both)
    f32x16 O[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[dt][i] = 0.f;

    // operand addresses within a stream's tile: the permutations only touch the low three
    // bits of the row, so rows 32 n, 16 t and 8 further on are constant offsets
    int ka[4], va[DT];
#pragma unroll
    for (int d = 0; d < 4; ++d) ka[d] = ks * KT * ROW + l32 * ROW + kchunk(l32, 2 * d + h) * 16;
    const int vr = 4 * h + ((lane & 15) >> 2);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        va[dt] = kSetBytes + ks * KT * ROW + vr * ROW + vseg(vr, 2 * dt + ((lane >> 4) & 1)) * 32 + 8 * (lane & 3);
    // one stream's tile of a set: keys t0 .. t0 + KT - 1, LDS rows ks * KT ..
    auto compute = [&](int half, int t0, auto masked_tag) {
        constexpr bool MASKED = decltype(masked_tag)::value;
        const char* buf = &s_kv[0][0][0] + half * (2 * kSetBytes);
        f32x16 S[NS];
#pragma unroll
        for (int n = 0; n < NS; ++n) {
#pragma unroll
            for (int i = 0; i < 16; ++i) S[n][i] = 0.f;
#pragma unroll
            for (int d = 0; d < KD; ++d) {
                const f16x8v a = *reinterpret_cast<const f16x8v*>(buf + ka[d & 3] + 32 * n * ROW + (d >> 2) * 128);
                S[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qb[d], S[n], 0, 0, 0);
            }
        }
        // S[n][i] is key t0 + 32 n + 8 (i / 4) + 4 h + i % 4
        const int lim = qlast - t0 - 4 * h;  // seen when 32 n + 8 (i / 4) + i % 4 <= lim
        // each 32-key subtile against its own maximum (over 64 keys at a time the error
        // against 64 bits was 1% larger: fewer probabilities are exactly 1)
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            auto seen = [&](int i) { return !MASKED || 32 * n + 8 * (i >> 2) + (i & 3) <= lim; };
            float mx = -FLT_MAX;
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = seen(i) ? fmaxf(mx, S[n][i]) : mx;
            mx = max_xor32(mx) * sl2;
            if (__any(mx > (D == 128 ? top : m))) {
                if constexpr (D == 128) top = fmaxf(top, mx);
                const float mn = D == 128 ? fmaxf(mx, top - 8.f) : fmaxf(m, mx);
                const float corr = fast_exp2(m - mn);
                m = mn;
                l *= corr;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) O[dt][i] *= corr;
            }
            float ps = 0.f;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f16x8v pb;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float e = fast_exp2(__builtin_fmaf(S[n][8 * t + j], sl2, -m));
                    e = seen(8 * t + j) ? e : 0.f;
                    ps += e;
                    pb[j] = (_Float16)e;
                }
                // V^T operand: k slots (h, j) are keys 32 n + 16 t + 8 (j / 4) + 4 h + j % 4,
                // of dim 32 dt + l % 32; two transposing reads of four keys each (16 lanes
                // address four rows of 16 dims: lane i row i / 4, dims 4 (i % 4) .. +3)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    const char* vt = buf + va[dt] + (32 * n + 16 * t) * ROW;
                    const s16x4v lo = ds_read_tr16(vt), hi2 = ds_read_tr16(vt + 8 * ROW);
                    const f16x8v a = __builtin_bit_cast(f16x8v, __builtin_shufflevector(lo, hi2, 0, 1, 2, 3, 4, 5, 6, 7));
                    O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pb, O[dt], 0, 0, 0);
                }
            }
            l += ps;
        }
    };

    const int wlast = base + min(qw + 31, p.N - 1);  // last key any query of the wave sees
    store(0, nfull == 0);
    issue_k(1);
    issue_v();
    // one set: the next one from its registers into the other half of the buffer, the
    // one after that into flight, then this one's arithmetic
    auto set = [&](int s, auto masked_tag) {
        __syncthreads();
        store((s + 1) & 1, decltype(masked_tag)::value || s + 1 >= nfull);
        if (((s + 2) & (kWave - 1)) == 0) load_ids(s + 2);
        issue_k(s + 2);  // (sets past the end read nothing: zero-size descriptors)
        issue_v();
        const int t0 = s * kPromptSet + ks * KT;
        if (!decltype(masked_tag)::value || (qw < p.N && t0 <= wlast)) compute(s & 1, t0, masked_tag);
    };
    // (loops of their own: one loop with both forms copied O between them in every set)
    int s = 0;
    for (; s < nfull; ++s) set(s, std::false_type{});
    for (; s < nsets; ++s) set(s, std::true_type{});
    __syncthreads();
    l = sum_xor32(l);

    // every stream leaves (m, l, O) in LDS; then wave (qg, ks) combines its share of the
    // group's dims: slots of four consecutive dims of a column
    constexpr int SL = DT * 4 / KS;  // slots per wave
    static_assert(DT * 4 % KS == 0, "slots divide among the streams");
    f32x4* part = reinterpret_cast<f32x4*>(&s_kv[0][0][0]);
    auto slot = [&](int k, int i4) { return part + ((k * QG + qg) * (DT * 4) + i4) * kWave + lane; };
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int b = 0; b < 4; ++b)
            *slot(ks, dt * 4 + b) = f32x4{O[dt][4 * b], O[dt][4 * b + 1], O[dt][4 * b + 2], O[dt][4 * b + 3]};
    if (h == 0) {
        s_ml[ks][qg][l32][0] = m;
        s_ml[ks][qg][l32][1] = l;
    }
    if (lane == 0) s_bad[wave] = bad;
    __syncthreads();
    float M = -FLT_MAX;
#pragma unroll
    for (int k = 0; k < KS; ++k) M = fmaxf(M, s_ml[k][qg][l32][0]);
    float lt = 0.f;
    f32x4 acc[SL];
#pragma unroll
    for (int i = 0; i < SL; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const float wk = fast_exp2(s_ml[k][qg][l32][0] - M);
        lt = __builtin_fmaf(wk, s_ml[k][qg][l32][1], lt);
#pragma unroll
        for (int i = 0; i < SL; ++i) {
            const f32x4 x = *slot(k, ks * SL + i);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][r] = __builtin_fmaf(wk, x[r], acc[i][r]);
        }
    }
    const int q = qw + l32;
    if (q >= p.N) return;
    int any_bad = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) any_bad |= s_bad[w];
    if (any_bad)
#pragma unroll
        for (int i = 0; i < SL; ++i)
            acc[i] = add_nonfinite<D>(acc[i], vb, p.table_all, bsh, p.Hkv, hk, nfull * kPromptSet, qlast,
                                      8 * (ks * SL + i) + 4 * h);
    const float inv = lt > 0.f ? 1.0f / lt : 0.f;
    _Float16* ob = static_cast<_Float16*>(p.out) + ((size_t)q * p.Hq + qh) * D + 4 * h;
#pragma unroll
    for (int i = 0; i < SL; ++i) {
        f16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (_Float16)(lt > 0.f ? acc[i][r] * inv : 0.f);
        *reinterpret_cast<f16x4*>(ob + 8 * (ks * SL + i)) = o;
    }
}

// Key streams of their own: wave w of 8 takes key tiles w, w + 8, ... of 32 keys for the 32
// queries of the workgroup, loading and staging them by itself, so no barrier holds the
// waves in step (where every wave meets the same unit at once: loads, then LDS writes, then
// MFMAs).
template <int D>
__global__ __launch_bounds__(8 * kWave, D == 64 ? 4 : 2) void prompt_stream_kernel(DecodeParams p) {
    constexpr int ROW = D * 2;
    constexpr int KD = D / 16, DT = D / 32;
    constexpr int VL = 16 * ROW / 1024;      // wave loads per 16-row subtile
    constexpr int W = 8;
    constexpr int kTile = 32 * ROW;          // bytes of one K (or V) tile
    __shared__ __attribute__((aligned(16))) char s_kv[W][2][kTile];
    __shared__ float s_ml[W][32][2];

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = uniform(threadIdx.x >> 6);
    const int l32 = lane & 31, h = lane >> 5;
    int unit = blockIdx.x;
    const int hi = unit % p.Hq;  unit /= p.Hq;
    const int hk = hi % p.Hkv, qh = hk * p.group + hi / p.Hkv;
    const int ntq = (p.N + 31) / 32;
    const int q0 = (ntq - 1 - unit % ntq) * 32;
    const int c = unit / ntq;
    // the position and, with it, the chunks: from the host, or from device memory
    int base = p.fixed_len, chunk = p.chunk_tokens;
    if (p.dev_base) {
        base = uniform(*p.dev_base);
        const int lall = (int)min((long long)base + p.N, (long long)INT_MAX);
        // past the planning budget of the device-length launches (self_plan_setup's rule:
        // mean length over the records, longest length over the mergeable chunks)
        const long long M63 = (long long)(p.sp_records - 1) * p.sp_max_chunk;
        if (2LL * base + p.N + 1 > 2 * M63 || (p.sp_nc_max && lall > 63LL * p.sp_max_chunk)) {
            if (c == 0) {
                for (int q = q0; q < min(q0 + 32, p.N); ++q) {
                    _Float16* ob = static_cast<_Float16*>(p.out) + ((size_t)q * p.Hq + qh) * D;
                    for (int e = threadIdx.x; e < D; e += W * kWave) ob[e] = (_Float16)__builtin_nanf("");
                }
                report_device_error(p, kDevErrBudget);
            }
            return;
        }
        const int nch = lall < kPromptSplitMin ? 1 : min(max(lall / p.sp_min_chunk, 1), p.max_chunks);
        const int al = max(p.block, 256);
        chunk = max((lall / nch + al) / al * al, al);  // nch chunks of it cover lall
    }
    const int lmax = base + min(q0 + 32, p.N);
    const int j0 = c * chunk, j1 = min(j0 + chunk, lmax);
    if (j0 >= lmax && c > 0) return;
    const int ntiles = max(0, j1 - j0 + 31) / 32;  // (none: a position below -q, whose rows are 0)
    const int kmax = wave < ntiles ? (ntiles - wave + W - 1) / W : 0;

    const int bsh = __builtin_ctz((unsigned)p.block), bmask = p.block - 1;
    const unsigned blk_bytes = (unsigned)p.block * ROW;
    const char* kb = static_cast<const char*>(p.k);
    const char* vb = static_cast<const char*>(p.v);
    // subtile u (16 rows) of this wave: first token; block ids one subtile per lane
    auto first_tok = [&](int u) { return j0 + (wave + W * (u >> 1)) * 32 + 16 * (u & 1); };
    int ids = 0;
    auto load_ids = [&](int u) { ids = ntiles > 0 ? p.table_all[min(first_tok(u + lane), j1 - 1) >> bsh] : 0; };
    u32x4 rk[2][VL], rv[2][VL];
    auto issue = [&](int k) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int tok = first_tok(2 * k + t);
            const int id = __builtin_amdgcn_readlane(ids, (2 * k + t) & (kWave - 1));
            int rows = max(j1 - tok, 0);
            asm("" : "+s"(rows));
            const int bytes = min(rows, 16) * ROW;
            const size_t off = (size_t)(unsigned)(id * p.Hkv + hk) * blk_bytes + (unsigned)((tok & bmask) * ROW);
            const __amdgpu_buffer_rsrc_t kr = tile_rsrc(kb + off, bytes), vr = tile_rsrc(vb + off, bytes);
#pragma unroll
            for (int i = 0; i < VL; ++i) rk[t][i] = buffer_load16(kr, i * 1024 + lane * 16);
#pragma unroll
            for (int i = 0; i < VL; ++i) rv[t][i] = buffer_load16(vr, i * 1024 + lane * 16);
        }
    };
    auto kchunk = [](int r, int ch) { return ch ^ (r & 7); };
    auto vseg = [](int r, int seg) { return seg ^ (D == 64 ? (r >> 1) & 3 : r & 7); };
    char* kt = s_kv[wave][0];
    char* vt = s_kv[wave][1];
    auto stage = [&]() {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < VL; ++i) {
                const int off = i * 1024 + lane * 16;
                const int r = 16 * t + off / ROW, cb = off % ROW;
                *reinterpret_cast<u32x4*>(kt + r * ROW + kchunk(r, cb >> 4) * 16) = rk[t][i];
                *reinterpret_cast<u32x4*>(vt + r * ROW + vseg(r, cb >> 5) * 32 + (cb & 31)) = rv[t][i];
            }
    };

    load_ids(0);
    issue(0);
    f16x8v qb[KD];
    {
        const __amdgpu_buffer_rsrc_t qr = tile_rsrc(p.q, p.N * p.Hq * ROW);
        const int qoff = ((q0 + l32) * p.Hq + qh) * ROW + h * 16;
#pragma unroll
        for (int d = 0; d < KD; ++d) qb[d] = __builtin_bit_cast(f16x8v, buffer_load16(qr, qoff + d * 32));
    }
    const float sl2 = fabsf(p.scale_log2);
    if (p.scale_log2 < 0.f) {
#pragma unroll
        for (int d = 0; d < KD; ++d) qb[d] = -qb[d];
    }
    float m = -FLT_MAX, l = 0.f, top = -FLT_MAX;  // as prompt_kernel's
    f32x16 O[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[dt][i] = 0.f;
    int ka[4], va[DT];
#pragma unroll
    for (int d = 0; d < 4; ++d) ka[d] = l32 * ROW + kchunk(l32, 2 * d + h) * 16;
    const int vr0 = 4 * h + ((lane & 15) >> 2);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) va[dt] = vr0 * ROW + vseg(vr0, 2 * dt + ((lane >> 4) & 1)) * 32 + 8 * (lane & 3);

    auto compute = [&](int t0, auto masked_tag) {
        constexpr bool MASKED = decltype(masked_tag)::value;
        f32x16 S;
#pragma unroll
        for (int i = 0; i < 16; ++i) S[i] = 0.f;
#pragma unroll
        for (int d = 0; d < KD; ++d) {
            const f16x8v a = *reinterpret_cast<const f16x8v*>(kt + ka[d & 3] + (d >> 2) * 128);
            S = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qb[d], S, 0, 0, 0);
        }
        f16x8v pb[2];
        const int lim = base + q0 + l32 - t0 - 4 * h;
        auto seen = [&](int i) { return !MASKED || 8 * (i >> 2) + (i & 3) <= lim; };
        float mx = -FLT_MAX;
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = seen(i) ? fmaxf(mx, S[i]) : mx;
        mx = max_xor32(mx) * sl2;
        if (__any(mx > (D == 128 ? top : m))) {
            if constexpr (D == 128) top = fmaxf(top, mx);
            const float mn = D == 128 ? fmaxf(mx, top - 8.f) : fmaxf(m, mx);
            const float corr = fast_exp2(m - mn);
            m = mn;
            l *= corr;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) O[dt][i] *= corr;
        }
        float ps = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float e = fast_exp2(__builtin_fmaf(S[i], sl2, -m));
            e = seen(i) ? e : 0.f;
            ps += e;
            pb[i >> 3][i & 7] = (_Float16)e;
        }
        l += ps;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const s16x4v lo = ds_read_tr16(vt + va[dt] + 16 * t * ROW), hi2 = ds_read_tr16(vt + va[dt] + (16 * t + 8) * ROW);
                const f16x8v a = __builtin_bit_cast(f16x8v, __builtin_shufflevector(lo, hi2, 0, 1, 2, 3, 4, 5, 6, 7));
                O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pb[t], O[dt], 0, 0, 0);
            }
    };
    bool bad = false;  // this wave cleared elements of V in its tiles of the causal edge
    auto step = [&](int k, auto masked_tag) {
        __builtin_amdgcn_wave_barrier();
        stage();
        if constexpr (decltype(masked_tag)::value) {  // (while the LDS writes are under way)
            const bool bad0 = any_nonfinite(rv[0]), bad1 = any_nonfinite(rv[1]);
            if (bad0 || bad1) {
                clear_nonfinite(rv[0]);
                clear_nonfinite(rv[1]);
                bad = true;
                stage();
            }
        }
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
        if (((2 * (k + 1)) & (kWave - 1)) == 0) load_ids(2 * (k + 1));
        issue(k + 1);
        compute(j0 + (wave + W * k) * 32, masked_tag);
        asm volatile("" ::: "memory");
    };
    // tiles every query sees whole, then those with the causal edge
    const int full = max(0, (base + q0 + 1 - j0) / 32);  // leading tiles of the chunk that are whole
    const int kfull = min(kmax, full > wave ? (full - wave + W - 1) / W : 0);
    int k = 0;
    for (; k < kfull; ++k) step(k, std::false_type{});
    for (; k < kmax; ++k) step(k, std::true_type{});

    // combine: every wave's O through LDS, then wave w sums its share of the slots of four
    // consecutive dims of a column (a slot: 64 lanes x 4 dims)
    constexpr int kSlots = DT * 4;
    constexpr int kPer = kSlots / W;
    static_assert(kSlots % W == 0 && W * kSlots * kWave * 16 <= (int)sizeof(s_kv), "the partials fit the tiles");
    f32x4* part = reinterpret_cast<f32x4*>(&s_kv[0][0][0]);
    __syncthreads();
    const int nw = min(W, ntiles);  // waves that had tiles
    if (wave < max(nw, 2) || nw > 2) {
        const float lt = sum_xor32(l);
        if (h == 0) {
            s_ml[wave][l32][0] = m;
            s_ml[wave][l32][1] = bad ? -lt : lt;  // (the sign, also of 0: elements to add)
        }
#pragma unroll
        for (int i = 0; i < kSlots; ++i)
            part[(wave * kSlots + i) * kWave + lane] =
                f32x4{O[i >> 2][4 * (i & 3)], O[i >> 2][4 * (i & 3) + 1], O[i >> 2][4 * (i & 3) + 2], O[i >> 2][4 * (i & 3) + 3]};
    }
    __syncthreads();
    float M = -FLT_MAX, lt = 0.f;
    unsigned any_bad = 0;
    f32x4 acc[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto combine = [&](auto n_tag) {
        constexpr int NW = decltype(n_tag)::value;
        float mw[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            mw[w] = s_ml[w][l32][0];
            M = fmaxf(M, mw[w]);
        }
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float wk = fast_exp2(mw[w] - M), lw = s_ml[w][l32][1];
            any_bad |= __float_as_uint(lw) & 0x80000000u;
            lt = __builtin_fmaf(wk, fabsf(lw), lt);
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const f32x4 x = part[(w * kSlots + wave * kPer + i) * kWave + lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][r] = __builtin_fmaf(wk, x[r], acc[i][r]);
            }
        }
    };
    // prompts of up to 64 keys leave two waves' partials (8 queries: 5.0 us with all eight, 4.5)
    if (nw > 2) combine(std::integral_constant<int, W>{});
    else combine(std::integral_constant<int, 2>{});
    const int q = q0 + l32;
    const int ncq = max(base + q, 0) / chunk + 1;  // chunks of the query
    if (any_bad)
#pragma unroll
        for (int i = 0; i < kPer; ++i)
            acc[i] = add_nonfinite<D>(acc[i], vb, p.table_all, bsh, p.Hkv, hk, j0 + 32 * full, min(base + q, j1 - 1),
                                      8 * (wave * kPer + i) + 4 * h);
    // host positions: merge_kernel follows (20 queries, 14 heads, behind 5900 keys: 10.5 us,
    // 13.9 merged in here); a device position does not know on the host whether one is needed
    const bool fused = p.merge_mode == kMergeAtomic;
    if (q < p.N && c < ncq) {
        const float inv = lt > 0.f ? 1.0f / lt : 0.f;
        const size_t rec = ((size_t)q * p.max_chunks + c) * p.Hq + qh;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int d0 = 8 * (wave * kPer + i) + 4 * h;
            if (ncq == 1) {
                f16x4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = (_Float16)(lt > 0.f ? acc[i][r] * inv : 0.f);
                *reinterpret_cast<f16x4*>(static_cast<_Float16*>(p.out) + ((size_t)q * p.Hq + qh) * D + d0) = o;
            } else if (!fused) {
                *reinterpret_cast<f32x4*>(p.part_acc + rec * D + d0) = acc[i];
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    __hip_atomic_store(p.part_acc + rec * D + d0 + r, acc[i][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (ncq > 1 && wave == 0 && h == 0) {  // (the merge kernel's plain loads see these stores too)
            __hip_atomic_store(p.part_ml + rec * 2, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(p.part_ml + rec * 2 + 1, lt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    const int nct = (lmax - 1) / chunk + 1;  // chunks of the tile
    if (!fused || nct <= 1) return;
    // the tile's last chunk to arrive merges its split queries
    __shared__ int s_last;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);  // every thread's partial stores complete before the arrival
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    unsigned long long* ctr = p.counters + ctr_slot((size_t)(q0 / 32) * p.Hq + qh, p.ctr_shift);
    if (threadIdx.x == 0) s_last = arrive(ctr, p.epoch) == (unsigned)(nct - 1);
    __syncthreads();
    if (!s_last) return;
    auto ld = [](const float* a) { return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    for (int i = threadIdx.x; i < 32 * (D / 4); i += W * kWave) {
        const int qm = q0 + i / (D / 4), d0 = i % (D / 4) * 4;
        const int nm = max(base + qm, 0) / chunk + 1;
        if (qm >= p.N || nm == 1) continue;
        const size_t r0 = (size_t)qm * p.max_chunks * p.Hq + qh;
        // eight chunks per round of loads (unconditional: past the count the last chunk's
        // again, with weight 0), each round against its own maximum
        float Mm = -FLT_MAX, lm = 0.f;
        f32x4 am = {0.f, 0.f, 0.f, 0.f};
        for (int c0 = 0; c0 < nm; c0 += 8) {
            float mv[8], lv[8];
            f32x4 av[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const size_t rc = r0 + (size_t)min(c0 + u, nm - 1) * p.Hq;
                mv[u] = ld(p.part_ml + rc * 2);
                lv[u] = ld(p.part_ml + rc * 2 + 1);
#pragma unroll
                for (int r = 0; r < 4; ++r) av[u][r] = ld(p.part_acc + rc * D + d0 + r);
            }
            float Mb = Mm;
#pragma unroll
            for (int u = 0; u < 8; ++u) Mb = fmaxf(Mb, mv[u]);
            const float wb = fast_exp2(Mm - Mb);
            Mm = Mb;
            lm *= wb;
#pragma unroll
            for (int r = 0; r < 4; ++r) am[r] *= wb;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float wk = c0 + u < nm ? fast_exp2(mv[u] - Mb) : 0.f;
                lm = __builtin_fmaf(wk, lv[u], lm);
#pragma unroll
                for (int r = 0; r < 4; ++r) am[r] = __builtin_fmaf(wk, av[u][r], am[r]);
            }
        }
        const float im = lm > 0.f ? 1.0f / lm : 0.f;
        f16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (_Float16)(lm > 0.f ? am[r] * im : 0.f);
        *reinterpret_cast<f16x4*>(static_cast<_Float16*>(p.out) + ((size_t)qm * p.Hq + qh) * D + d0) = o;
    }
    if (threadIdx.x == 0) __hip_atomic_store(ctr, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

#include "gemm_tile.h"

// X range flags (XRange in gemm_decode.h), for every kernel of this code object
// and the 256 x 256 tiles'
__device__ unsigned cima_gemm_status;

// ------------------------------------------------------- prefill GEMM (MFMA)
//
// Y[m, n] (row stride ldy) = X[m, k] . W[n, k]^T: X holds m tokens, W is the
// packed GGUF weight (the engine's lin_gemm, src/models/transformer.rs:
// 618-655, which dequantises W to an f16 slab and runs an f16 GEMM).
// Each stage a workgroup dequantises its weight tile to f16 -- bit-exact
// with the host decoders, so the operand equals the reference's
// dequantised weight -- stages the X tile as f16 in LDS (bf16 -> f16 is
// exact for 2^-17 <= |x| < 65536), and multiplies with f16 MFMA, fp32
// accumulation.  Three kernel bodies: gemm_body_sk16 (16 tokens, here),
// gemm_group (32 to 128 tokens) and gemm_wide (256 tokens), in gemm_tile.h.

// Split-k tiles for up to 16 tokens: a workgroup of 4 RT waves owns 16 RT
// weight rows x 16 tokens; wave w takes the 16-row tile w % RT and the
// k-split w / RT, whose 128-k stages are s = w / RT, w / RT + 4, ...  Lane l
// takes row l % 16 of its tile and dequantises sub-block g = l / 16 of the
// stage straight into its A operand registers; v_mfma_f32_16x16x32_f16
// step q uses elements [8q, 8q+8) of it, so its B fragment is x[32g + 8q,
// +8) of token l % 16, read from the split's activation tile in LDS (the
// split's RT waves stage it together).  The four splits' partial tiles are
// summed through LDS at the end.
//
// Bound by memory round trips, with one or two stages in flight per wave, so
// the order of a stage's instructions counts.  SER: weights and X by
// SerialDeq and f2h2.  EARLY: the loads of the stage PF on go out before the
// barrier of this one.
template <typename D, int XT, int YT, int PF, int RT, bool SER, bool EARLY>
__device__ void gemm_body_sk16(const void* __restrict__ x, const uint8_t* __restrict__ w, void* __restrict__ y,
                               int m, int n, int k, int ldy, const GemmExt& ext) {
    constexpr int ES = XT == XT_F32 ? 4 : 2, KP = 136;  // tile pitch in halves (pads away bank conflicts)
    constexpr int NW = 4 * RT;                           // waves: RT row tiles x 4 k-splits
    constexpr int E = 32 / RT;                           // x elements per lane and stage
    constexpr int XW = E * ES / 16;                      // 16-byte x loads per lane and stage
    __shared__ __align__(16) uint16_t xl[2][4][16 * KP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rt = wave % RT, ks = wave / RT, g = lane >> 4;
    const int r0 = blockIdx.x * (16 * RT), t0 = blockIdx.y * 16;
    const size_t row_bytes = (size_t)(k / D::BE) * D::BB;
    const auto dc = D::ctx(w, ext);
    fmt_init<D>(dc, ext);
    XScan<XT, 64 * NW> xscan;
    // k-split over workgroups (blockIdx.z of ext.ksplit; the host makes the
    // 128-k stages divide evenly): this workgroup's stages [s0, s0 + nk)
    const int ksp = ext.ksplit > 1 ? ext.ksplit : 1;
    const int nk = k / 128 / ksp, s0 = (int)blockIdx.z * nk;
    const int cnt = (nk + 3) >> 2;  // every wave runs cnt steps (a uniform barrier count)
    const uint8_t* wp = w + (size_t)min(r0 + 16 * rt + (lane & 15), n - 1) * row_bytes;
    // this lane's share of the split's x tile: E elements of one token
    const int lt = 64 * rt + lane, xtok = (lt * E) >> 7, xk = (lt * E) & 127;
    const uint8_t* xp = static_cast<const uint8_t*>(x) + ((size_t)min(t0 + xtok, m - 1) * k + xk) * ES;
    struct Stage {
        typename D::Raw wr;
        uint4 xr[XW];
    };
    auto issue = [&](Stage& st, int i) {
        const int s = s0 + min(ks + 4 * i, nk - 1);  // past the split's last stage: re-load the last one
        st.wr = D::load(dc, wp, 4 * s + g);
#pragma unroll
        for (int j = 0; j < XW; j++) st.xr[j] = reinterpret_cast<const uint4*>(xp + (size_t)s * 128 * ES)[j];
    };
    float4_t acc = float4_t{0.f, 0.f, 0.f, 0.f};
    Stage ring[PF];
#pragma unroll
    for (int i = 0; i < PF; i++) issue(ring[i], i);
    auto step = [&](Stage& st, int i, bool next) {
        const int buf = i & 1;
        auto xcvt = [](float lo, float hi) { return SER ? f2h2(lo, hi) : pack_f16(lo, hi); };
        // the lane's activations -> f16 in the split's tile
        uint4* dst = reinterpret_cast<uint4*>(&xl[buf][ks][xtok * KP + xk]);
        if constexpr (XT == XT_F32) {
#pragma unroll
            for (int j = 0; j < XW / 2; j++) {
                const uint4 a = st.xr[2 * j], b = st.xr[2 * j + 1];
                dst[j] = make_uint4(xcvt(__builtin_bit_cast(float, a.x), __builtin_bit_cast(float, a.y)),
                                    xcvt(__builtin_bit_cast(float, a.z), __builtin_bit_cast(float, a.w)),
                                    xcvt(__builtin_bit_cast(float, b.x), __builtin_bit_cast(float, b.y)),
                                    xcvt(__builtin_bit_cast(float, b.z), __builtin_bit_cast(float, b.w)));
            }
        } else {
#pragma unroll
            for (int j = 0; j < XW; j++) {
                const uint32_t v[4] = {st.xr[j].x, st.xr[j].y, st.xr[j].z, st.xr[j].w};
                uint32_t o[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    o[e] = XT == XT_F16 ? v[e]
                                        : xcvt(__builtin_bit_cast(float, v[e] << 16),
                                               __builtin_bit_cast(float, v[e] & 0xffff0000u));
                }
                dst[j] = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
        uint32_t o[16];
        const int jw = 4 * (s0 + min(ks + 4 * i, nk - 1)) + g;
        if constexpr (SER) SerialDeq<D>::deq(dc, st.wr, jw, o);
        else deq<D>(dc, st.wr, wp, jw, o);
        if constexpr (EARLY) {
            __builtin_amdgcn_sched_barrier(0);
            if (next) issue(st, i + PF);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        } else {
            __syncthreads();
            if (next) issue(st, i + PF);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (ks + 4 * i < nk) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const half8_t bv =
                    *reinterpret_cast<const half8_t*>(&xl[buf][ks][(lane & 15) * KP + 32 * g + 8 * q]);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(half8_t, make_uint4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3])), bv,
                    acc, 0, 0, 0);
            }
        }
    };
    int base = 0;
    for (; base + PF <= cnt; base += PF) {
#pragma unroll
        for (int b0 = 0; b0 < PF; b0++) step(ring[b0], base + b0, true);
    }
#pragma unroll
    for (int b0 = 0; b0 < PF - 1; b0++)
        if (base + b0 < cnt) step(ring[b0], base + b0, false);

    xscan.issue(x, m, k, ext.status);  // the range check's loads overlap the split reduction
    // lane l holds D[row 4(l/16) + i][token l%16] of its tile; sum the splits
    __syncthreads();
    float* red = reinterpret_cast<float*>(&xl[0][0][0]);  // [NW waves][256]
#pragma unroll
    for (int i = 0; i < 4; i++) red[wave * 256 + (4 * g + i) * 16 + (lane & 15)] = acc[i];
    __syncthreads();
    for (int o = tid; o < 256 * RT; o += 64 * NW) {
        const int orow = o >> 4, otok = o & 15, ot = orow >> 4, oi = (orow & 15) * 16 + otok;
        const float v = (red[ot * 256 + oi] + red[(RT + ot) * 256 + oi]) +
                        (red[(2 * RT + ot) * 256 + oi] + red[(3 * RT + ot) * 256 + oi]);
        const int row = r0 + orow, tok = t0 + otok;
        if (row < n && tok < m) {
            if (ksp > 1) {
                ext.part[((size_t)blockIdx.z * m + tok) * n + row] = v;  // summed by cima_gemm_ksum_*
            } else {
                const size_t off = (size_t)tok * ldy + row;
                if constexpr (YT == XT_F32) static_cast<float*>(y)[off] = v;
                else static_cast<uint16_t*>(y)[off] = (uint16_t)f2h(v);
            }
        }
    }

    xscan.finish(x, ext.status);
}

// Raw weights in flight per wave of the group tiles: two stages, and at 64
// tokens four where the raw sub-block is small (measured on MI355X, Q4_K,
// 14336x4096 at 64 tokens: 23.2 us; two stages at four waves per SIMD
// instead spill registers: 38.8 us).
template <typename D, int BN>
constexpr int group_pf() { return BN == 64 && sizeof(typename D::Raw) <= 48 ? 4 : 2; }
// Waves per SIMD asked for: 32-token tiles fit four in 128 registers except
// with f32 X or the largest raw sub-blocks.
template <typename D, int BN, int XT>
constexpr int group_occ() { return BN == 32 && XT != XT_F32 && sizeof(typename D::Raw) <= 48 ? 4 : 2; }

// Waves of 32 rows side by side: two (64-row tiles, four k groups), but four
// (128 rows, two k groups) for f32 X at 128 tokens, whose words in flight
// per thread would not fit the registers otherwise.
template <int BN, int XT>
constexpr int group_rg() { return BN == 128 && XT == XT_F32 ? 4 : 2; }

// 32-row 16-token tiles built with SerialDeq, and with part() as _b16l_; which
// one runs follows from k and the workgroups per CU (b16_serial in
// cima_hip.cpp).  part() lets three workgroups share a CU, SerialDeq two.
// The other formats, and f32 X, are no faster with SerialDeq (measured on
// MI355X, 14336x4096 at 16 tokens, cold, us, part() / SerialDeq: Q4_1 16.1 /
// 16.2, Q5_1 16.3 / 18.1, NF4, bf16 X, 16.3 / 21.9).
template <typename D, int XT>
constexpr bool sk16_serial() {
    return XT != XT_F32 && (std::is_same<D, GG<DQ4_K>>::value || std::is_same<D, GG<DQ5_K>>::value ||
                            std::is_same<D, GG<DIQ4_XS>>::value || (std::is_same<D, DNF4>::value && XT == XT_F16));
}

// name: cima_gemm_<fmt>_b<BN>_<x type>_<y type>
// (HIP's second bound is the minimum waves per SIMD: the 16-token tiles
// ask for 4, two 512-thread workgroups per CU, which the compiler then
// schedules for -- measured on MI355X, Q4_K, bf16 X, bit-identical:
// 14336x4096 18.4 -> 17.6 us at 16 tokens)
#define GEMM_KERNEL(FN, D, BN, XT, XN, YT, YN)                                                       \
    extern "C" __global__ __launch_bounds__(512, (BN == 16 ? 4 : BN == 256 ? 2 : group_occ<D, BN, XT>())) void \
    cima_gemm_##FN##_b##BN##_##XN##_##YN(                                                             \
        const void* x, const uint8_t* w, void* y, int m, int n, int k, int ldy, GemmExt ext) {      \
        if constexpr (BN == 16)                                                                       \
            gemm_body_sk16<D, XT, YT, 1, 2, sk16_serial<D, XT>(), false>(x, w, y, m, n, k, ldy, ext); \
        else if constexpr (BN == 256) gemm_wide<D, XT, YT, 2, 2, 2, 4>(x, w, y, m, n, k, ldy, ext);   \
        else \
            gemm_group<D, XT, YT, BN / 32, group_rg<BN, XT>(), 8 / group_rg<BN, XT>(), group_pf<D, BN>()>(x, w, y, m, n, k, ldy, ext); \
    }
#define GEMM_XY(FN, D, BN)                                                    \
    GEMM_KERNEL(FN, D, BN, XT_F32, f32, XT_F32, f32)                          \
    GEMM_KERNEL(FN, D, BN, XT_F16, f16, XT_F32, f32)                          \
    GEMM_KERNEL(FN, D, BN, XT_BF16, bf16, XT_F32, f32)                        \
    GEMM_KERNEL(FN, D, BN, XT_F32, f32, XT_F16, f16)                          \
    GEMM_KERNEL(FN, D, BN, XT_F16, f16, XT_F16, f16)                          \
    GEMM_KERNEL(FN, D, BN, XT_BF16, bf16, XT_F16, f16)
// 16-row split-k tiles (four waves) for weights too narrow to fill the CUs
// with 32-row tiles: the _b16n_ kernels.  Two stages in flight at three
// workgroups per CU where a stage's registers allow it without spilling
// (not for f32 X, eight load words per stage, nor Q6_K, Q5_K and f16
// weights, whose stages are the largest), else one at four
// (measured on MI355X, Q4_K, bf16 X, 16 tokens: 38.8 -> 25.0 us on
// 4096x14336, 12.9 -> 9.2 on 4096x4096).
template <typename D, int XT>
constexpr int sk16n_pf() {
    return (XT != XT_F32 && !std::is_same<D, GG<DQ6_K>>::value && !std::is_same<D, GG<DQ5_K>>::value &&
            !std::is_same<D, DF16>::value)
               ? 2
               : 1;
}
//
// Their next loads go out before the barrier, with the spread decoders
// (measured on MI355X, 16 tokens, us, SerialDeq and loads behind the barrier /
// part() and loads behind / part() and loads before: Q4_K, f16 X, 4096x14336
// 23.9 / 25.1 / 23.1, 4096x4096 8.5 / 8.0 / 7.9; bf16 X 25.7 / 27.9 / 25.8
// and 9.4 / 9.5 / 9.0), but for NF4, whose table lookups are faster in one
// go (f16 X, 4096x14336 21.4 / 27.0 / 27.4, 4096x4096 7.8 / 8.9 / 9.1).
#define GEMM_KERNEL_NARROW(FN, D, XT, XN, YT, YN)                                                   \
    extern "C" __global__ __launch_bounds__(256, (sk16n_pf<D, XT>() == 2 ? 3 : 4)) void            \
    cima_gemm_##FN##_b16n_##XN##_##YN(const void* x, const uint8_t* w, void* y, int m, int n, int k, \
                                      int ldy, GemmExt ext) {                                       \
        constexpr bool nf4 = std::is_same<D, DNF4>::value;                                          \
        gemm_body_sk16<D, XT, YT, sk16n_pf<D, XT>(), 1, nf4, !nf4>(x, w, y, m, n, k, ldy, ext);     \
    }
#define GEMM_XY_NARROW(FN, D)                                                 \
    GEMM_KERNEL_NARROW(FN, D, XT_F32, f32, XT_F32, f32)                       \
    GEMM_KERNEL_NARROW(FN, D, XT_F16, f16, XT_F32, f32)                       \
    GEMM_KERNEL_NARROW(FN, D, XT_BF16, bf16, XT_F32, f32)                     \
    GEMM_KERNEL_NARROW(FN, D, XT_F32, f32, XT_F16, f16)                       \
    GEMM_KERNEL_NARROW(FN, D, XT_F16, f16, XT_F16, f16)                       \
    GEMM_KERNEL_NARROW(FN, D, XT_BF16, bf16, XT_F16, f16)
#define GEMM_KERNEL_LOW(FN, D, XT, XN, YT, YN)                                                      \
    extern "C" __global__ __launch_bounds__(512, 4) void cima_gemm_##FN##_b16l_##XN##_##YN(         \
        const void* x, const uint8_t* w, void* y, int m, int n, int k, int ldy, GemmExt ext) {      \
        static_assert(sk16_serial<D, XT>(), "_b16_ is the same kernel");                            \
        gemm_body_sk16<D, XT, YT, 1, 2, false, false>(x, w, y, m, n, k, ldy, ext);                  \
    }
#define GEMM_XY_LOW(FN, D, XT, XN) GEMM_KERNEL_LOW(FN, D, XT, XN, XT_F32, f32) GEMM_KERNEL_LOW(FN, D, XT, XN, XT_F16, f16)
#define GEMM_LOW(FN, D) GEMM_XY_LOW(FN, D, XT_F16, f16) GEMM_XY_LOW(FN, D, XT_BF16, bf16)
#define GEMM_FMT(FN, D) \
    GEMM_XY(FN, D, 16) GEMM_XY_NARROW(FN, D) GEMM_XY(FN, D, 32) GEMM_XY(FN, D, 64) GEMM_XY(FN, D, 128) GEMM_XY(FN, D, 256)

GEMM_FMT(q8_0, GG<DQ8_0>)
GEMM_FMT(q4_0, GG<DQ4_0>)
GEMM_FMT(q4_1, GG<DQ4_1>)
GEMM_FMT(q5_0, GG<DQ5_0>)
GEMM_FMT(q5_1, GG<DQ5_1>)
GEMM_FMT(q4_k, GG<DQ4_K>)
GEMM_FMT(q5_k, GG<DQ5_K>)
GEMM_FMT(q6_k, GG<DQ6_K>)
GEMM_FMT(iq4_xs, GG<DIQ4_XS>)
// bitsandbytes 4-bit weights decoded in the tiles, and plain f16 weights
GEMM_FMT(nf4, DNF4)
GEMM_FMT(f16w, DF16)
GEMM_LOW(q4_k, GG<DQ4_K>)
GEMM_LOW(q5_k, GG<DQ5_K>)
GEMM_LOW(iq4_xs, GG<DIQ4_XS>)
GEMM_XY_LOW(nf4, DNF4, XT_F16, f16)

// f16 weights of any k (the slab route for k % 64 != 0): one thread per
// output, X rounded to f16 as the tiles round it, fp32 accumulation in k
// order.  Not a fast kernel: it serves shapes no real checkpoint has.
template <int XT, int YT>
__device__ void gemm_small_body(const void* __restrict__ x, const uint16_t* __restrict__ w, void* __restrict__ y,
                                int m, int n, int k, int ldy) {
    const long long o = (long long)blockIdx.x * 256 + threadIdx.x;
    if (o >= (long long)m * n) return;
    const int tok = (int)(o / n), row = (int)(o % n);
    const uint16_t* wr = w + (size_t)row * k;
    float acc = 0.f;
    for (int i = 0; i < k; i++) {
        float xv;
        if constexpr (XT == XT_F32) xv = h2f(f2h(static_cast<const float*>(x)[(size_t)tok * k + i]));
        else if constexpr (XT == XT_F16) xv = h2f(static_cast<const uint16_t*>(x)[(size_t)tok * k + i]);
        else xv = h2f(f2h(__builtin_bit_cast(float, (uint32_t)static_cast<const uint16_t*>(x)[(size_t)tok * k + i] << 16)));
        acc = fmaf(xv, h2f(wr[i]), acc);
    }
    const size_t off = (size_t)tok * ldy + row;
    if constexpr (YT == XT_F32) static_cast<float*>(y)[off] = acc;
    else static_cast<uint16_t*>(y)[off] = (uint16_t)f2h(acc);
}
#define GEMM_SMALL(XT, XN, YT, YN)                                                                      \
    extern "C" __global__ __launch_bounds__(256) void cima_gemm_f16w_small_##XN##_##YN(                 \
        const void* x, const uint16_t* w, void* y, int m, int n, int k, int ldy) {                      \
        gemm_small_body<XT, YT>(x, w, y, m, n, k, ldy);                                                 \
    }
GEMM_SMALL(XT_F32, f32, XT_F32, f32)
GEMM_SMALL(XT_F16, f16, XT_F32, f32)
GEMM_SMALL(XT_BF16, bf16, XT_F32, f32)
GEMM_SMALL(XT_F32, f32, XT_F16, f16)
GEMM_SMALL(XT_F16, f16, XT_F16, f16)
GEMM_SMALL(XT_BF16, bf16, XT_F16, f16)


// Y[tok, row] (row stride ldy) = sum over z < S of part[z][tok][row], z in
// order: the k-split partial tiles, added in one fixed order (results do not
// depend on the launch)
template <int YT>
__device__ void ksum_body(const float* __restrict__ part, void* __restrict__ y, int m, int n, int ldy, int S) {
    const long long o = (long long)blockIdx.x * 256 + threadIdx.x;
    if (o >= (long long)m * n) return;
    const int tok = (int)(o / n), row = (int)(o % n);
    float v = part[o];
    for (int z = 1; z < S; z++) v += part[(size_t)z * m * n + o];
    const size_t off = (size_t)tok * ldy + row;
    if constexpr (YT == XT_F32) static_cast<float*>(y)[off] = v;
    else static_cast<uint16_t*>(y)[off] = (uint16_t)f2h(v);
}
extern "C" __global__ __launch_bounds__(256) void cima_gemm_ksum_f32(const float* part, void* y, int m, int n, int ldy,
                                                                     int S) {
    ksum_body<XT_F32>(part, y, m, n, ldy, S);
}
extern "C" __global__ __launch_bounds__(256) void cima_gemm_ksum_f16(const float* part, void* y, int m, int n, int ldy,
                                                                     int S) {
    ksum_body<XT_F16>(part, y, m, n, ldy, S);
}

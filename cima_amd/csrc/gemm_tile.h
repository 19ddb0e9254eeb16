// Tiles of the prefill GEMM for more than 16 tokens.
#pragma once
#include <utility>

#include "gemm_decode.h"

#define INL __attribute__((always_inline))

// f(integral_constant<0>) ... f(integral_constant<N - 1>): a loop whose index
// is a constant in the body
template <typename F, int... I>
DEV void static_for_seq(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
DEV void static_for(F&& f) {
    static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// Four rows [row, row + 4) of token tok to Y; vec: n is a multiple of 4, so
// a run that starts inside n ends inside it
template <int YT>
DEV void store4(void* y, float4_t o, int tok, int row, int m, int n, int ldy, bool vec) {
    if (tok >= m || row >= n) return;
    const size_t off = (size_t)tok * ldy + row;
    if constexpr (YT == XT_F32) {
        float* d = static_cast<float*>(y) + off;
        if (vec) {
            __builtin_memcpy(d, &o, 16);
        } else {
            static_for<4>([&](auto E) INL { if (row + E < n) d[E] = o[decltype(E)::value]; });
        }
    } else {
        uint16_t* d = static_cast<uint16_t*>(y) + off;
        if (vec) {
            const uint2 u = make_uint2(pack_f16(o[0], o[1]), pack_f16(o[2], o[3]));
            __builtin_memcpy(d, &u, 8);
        } else {
            static_for<4>([&](auto E) INL { if (row + E < n) d[E] = (uint16_t)f2h(o[decltype(E)::value]); });
        }
    }
}

// 16 bytes of X to LDS as f16: eight elements, four of f32
template <int XT>
DEV void store_x(uint16_t* dst, uint4 x) {
    const uint32_t v[4] = {x.x, x.y, x.z, x.w};
    if constexpr (XT == XT_F16) {
        *reinterpret_cast<uint4*>(dst) = x;
    } else if constexpr (XT == XT_BF16) {
        uint32_t o[4];
        static_for<4>([&](auto E) INL {
            o[E] = pack_f16(__builtin_bit_cast(float, v[E] << 16), __builtin_bit_cast(float, v[E] & 0xffff0000u));
        });
        *reinterpret_cast<uint4*>(dst) = make_uint4(o[0], o[1], o[2], o[3]);
    } else {
        *reinterpret_cast<uint2*>(dst) =
            make_uint2(pack_f16(__builtin_bit_cast(float, v[0]), __builtin_bit_cast(float, v[1])),
                       pack_f16(__builtin_bit_cast(float, v[2]), __builtin_bit_cast(float, v[3])));
    }
}

// Group tiles (17 to about 256 tokens): 64 weight rows x T = 32, 64 or 128
// tokens in 8 waves.  Four k groups of two waves take every fourth 64-k
// stage each; a wave owns 32 rows and all T tokens of its group's stages,
// and the groups' partial tiles are added in group order at the end.
//
// Weights never pass through LDS: lane l of a wave takes row l % 32 and
// decodes sub-block h = l / 32 of the stage's two straight into its A
// operand registers, step q of v_mfma_f32_32x32x16_f16 holding elements
// [8q, 8q + 8); the MFMA sums over k in any order as long as A and B agree,
// so its B fragment is x[32h + 8q, +8) of token l % 32, from the group's X
// tile in LDS (f16, rows of 144 bytes: no bank conflicts).
//
// What bounds it: instruction issue, and with few stages per group the first
// loads and the exchange at the end.  One wave issues a vector instruction
// every 8 cycles and two waves on a SIMD one every 4 (measured on MI355X),
// and an MFMA takes 32, so each SIMD needs two waves with at most about six
// other instructions per MFMA; the weights of stage s + 1 and its X words
// are therefore decoded between the MFMAs of stage s, a few instructions
// behind each (sched_barrier keeps them there).  k groups instead of more
// rows give a narrow weight enough waves: 14336 rows are 224 workgroups.
// Measured on MI355X (Q4_K, bf16 X, 14336x4096, cold, us) against tiles of
// 128 rows x 32-64 tokens in four waves that decoded a stage before
// multiplying it: 32 / 64 / 128 tokens 33.5 / 36.2 / 47.5 -> 17.8 / 23.2 /
// 30.7; Q8_0, f16 X: 56.0 / 52.9 / 64.0 -> 22.8 / 28.2 / 35.6; Q6_K 77.1 /
// 86.4 / 95.5 -> 30.6 / 37.1 / 43.8.
template <typename D, int XT, int YT, int TB, int RG, int KG, int PFW>
DEV void gemm_group(const void* __restrict__ x, const uint8_t* __restrict__ w, void* __restrict__ y, int m,
                          int n, int k, int ldy, const GemmExt& ext) {
    // 32-row tiles per wave: one; more rows go to more workgroups (two leave
    // too few registers for two waves per SIMD).  The arrays of one stay
    // arrays: with scalars and references in their place the compiler spills
    // the ring of raw weights (measured on MI355X, 64 x 128 tiles, Q4_K: 2.3
    // times the time).
    constexpr int RA = 1;
    constexpr int BK = 64, KP = BK + 8;          // stage depth and LDS pitch (halves)
    constexpr int T = 32 * TB, BM = 32 * RA * RG;
    constexpr int NT = 64 * RG;                  // threads of a k group
    constexpr int ES = XT == XT_F32 ? 4 : 2, V = 16 / ES, LR = BK / V, RPI = NT / LR, NL = T / RPI;
    static_assert(T % RPI == 0 && NL >= 1, "x tile");
    constexpr int NS = 4 * TB;                   // slots (RA MFMAs each) per stage
    constexpr int XBYTES = KG * 2 * T * KP * 2;
    constexpr int RBYTES = (KG - 1) * BM * T * 4;
    constexpr int LBYTES = XBYTES > RBYTES ? XBYTES : RBYTES;
    __shared__ __align__(16) uint8_t lds[LBYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave % RG, kg = wave / RG, gt = tid - kg * NT;
    const int r0 = blockIdx.x * BM + 32 * RA * rg, t0 = blockIdx.y * T;
    const size_t row_bytes = (size_t)(k / D::BE) * D::BB;
    const auto dc = D::ctx(w, ext);
    fmt_init<D>(dc, ext);
    uint16_t* xl = reinterpret_cast<uint16_t*>(lds) + kg * 2 * T * KP;
    // this workgroup's stages: all of k, or the blockIdx.z-th of ext.ksplit
    // ranges (the host makes them divide evenly)
    const int ksp = ext.ksplit > 1 ? ext.ksplit : 1;
    const int nk = k / BK / ksp, z0 = (int)blockIdx.z * nk, h = lane >> 5;
    const int full = nk / KG;
    XScan<XT, NT * KG> xscan;

    const uint8_t* wp[RA];
#pragma unroll
    for (int a = 0; a < RA; a++) wp[a] = w + (size_t)min(r0 + 32 * a + (lane & 31), n - 1) * row_bytes;
    uint32_t xoff[NL];
    const int xkk = (gt % LR) * V;
    const int xls = (gt / LR) * KP + xkk;
#pragma unroll
    for (int i = 0; i < NL; i++) xoff[i] = (uint32_t)(min(t0 + gt / LR + i * RPI, m - 1) * k + xkk) * ES;
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(x), 0, (int)((uint32_t)m * (uint32_t)k * (uint32_t)ES), 0x00027000);
    auto stage_of = [&](int i) INL { return z0 + min(i * KG + kg, nk - 1); };

    typename D::Raw wr[PFW][RA];
    uint4 xr[NL];
    auto wissue = [&](typename D::Raw (&r)[RA], int i) INL {
        const int s = stage_of(i);
#pragma unroll
        for (int a = 0; a < RA; a++) r[a] = D::load(dc, wp[a], 2 * s + h);
    };
    auto xload = [&](int p, int i) INL {
        xr[p] = __builtin_bit_cast(
            uint4, __builtin_amdgcn_raw_buffer_load_b128(xrs, (int)xoff[p], stage_of(i) * (BK * ES), 0));
    };
    auto xstore = [&](int p, int buf) INL { store_x<XT>(xl + buf * (T * KP) + xls + p * (RPI * KP), xr[p]); };

    float16_t acc[RA][TB];
    static_for<RA * TB>([&](auto I) INL { acc[decltype(I)::value / TB][decltype(I)::value % TB] = float16_t{}; });

    uint32_t av[2][RA][16];
    // stage 0 of the group: X into buffer 0, its weights into av[0]
#pragma unroll
    for (int p = 0; p < NL; p++) xload(p, 0);
#pragma unroll
    for (int i = 0; i < PFW; i++) wissue(wr[i], i);
#pragma unroll
    for (int p = 0; p < NL; p++) {
        xstore(p, 0);
        xload(p, 1);
    }
#pragma unroll
    for (int a = 0; a < RA; a++) deq<D>(dc, wr[0][a], wp[a], 2 * stage_of(0) + h, av[0][a]);
    wissue(wr[0], PFW);
    __syncthreads();

    // One stage: its MFMAs, and between them the weights of the group's next
    // stage, from slot nxt of the ring, and its X into the other buffer
    // (past the last stage the last one is decoded again, unused).
    auto afrag = [&](const uint32_t (&v)[16], int q) INL {
        return __builtin_bit_cast(half8_t, make_uint4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]));
    };
    auto step = [&](int i, auto CUR, typename D::Raw (&nxt_)[1]) INL {
        constexpr int cur = decltype(CUR)::value;
        typename D::Raw& nxt = nxt_[0];
        const uint16_t* src = xl + cur * (T * KP) + (lane & 31) * KP + 32 * h;
        half8_t f[4];
        auto frag = [&](int j) INL {
            return *reinterpret_cast<const half8_t*>(src + (j % TB) * (32 * KP) + 8 * (j / TB));
        };
        f[0] = frag(0);
        f[1] = frag(1);
        f[2] = frag(2);
        const int jn = 2 * stage_of(i + 1) + h;
        const typename D::P pr = D::prep(dc, nxt, wp[0], jn);
        __builtin_amdgcn_sched_barrier(0);
        static_for<NS>([&](auto J) INL {
            constexpr int j = decltype(J)::value, q = j / TB, b = j % TB;
            if constexpr (j + 3 < NS) f[(j + 3) & 3] = frag(j + 3);
            acc[0][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(afrag(av[cur][0], q), f[j & 3], acc[0][b], 0, 0, 0);
            // weight parts and X words due behind this MFMA
            constexpr int p0 = (j * 8 + NS - 1) / NS, p1 = ((j + 1) * 8 + NS - 1) / NS;
            static_for<p1 - p0>([&](auto Q) INL {
                constexpr int p = p0 + decltype(Q)::value;
                D::part(dc, nxt, pr, jn, p, av[cur ^ 1][0][2 * p], av[cur ^ 1][0][2 * p + 1]);
            });
            constexpr int x0 = (j * NL + NS / 2) / NS, x1 = ((j + 1) * NL + NS / 2) / NS;
            static_for<x1 - x0>([&](auto Q) INL {
                constexpr int p = x0 + decltype(Q)::value;
                xstore(p, cur ^ 1);
                xload(p, i + 2);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        wissue(nxt_, i + 1 + PFW);
        __syncthreads();
    };
    static_assert(PFW == 2 || PFW == 4, "ring and buffer parity");
    using std::integral_constant;
    // whole rounds of PFW stages of every group, pipelined
    const int rounds = full / PFW;
    for (int i = 0; i < rounds * PFW; i += PFW)
        static_for<PFW>([&](auto U) INL {
            constexpr int u = decltype(U)::value;
            step(i + u, integral_constant<int, u & 1>{}, wr[(u + 1) % PFW]);
        });
    // the remaining stages one at a time: stage i is in buffer 0 and, its
    // weights, in av[0] (a group past its last stage only joins the barriers)
    for (int i = rounds * PFW; i * KG < nk; i++) {
        if (i * KG + kg < nk) {
            const uint16_t* src = xl + (lane & 31) * KP + 32 * h;
            static_for<NS>([&](auto J) INL {
                constexpr int j = decltype(J)::value, q = j / TB, b = j % TB;
                const half8_t f = *reinterpret_cast<const half8_t*>(src + b * (32 * KP) + 8 * q);
                static_for<RA>([&](auto A) INL {
                    constexpr int a = decltype(A)::value;
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                        __builtin_bit_cast(half8_t, make_uint4(av[0][a][4 * q], av[0][a][4 * q + 1],
                                                               av[0][a][4 * q + 2], av[0][a][4 * q + 3])),
                        f, acc[a][b], 0, 0, 0);
                });
            });
        }
        __syncthreads();
        static_for<NL>([&](auto P) INL { xload(P, i + 1); });
        wissue(wr[0], i + 1);
        static_for<NL>([&](auto P) INL { xstore(P, 0); });
        static_for<RA>([&](auto A) INL { deq<D>(dc, wr[0][A], wp[A], 2 * stage_of(i + 1) + h, av[0][A]); });
        __syncthreads();
    }
    __syncthreads();

    // k groups: group g keeps the row quads v with v % KG == g of every tile
    // and adds the others' partial quads to them in group order
    auto quad = [&](auto B, auto VV) INL {
        constexpr int b = decltype(B)::value, v = decltype(VV)::value;
        return float4_t{acc[0][b][4 * v], acc[0][b][4 * v + 1], acc[0][b][4 * v + 2], acc[0][b][4 * v + 3]};
    };
    // LDS place of quad v of token tile b from group `from`, for its owner
    auto place = [&](int from, int b, int v) INL {
        const int dst = v % KG;
        return reinterpret_cast<float*>(lds) +
               ((((dst * (KG - 1) + (from < dst ? from : from - 1)) * RG + rg) * TB + b) * (4 / KG) + v / KG) * 256 +
               lane * 4;
    };
    static_assert(KG == 2 || KG == 4, "quads divide over the groups");
    static_for<TB>([&](auto B) INL {
        static_for<4>([&](auto VV) INL {
            if (VV % KG != kg) *reinterpret_cast<float4_t*>(place(kg, B, VV)) = quad(B, VV);
        });
    });
    __syncthreads();
    xscan.issue(x, m, k, ext.status);  // the range check's loads overlap the output stores
    const bool vec = (n & 3) == 0;
    // split along k: Y is the partial tiles [ksplit][m][ldy], fp32, summed
    // by cima_gemm_ksum_*
    void* yz = static_cast<uint8_t*>(y) + (size_t)blockIdx.z * m * ldy * (YT == XT_F32 ? 4 : 2);
    static_for<TB>([&](auto B) INL {
        const int tok = t0 + 32 * B + (lane & 31);
        static_for<4>([&](auto VV) INL {
            if (VV % KG != kg) return;
            float4_t o = float4_t{};
            static_for<KG>([&](auto G) INL {
                constexpr int own = decltype(VV)::value % KG, g = decltype(G)::value;
                const float4_t t = g == own ? quad(B, VV) : *reinterpret_cast<const float4_t*>(place(g, B, VV));
                o = g ? o + t : t;
            });
            const int row = r0 + 8 * VV + 4 * h;
            store4<YT>(yz, o, tok, row, m, n, ldy, vec);
        });
    });
    xscan.finish(x, ext.status);
}

// Wide tiles (beyond): 32 RA WR weight rows x 32 TB WC tokens in 8 waves on a
// WR x WC grid, each wave a (32 RA) x (32 TB) tile -- 128 x 256 (RA = TB = 2
// on 2 x 4 waves) or 256 x 256 (RA = 2, TB = 4 on 4 x 2).  Both operands
// go through LDS: every weight is decoded once per workgroup.  X comes in
// 64-k stages, weights in units of U stages, so that a thread decodes
// exactly one 32-element sub-block per unit and neighbouring threads read
// neighbouring sub-blocks of a row.  Both are double-buffered; a unit's
// eight weight parts, the stage's X words and the fragments of the next
// 16-k step are spread between the MFMAs, and the one barrier per stage
// stands before its last step, whose fragments are already in registers.
//
// Bound by instruction issue where decoding is dear (Q4_K, bf16 X, 512
// tokens: 7.8 vector instructions per MFMA, 0.46 of the SIMDs' time their
// issue, 0.34 MFMAs); Q8_0 with f16 X (3.7 per MFMA) by the rounds of
// workgroups: at 2048 tokens on 14336 rows 448 tiles on 256 CUs take two, with
// MFMAs 0.51 of the time.  Measured on MI355X (14336x4096, cold, us) against
// 128 x 128 and 128 x 256 tiles of four waves: Q4_K, bf16 X: 512 tokens
// 100 -> 73 (128 x 256), 2048 tokens 400 -> 260 (256 x 256; 128 x 256: 299);
// Q8_0, f16 X: 122 -> 72 and 434 -> 245.
template <typename D, int XT, int YT, int RA, int TB, int WR, int WC>
DEV void gemm_wide(const void* __restrict__ x, const uint8_t* __restrict__ w, void* __restrict__ y, int m, int n,
                   int k, int ldy, const GemmExt& ext) {
    constexpr int BK = 64, XP = BK + 8;              // X stage depth and LDS pitch (halves)
    constexpr int BM = 32 * RA * WR, T = 32 * TB * WC, NT = 64 * WR * WC;
    constexpr int U = NT / (2 * BM);                 // 64-k stages per weight unit: one sub-block per thread
    constexpr int WK = BK * U, WP = WK + 8;
    static_assert(U * 2 * BM == NT && U >= 1, "one sub-block per thread and unit");
    constexpr int ES = XT == XT_F32 ? 4 : 2, V = 16 / ES, LR = BK / V, RPI = NT / LR, NL = T / RPI;
    static_assert(T % RPI == 0 && NL >= 1, "x tile");
    constexpr int NM = RA * TB;                      // MFMAs per 16-k step
    __shared__ __align__(16) uint16_t wl[2][BM * WP];
    __shared__ __align__(16) uint16_t xl[2][T * XP];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / WC, wc = wave % WC, h = lane >> 5;
    const int r0 = blockIdx.x * BM, t0 = blockIdx.y * T;
    const size_t row_bytes = (size_t)(k / D::BE) * D::BB;
    const auto dc = D::ctx(w, ext);
    fmt_init<D>(dc, ext);
    const int nk = k / BK, nsub = k / 32;

    XScan<XT, NT> xscan;

    // this thread's weight sub-block of a unit and its X words
    const int wrow = tid / (2 * U), wsub = tid % (2 * U);
    const uint8_t* wp = w + (size_t)min(r0 + wrow, n - 1) * row_bytes;
    const int wst = wrow * WP + 32 * wsub;
    uint32_t xoff[NL];
    const int xkk = (tid % LR) * V, xst = (tid / LR) * XP + xkk;
    static_for<NL>([&](auto P) INL { xoff[P] = (uint32_t)(min(t0 + tid / LR + P * RPI, m - 1) * k + xkk) * ES; });
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(x), 0, (int)((uint32_t)m * (uint32_t)k * (uint32_t)ES), 0x00027000);

    typename D::Raw raw[2];
    uint4 xr[NL];
    auto sub_of = [&](int u) INL { return min(2 * U * u + wsub, nsub - 1); };
    auto xload = [&](auto P, int s) INL {
        xr[P] = __builtin_bit_cast(
            uint4, __builtin_amdgcn_raw_buffer_load_b128(xrs, (int)xoff[P], min(s, nk - 1) * (BK * ES), 0));
    };
    auto xstore = [&](auto P, int buf) INL { store_x<XT>(&xl[buf][xst + P * (RPI * XP)], xr[P]); };

    float16_t acc[RA][TB];
    static_for<NM>([&](auto I) INL { acc[I / TB][I % TB] = float16_t{}; });
    half8_t fa[2][RA], fb[2][TB];
    // fragment F (RA of weights, then TB of X) of step q of the unit's stage c
    auto frag = [&](auto F, auto SET, int wbuf, int xbuf, int c, int q) INL {
        constexpr int f = decltype(F)::value, set = decltype(SET)::value;
        if constexpr (f < RA)
            fa[set][f] = *reinterpret_cast<const half8_t*>(
                &wl[wbuf][(32 * RA * wr + 32 * f + (lane & 31)) * WP + BK * c + 16 * q + 8 * h]);
        else
            fb[set][f - RA] = *reinterpret_cast<const half8_t*>(
                &xl[xbuf][(32 * TB * wc + 32 * (f - RA) + (lane & 31)) * XP + 16 * q + 8 * h]);
    };

    // first unit's weights, first stage of X
    static_for<NL>([&](auto P) INL { xload(P, 0); });
    raw[0] = D::load(dc, wp, sub_of(0));
    raw[1] = D::load(dc, wp, sub_of(1));
    static_for<NL>([&](auto P) INL {
        xstore(P, 0);
        xload(P, 1);
    });
    {
        uint32_t o[16];
        deq<D>(dc, raw[0], wp, sub_of(0), o);
        static_for<4>([&](auto I) INL {
            *reinterpret_cast<uint4*>(&wl[0][wst + 8 * I]) = make_uint4(o[4 * I], o[4 * I + 1], o[4 * I + 2], o[4 * I + 3]);
        });
    }
    raw[0] = D::load(dc, wp, sub_of(2));
    __syncthreads();
    static_for<RA + TB>([&](auto F) INL { frag(F, std::integral_constant<int, 0>{}, 0, 0, 0, 0); });

    // Unit u (weights in wl[WB]): its U stages; nxt holds the raw weights of
    // unit u + 1, decoded into the other buffer meanwhile.
    auto unit = [&](int u, auto WB, typename D::Raw& nxt) INL {
        constexpr int wb = decltype(WB)::value;
        constexpr int NSLOT = U * 4 * NM, LAST = NSLOT - NM;  // slots; weights are in LDS before the last step
        const int jn = sub_of(u + 1);
        const typename D::P pr = D::prep(dc, nxt, wp, jn);
        uint32_t o[4];
        __builtin_amdgcn_sched_barrier(0);
        static_for<U * 4>([&](auto QQ) INL {
            constexpr int qq = decltype(QQ)::value, c = qq / 4, q = qq % 4, set = qq & 1;
            constexpr int xb = (U * wb + c) & 1;   // U = 1: buffers alternate with the unit
            const int s = U * u + c;
            if constexpr (q == 3) __syncthreads();
            static_for<NM>([&](auto I) INL {
                constexpr int i = decltype(I)::value, a = i / TB, b = i % TB, slot = qq * NM + i;
                // a fragment of the next step a slot, from this one's start
                if constexpr (i < RA + TB) {
                    std::integral_constant<int, set ^ 1> S;
                    if constexpr (q < 3) frag(I, S, wb, xb, c, q + 1);
                    else if constexpr (c + 1 < U) frag(I, S, wb, xb ^ 1, c + 1, 0);
                    else frag(I, S, wb ^ 1, xb ^ 1, 0, 0);
                }
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[set][a], fb[set][b], acc[a][b], 0, 0, 0);
                // weight parts due: eight over the slots before the last step
                constexpr int p0 = slot < LAST ? slot * 8 / LAST : 8, p1 = slot < LAST ? (slot + 1) * 8 / LAST : 8;
                static_for<p1 - p0>([&](auto G) INL {
                    constexpr int p = p0 + decltype(G)::value;
                    D::part(dc, nxt, pr, jn, p, o[2 * (p & 1)], o[2 * (p & 1) + 1]);
                    if constexpr (p & 1)
                        *reinterpret_cast<uint4*>(&wl[wb ^ 1][wst + 4 * (p - 1)]) = make_uint4(o[0], o[1], o[2], o[3]);
                });
                // X words of the next stage, over this stage's first three steps
                constexpr int xs = (q * NM + i), XL = 3 * NM;
                constexpr int x0 = xs < XL ? (xs * NL + XL / 2) / XL : NL, x1 = xs < XL ? ((xs + 1) * NL + XL / 2) / XL : NL;
                static_for<x1 - x0>([&](auto G) INL {
                    std::integral_constant<int, x0 + decltype(G)::value> P;
                    xstore(P, xb ^ 1);
                    xload(P, s + 2);
                });
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        nxt = D::load(dc, wp, sub_of(u + 3));
    };
    // whole pairs of units, pipelined; what is left (at most 2 U - 1 stages)
    // one stage at a time
    const int pairs = nk / (2 * U);
    for (int u = 0; u < 2 * pairs; u += 2) {
        unit(u, std::integral_constant<int, 0>{}, raw[1]);
        unit(u + 1, std::integral_constant<int, 1>{}, raw[0]);
    }
    // here: unit 2 pairs in wl[0], its first stage in xl[0]
    for (int s = 2 * U * pairs; s < nk; s++) {
        const int c = s % U;
        static_for<4>([&](auto Q) INL {
            static_for<RA + TB>([&](auto F) INL { frag(F, std::integral_constant<int, 0>{}, 0, 0, c, Q); });
            static_for<NM>([&](auto I) INL {
                constexpr int a = decltype(I)::value / TB, b = decltype(I)::value % TB;
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[0][a], fb[0][b], acc[a][b], 0, 0, 0);
            });
        });
        __syncthreads();
        if (s + 1 < nk) {
            static_for<NL>([&](auto P) INL { xload(P, s + 1); });
            static_for<NL>([&](auto P) INL { xstore(P, 0); });
            if (c + 1 == U) {
                const int j = sub_of(s / U + 1);
                raw[0] = D::load(dc, wp, j);
                uint32_t o[16];
                deq<D>(dc, raw[0], wp, j, o);
                static_for<4>([&](auto I) INL {
                    *reinterpret_cast<uint4*>(&wl[0][wst + 8 * I]) =
                        make_uint4(o[4 * I], o[4 * I + 1], o[4 * I + 2], o[4 * I + 3]);
                });
            }
        }
        __syncthreads();
    }

    xscan.issue(x, m, k, ext.status);  // the range check's loads overlap the output stores
    const bool vec = (n & 3) == 0;
    static_for<TB>([&](auto B) INL {
        const int tok = t0 + 32 * TB * wc + 32 * B + (lane & 31);
        static_for<RA>([&](auto A) INL {
            static_for<4>([&](auto VV) INL {
                constexpr int a = decltype(A)::value, b = decltype(B)::value, v = decltype(VV)::value;
                store4<YT>(y, float4_t{acc[a][b][4 * v], acc[a][b][4 * v + 1], acc[a][b][4 * v + 2], acc[a][b][4 * v + 3]},
                       tok, r0 + 32 * RA * wr + 32 * a + 8 * v + 4 * h, m, n, ldy, vec);
            });
        });
    });
    xscan.finish(x, ext.status);
}

// Weight decoders, per-call operands and the X range check shared by the
// prefill GEMM kernels (gguf_gemm.hip, gguf_gemm_wide.hip).
#pragma once
#include <type_traits>

#include "gguf_formats.h"

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
enum { XT_F32 = 0, XT_F16 = 1, XT_BF16 = 2 };

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

// two fp32 -> packed f16 bits, v_cvt_pk_f16_f32.  Unlike f2h2 (which hides
// its operands from the compiler) this costs no wait states between the
// arithmetic and the conversion; the vector conversion is a legal operation
// on gfx950, so LLVM keeps the fp32 result and does not fold the pair into
// v_fma_mixlo / mixhi, which would skip its rounding.
DEV uint32_t pack_f16(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t){lo, hi}, half2_t));
}

// Integer quants as f16.  The bits of a small integer u are the f16
// subnormal u 2^-24, exactly; v_fma_mix_f32 takes either half of a word as
// its f16 operand, so s24 = s 2^24 gives fma(s, u, t) without converting u
// to fp32 first: per four quants two byte permutes, four fused
// multiply-adds and two packed conversions (v_cvt_f32_ubyte took two more).
// Bytes 0..3 of v are u; fp32 results s u + t, rounded once where s u is
// exact, then to f16.
DEV void affine4(uint32_t v, float s24, float t, uint32_t& lo, uint32_t& hi) {
    const half2_t a = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, v, 0x0c010c00u));
    const half2_t b = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, v, 0x0c030c02u));
    // the four products first: a conversion right behind the product it
    // takes would wait a state
    const float f0 = __builtin_fmaf((float)a[0], s24, t), f1 = __builtin_fmaf((float)a[1], s24, t);
    const float f2 = __builtin_fmaf((float)b[0], s24, t), f3 = __builtin_fmaf((float)b[1], s24, t);
    lo = pack_f16(f0, f1);
    hi = pack_f16(f2, f3);
}
// f16(d (u - c)) of the bytes u of v, d a pair of equal f16 scales: byte u
// under 0x64 is the f16 1024 + u, so u - c is one exact packed subtraction
// and the packed product rounds once, like fp32 d (u - c) -- exact -- then
// rounded to f16.
DEV void scaled4(uint32_t v, half2_t d, float c, uint32_t& lo, uint32_t& hi) {
    const half2_t o = {(_Float16)(1024.f + c), (_Float16)(1024.f + c)};
    const half2_t a = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u));
    const half2_t b = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u));
    lo = __builtin_bit_cast(uint32_t, (a - o) * d);
    hi = __builtin_bit_cast(uint32_t, (b - o) * d);
}

// Block bytes at 2-byte alignment, read as aligned words: a 16-byte load
// at 2 mod 4 occupies the address unit about 1.7 times as long as an
// aligned one (measured on MI355X, one row per lane), and the tiles issue
// several per stage and wave.  The words from p & ~3 on hold the bytes from
// p; sel is the byte permute that extracts word i of the run that starts
// 2 bytes after p (after a leading f16) from words i and i + 1, or of the
// run at p itself.
DEV const uint32_t* word_of(const uint8_t* p) {
    return reinterpret_cast<const uint32_t*>(p - (reinterpret_cast<uintptr_t>(p) & 2));
}
DEV bool word_odd(const uint8_t* p) { return (reinterpret_cast<uintptr_t>(p) & 2) != 0; }
DEV uint32_t sel_after2(bool odd) { return odd ? 0x07060504u : 0x05040302u; }  // bytes p + 2 ..
DEV uint32_t sel_at(bool odd) { return odd ? 0x05040302u : 0x03020100u; }      // bytes p ..
DEV half2_t lead_pair(uint32_t w0, bool odd) {  // the f16 at p, twice
    return __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, w0, odd ? 0x03020302u : 0x01000100u));
}
DEV uint4 ldw4(const uint32_t* p) {
    uint4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 4), 16);
    return v;
}

DEV void ldw9(const uint32_t* p, uint32_t (&o)[9]) {
    const uint4 a = ldw4(p), b = ldw4(p + 4);
    o[0] = a.x, o[1] = a.y, o[2] = a.z, o[3] = a.w;
    o[4] = b.x, o[5] = b.y, o[6] = b.z, o[7] = b.w;
    o[8] = p[8];
}

// quants of elements [4i, 4i + 4) of a 32-element block whose byte j holds
// element j (low nibble) and j + 16 (high): q[i % 4]'s nibbles
DEV uint32_t nibbles(uint32_t q, int i) { return (i < 4 ? q : q >> 4) & 0x0F0F0F0Fu; }

// Scales of sub-block s of a Q4_K / Q5_K header: d sc as s24 for quants in
// the low nibbles (s even) or left in the high ones (odd, sixteen times the
// quant), the nibble mask of the same, and dmin m.
struct K45 {
    float s24, t;
    uint32_t mask;
};
DEV K45 q4k_affine(const uint4& h, int s) {
    // all eight 6-bit pairs a byte each, then byte s of both
    const uint32_t sclo = h.y & 0x3F3F3F3Fu, mlo = h.z & 0x3F3F3F3Fu;
    const uint32_t schi = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
    const uint32_t mhi = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
    const uint32_t sel = 0x0c0c0c00u | (uint32_t)s;
    const uint32_t sc = __builtin_amdgcn_perm(schi, sclo, sel), m = __builtin_amdgcn_perm(mhi, mlo, sel);
    const bool hi = s & 1;
    const float ds = h2f(h.x & 0xffffu) * (float)sc;
    return K45{ds * (hi ? 0x1p20f : 0x1p24f), -(h2f(h.x >> 16) * (float)m),
               hi ? 0xF0F0F0F0u : 0x0F0F0F0Fu};
}

// A decoder D turns sub-block j of a row -- 32 contiguous elements [32j,
// 32j + 32) -- into f16 bits, 2 per dword: load() reads its packed bytes,
// prep() its scales, part(i) gives elements [4i, 4i + 4), so that a tile can
// spread the eight parts between its matrix instructions; deq() is all of
// them.
//
// The values are those of the host decoders (where one multiplies only,
// d * (q - c), fma(d, q, -c d) is the same value, though a zero weight may
// come out +0 where the decoder gives -0 -- a difference no product sum
// shows)
struct DQ8_0 {
    static constexpr int BE = 32, BB = 34;
    struct Raw { uint4 a, b; uint32_t c; };  // words of the block's 34 bytes
    DEV static Raw load(const uint8_t* row, int j) {
        const uint32_t* p = word_of(row + (size_t)j * 34);
        return Raw{ldw4(p), ldw4(p + 4), p[8]};
    }
    struct P { half2_t d; uint32_t sel; };
    DEV static P prep(const Raw& r, bool odd) { return P{lead_pair(r.a.x, odd), sel_after2(odd)}; }
    DEV static void part(const Raw& r, const P& p, int, int i, uint32_t& lo, uint32_t& hi) {
        const uint32_t w[9] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w, r.c};
        scaled4(__builtin_amdgcn_perm(w[i + 1], w[i], p.sel) ^ 0x80808080u, p.d, 128.f, lo, hi);
    }
};
struct DQ4_0 {
    static constexpr int BE = 32, BB = 18;
    struct Raw { uint4 a; uint32_t c; };
    DEV static Raw load(const uint8_t* row, int j) {
        const uint32_t* p = word_of(row + (size_t)j * 18);
        return Raw{ldw4(p), p[4]};
    }
    struct P { half2_t d; uint32_t sel; };
    DEV static P prep(const Raw& r, bool odd) { return P{lead_pair(r.a.x, odd), sel_after2(odd)}; }
    DEV static void part(const Raw& r, const P& p, int, int i, uint32_t& lo, uint32_t& hi) {
        const uint32_t w[5] = {r.a.x, r.a.y, r.a.z, r.a.w, r.c};
        scaled4(nibbles(__builtin_amdgcn_perm(w[(i & 3) + 1], w[i & 3], p.sel), i), p.d, 8.f, lo, hi);
    }
};
struct DQ4_1 {
    static constexpr int BE = 32, BB = 20;
    using Raw = FQ4_1::Raw;
    DEV static Raw load(const uint8_t* row, int j) { return FQ4_1::load(row, j); }
    struct P { float s24, m; };
    DEV static P prep(const Raw& r, bool) { return P{h2f(r.dm & 0xffffu) * 0x1p24f, h2f(r.dm >> 16)}; }
    DEV static void part(const Raw& r, const P& p, int, int i, uint32_t& lo, uint32_t& hi) {
        // d q + m: the product is exact, the sum rounded once
        const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        affine4(nibbles(q[i & 3], i), p.s24, p.m, lo, hi);
    }
};
struct DQ5_0 {
    static constexpr int BE = 32, BB = 22;
    struct Raw { uint4 a; uint2 c; };
    DEV static Raw load(const uint8_t* row, int j) {
        const uint32_t* p = word_of(row + (size_t)j * 22);
        return Raw{ldw4(p), make_uint2(p[4], p[5])};
    }
    struct P { half2_t d; uint32_t sel, qh; };
    DEV static P prep(const Raw& r, bool odd) {
        const uint32_t sel = sel_after2(odd);
        return P{lead_pair(r.a.x, odd), sel, __builtin_amdgcn_perm(r.a.y, r.a.x, sel)};
    }
    DEV static void part(const Raw& r, const P& p, int, int i, uint32_t& lo, uint32_t& hi) {
        // elements [4i, 4i + 4): their 5th bits are bits 4i.. of qh
        const uint32_t w[5] = {r.a.y, r.a.z, r.a.w, r.c.x, r.c.y};
        const uint32_t q = nibbles(__builtin_amdgcn_perm(w[(i & 3) + 1], w[i & 3], p.sel), i);
        scaled4(q | spread4((p.qh >> (4 * i)) & 0xFu), p.d, 16.f, lo, hi);
    }
};
struct DQ5_1 {
    static constexpr int BE = 32, BB = 24;
    using Raw = FQ5_1::Raw;
    DEV static Raw load(const uint8_t* row, int j) { return FQ5_1::load(row, j); }
    struct P { float s24, m; };
    DEV static P prep(const Raw& r, bool) { return P{h2f(r.dm & 0xffffu) * 0x1p24f, h2f(r.dm >> 16)}; }
    DEV static void part(const Raw& r, const P& p, int, int i, uint32_t& lo, uint32_t& hi) {
        const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        affine4(nibbles(q[i & 3], i) | spread4((r.qh >> (4 * i)) & 0xFu), p.s24, p.m, lo, hi);
    }
};
// sub-block j: super-block j/8, s = j%8 -> chunk c = s/2 of Q4_K's nibble
// layout (low nibbles if s is even) with 5th bits = bit s of qh[l]
struct DQ5_K {
    static constexpr int BE = 256, BB = 176;
    struct Raw { uint4 h, q0, q1, qh0, qh1; };
    DEV static Raw load(const uint8_t* row, int j) {
        const uint8_t* blk = row + (size_t)(j >> 3) * 176;
        const int c = (j & 7) >> 1;
        Raw r;
        r.h = ld16a(blk);
        r.qh0 = ld16a(blk + 16);
        r.qh1 = ld16a(blk + 32);
        r.q0 = ld16a(blk + 48 + 32 * c);
        r.q1 = ld16a(blk + 64 + 32 * c);
        return r;
    }
    struct P { K45 k; };
    DEV static P prep(const Raw& r, int j, bool) {
        // the 5th bit joins the quant as a byte value of its own, so high
        // nibbles are shifted down here
        P p{q4k_affine(r.h, j & 7)};
        if (j & 1) p.k.s24 *= 16.f;
        return p;
    }
    DEV static void part(const Raw& r, const P& p, int j, int i, uint32_t& lo, uint32_t& hi) {
        const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        const uint32_t h[8] = {r.qh0.x, r.qh0.y, r.qh0.z, r.qh0.w, r.qh1.x, r.qh1.y, r.qh1.z, r.qh1.w};
        const uint32_t n = ((q[i] >> (4 * (j & 1))) & 0x0F0F0F0Fu) | (((h[i] >> (j & 7)) & 0x01010101u) << 4);
        affine4(n, p.k.s24, p.k.t, lo, hi);  // (d sc) q5 exact; one rounding
    }
};
// sub-block j: super-block j/8, ib = j%8: codebook values of qs[16 ib, +16)
struct DIQ4_XS {
    static constexpr int BE = 256, BB = 136;
    using Raw = FIQ4_XS::Raw;
    DEV static Raw load(const uint8_t* row, int j) { return FIQ4_XS::load(row, j); }
    struct P { float s24, t; };
    DEV static P prep(const Raw& r, int j, bool) {
        const float dl = iq4xs_dl(r.hdr, j & 7);
        return P{dl * 0x1p24f, -128.f * dl};
    }
    DEV static void part(const Raw& r, const P& p, int, int i, uint32_t& lo, uint32_t& hi) {
        const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        affine4(iq4nl_bytes(nibbles(q[i & 3], i)) ^ 0x80808080u, p.s24, p.t, lo, hi);
    }
};
// sub-block j: super-block j/8, sub s = j%8 -> qs bytes 32*(s/2) + [0,32),
// low nibbles if s is even, high if odd
struct DQ4_K {
    static constexpr int BE = 256, BB = 144;
    struct Raw { uint4 h, q0, q1; };
    DEV static Raw load(const uint8_t* row, int j) {
        const uint8_t* blk = row + (size_t)(j >> 3) * 144;
        const int c = (j & 7) >> 1;
        Raw r;
        r.h = ld16a(blk);
        r.q0 = ld16a(blk + 16 + 32 * c);
        r.q1 = ld16a(blk + 32 + 32 * c);
        return r;
    }
    struct P { K45 k; };
    DEV static P prep(const Raw& r, int j, bool) { return P{q4k_affine(r.h, j & 7)}; }
    DEV static void part(const Raw& r, const P& p, int, int i, uint32_t& lo, uint32_t& hi) {
        const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        // (d*sc)*q is exact, so the subtraction is the only fp32 rounding --
        // and a fused multiply-add rounds exactly there too
        affine4(q[i] & p.k.mask, p.k.s24, p.k.t, lo, hi);
    }
};
// sub-block j: super-block j/8, r = j%8 -> half h = r/4, group g = r%4:
// l in [0,32) takes nibble (g<2 low, else high) of ql[64h + 32(g&1) + l],
// bits 2g..2g+1 of qh[32h + l], scale sc[8h + l/16 + 2g]
struct DQ6_K {
    static constexpr int BE = 256, BB = 210;
    struct Raw { uint32_t a[9], h[9], scd; };
    DEV static Raw load(const uint8_t* row, int j) {
        const uint8_t* blk = row + (size_t)(j >> 3) * 210;
        const int hh = (j & 7) >> 2, g = j & 3;
        // the last word of a run only holds bytes of it where p is odd, and
        // reading past it stays inside the block (scales and d follow)
        const uint32_t* a = word_of(blk + 64 * hh + 32 * (g & 1));
        const uint32_t* h = word_of(blk + 128 + 32 * hh);
        Raw r;
        ldw9(a, r.a);
        ldw9(h, r.h);
        // sc[8h + 2g], sc[8h + 2g + 1], d
        r.scd = ld2(blk + 192 + 8 * hh + 2 * g) | (ld2(blk + 208) << 16);
        return r;
    }
    struct P { float s0, s1; uint32_t sel; };
    DEV static P prep(const Raw& r, int, bool odd) {
        const float d = h2f(r.scd >> 16) * 0x1p24f;
        return P{d * (float)(int8_t)(r.scd & 0xff), d * (float)(int8_t)((r.scd >> 8) & 0xff), sel_at(odd)};
    }
    DEV static void part(const Raw& r, const P& p, int j, int i, uint32_t& lo, uint32_t& hi) {
        const int g = j & 3;
        const uint32_t av = __builtin_amdgcn_perm(r.a[i + 1], r.a[i], p.sel);
        const uint32_t hv = __builtin_amdgcn_perm(r.h[i + 1], r.h[i], p.sel);
        // ds (u - 32) rounded once, as fma(ds, u, -32 ds) rounds it
        const float s = i < 4 ? p.s0 : p.s1;
        const uint32_t q = ((av >> (g < 2 ? 0 : 4)) & 0x0F0F0F0Fu) | (((hv >> (2 * g)) & 0x03030303u) << 4);
        affine4(q, s, s * -0x1p-19f, lo, hi);
    }
};

// Per-call operands of formats that need more than the packed weight:
// bitsandbytes 4-bit (absmax per `bsz` elements, the 16-entry codebook).
// The GGUF formats ignore them.
struct GemmExt {
    const float* absmax;
    const float* qmap;
    long long bsz;   // elements per absmax entry
    int bs_shift;    // log2(bsz) when bsz is a power of two, else -1
    unsigned* status;  // X range flags (cima_gemm_status), OR-ed in
    float* part;       // k-split partial tiles, [ksplit][m][n] fp32
    int ksplit;        // workgroups along k (blockIdx.z); 1 = Y written directly
};

// X range report.  The tiles round X to f16.  That is exact for bf16 values
// of 2^-17 <= |x| < 65536 (and zero); larger ones become +-inf, and smaller
// nonzero ones may lose bits (f16 subnormals step by 2^-24).  f32 X is
// rounded anyway (the 1e-3 bar), but |x| >= 65520 becomes inf too.  Every
// workgroup checks its own 1/(grid size) share of X once (XScan: a few
// 16-byte words per thread) and ORs flags into a word of device memory
// (cima_gemm_status in gguf_gemm.hip), which the host reads back on
// request (cima_hip_gemm_status): bit 0 = values beyond f16's range, or not
// finite; bit 1 = nonzero bf16 values below 2^-17.  The loads go out after
// the main loop, beside the output stores, and are checked last.  Measured
// on MI355X (Q4_K 14336x4096, bf16 X), against no check: +0.8-1.2 / +0.9 /
// +0.5 / +0.5 / +1-2 us at 16 / 32 / 64 / 128 / 512 tokens (1-6 %);
// checked before the main loop instead it cost 1.3-2.6 us at 16-32
// tokens, and inside the tiles' own conversions every stage (+1170 VALU
// instructions in the 256-token tile, 102 -> 150 us at 512 tokens).
struct XRange {
    // one word of flags, two bf16 halves at a time (magnitudes h <= 0x7fff,
    // so the additions below never carry out of a half): bit 15 of a half
    // <- h >= 0x4780 (65536: beyond f16, or inf / NaN); bit 14 <- 0 < h <
    // 0x3700 (below 2^-17); f32: bit 31 <- |x| >= 65520
    uint32_t acc = 0;
    DEV void bf16(uint32_t w) {
        const uint32_t a = w & 0x7fff7fffu;
        acc |= ((a + 0x38803880u) & 0x80008000u) | ((~(a + 0x49004900u) & (a + 0x7fff7fffu) & 0x80008000u) >> 1);
    }
    DEV void f32(uint32_t w) { acc |= ((w & 0x7fffffffu) + 0x38801000u) & 0x80000000u; }
    template <int XT>
    DEV void add(uint4 v) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (XT == XT_BF16) bf16(w[i]);
            else f32(w[i]);
        }
    }
    DEV void report(unsigned* st) const {
        const unsigned long long bo = __ballot((acc & 0x80008000u) != 0), bt = __ballot((acc & 0x40004000u) != 0);
        if ((bo | bt) && (threadIdx.x & 63) == 0 && st) atomicOr(st, (bo ? 1u : 0u) | (bt ? 2u : 0u));
    }
};

// This workgroup's share of X for the range check: words [w0, we) of X's
// 16-byte words, thread t taking w0 + t + T j.  issue() loads the first NB
// per thread, unconditionally inside a uniform branch (lanes past the share
// repeat its last word, which their wave's request coalesces; clamped to
// one word of X for every workgroup instead, 448 workgroups queued on one
// L2 line: +2 us at 16 tokens), so that the loads stay in flight beside the
// output stores; finish() checks them (and, for large X, the rest, batch by
// batch) and reports.  Nothing for f16 X.
template <int XT, int T>  // T: threads per workgroup (a constant: reading blockDim is a load, and a wait)
struct XScan {
    static constexpr int NB = 4;
    uint4 v[NB];
    long long w0 = 0, we = 0;
    DEV void issue(const void* x, int m, int k, const unsigned* st) {
        if constexpr (XT != XT_F16) {
            if (!st) return;  // uniform: a null status word switches the check off
            const long long nw = (long long)m * k * (XT == XT_F32 ? 4 : 2) / 16;
            const long long nwg = (long long)gridDim.x * gridDim.y * gridDim.z;
            const long long per = (nw + nwg - 1) / nwg;
            w0 = (((long long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * per;
            we = min(w0 + per, nw);
            const uint4* p = static_cast<const uint4*>(x);
            const long long last = max(we - 1, 0LL);
#pragma unroll
            for (int j = 0; j < NB; j++) {
                v[j] = make_uint4(0, 0, 0, 0);
                if (w0 + (long long)T * j < we) v[j] = p[min(w0 + threadIdx.x + (long long)T * j, last)];
            }
        }
    }
    DEV void finish(const void* x, unsigned* st) const {
        if constexpr (XT != XT_F16) {
            if (!st) return;
            XRange rg;
            const uint4* p = static_cast<const uint4*>(x);
#pragma unroll
            for (int j = 0; j < NB; j++) rg.add<XT>(v[j]);
            for (long long i = w0 + threadIdx.x + (long long)T * NB; i < we; i += T) rg.add<XT>(p[i]);
            rg.report(st);
        }
    }
};

// The tile bodies call D::ctx / init / load / prep / part with a per-call context;
// GG adapts the context-free GGUF decoders above.
template <typename DQ>
struct GG {
    static constexpr int BE = DQ::BE, BB = DQ::BB;
    using Raw = typename DQ::Raw;
    struct Ctx {};
    DEV static Ctx ctx(const uint8_t*, const GemmExt&) { return Ctx{}; }
    DEV static void init(const Ctx&) {}
    DEV static Raw load(const Ctx&, const uint8_t* row, int j) { return DQ::load(row, j); }
    using P = typename DQ::P;
    // odd: sub-block j starts 2 bytes past a word boundary (known from its
    // address, which the formats read at 2-byte alignment use)
    DEV static P prep(const Ctx&, const Raw& r, const uint8_t* row, int j) {
        const bool odd = word_odd(row + (size_t)(j / (BE / 32)) * BB);
        if constexpr (BE == 256) return DQ::prep(r, j, odd);
        else return DQ::prep(r, odd);
    }
    DEV static void part(const Ctx&, const Raw& r, const P& p, int j, int i, uint32_t& lo, uint32_t& hi) {
        DQ::part(r, p, j, i, lo, hi);
    }
};

// bitsandbytes NF4 / FP4 (src/quant.rs:18-70): a row is k/2 packed bytes,
// element 2i in the HIGH nibble of byte i; sub-block j of a row is 16
// bytes, and its 32 elements share one absmax (bsz % 32 == 0, k % 32 ==
// 0, checked on the host).  The value is f16(code[nib] * absmax): one fp32
// product rounded once to nearest even, the decode of dequant_host
// (src/quant.rs:401-437) and k_nf4_dequant (src/kernels.cu:320-329), so the
// MFMA operand equals the reference's decoded f16 weight.  The codebook
// sits in LDS (16 words in 16 banks: lanes never conflict).
struct DNF4 {
    static constexpr int BE = 32, BB = 16;
    struct Raw { uint4 q; float a; };
    struct Ctx {
        const uint8_t* base;
        const float* absmax;
        const float* code;
        long long bsz;
        int bs_shift;
    };
    DEV static Ctx ctx(const uint8_t* w, const GemmExt& e) {
        __shared__ float code[16];
        return Ctx{w, e.absmax, code, e.bsz, e.bs_shift};
    }
    // every thread of the workgroup calls it before its first deq
    DEV static void init(const Ctx& c, const float* qmap) {
        if (threadIdx.x < 16) const_cast<float*>(c.code)[threadIdx.x] = qmap[threadIdx.x];
        __syncthreads();
    }
    DEV static Raw load(const Ctx& c, const uint8_t* row, int j) {
        Raw r;
        r.q = *reinterpret_cast<const uint4*>(row + 16 * j);
        const long long e = (long long)(row - c.base) * 2 + 32 * j;  // flat index of the first element
        r.a = c.absmax[c.bs_shift >= 0 ? (e >> c.bs_shift) : (e / c.bsz)];
        return r;
    }
    struct P {};
    DEV static P prep(const Ctx&, const Raw&, const uint8_t*, int) { return P{}; }
    DEV static void part(const Ctx& c, const Raw& r, const P&, int, int i, uint32_t& lo, uint32_t& hi) {
        const uint32_t w[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        const uint32_t v = w[i >> 1] >> (16 * (i & 1)), b0 = v & 0xFFu, b1 = (v >> 8) & 0xFFu;
        lo = pack_f16(c.code[b0 >> 4] * r.a, c.code[b0 & 0xFu] * r.a);
        hi = pack_f16(c.code[b1 >> 4] * r.a, c.code[b1 & 0xFu] * r.a);
    }
};

// f16 weights as they stand (a row is k f16 values): the tile bodies as a
// plain f16 GEMM, for bitsandbytes shapes the fused decoder does not take,
// decoded into the caller's slab first
struct DF16 {
    static constexpr int BE = 32, BB = 64;
    struct Raw { uint4 a[4]; };
    struct Ctx {};
    DEV static Ctx ctx(const uint8_t*, const GemmExt&) { return Ctx{}; }
    DEV static void init(const Ctx&) {}
    DEV static Raw load(const Ctx&, const uint8_t* row, int j) {
        Raw r;
        const uint4* p = reinterpret_cast<const uint4*>(row + 64 * j);
#pragma unroll
        for (int i = 0; i < 4; i++) r.a[i] = p[i];
        return r;
    }
    struct P {};
    DEV static P prep(const Ctx&, const Raw&, const uint8_t*, int) { return P{}; }
    DEV static void part(const Ctx&, const Raw& r, const P&, int, int i, uint32_t& lo, uint32_t& hi) {
        lo = i & 1 ? r.a[i >> 1].z : r.a[i >> 1].x;
        hi = i & 1 ? r.a[i >> 1].w : r.a[i >> 1].y;
    }
};

// the whole sub-block at once
template <typename D>
DEV void deq(const typename D::Ctx& c, const typename D::Raw& r, const uint8_t* row, int j, uint32_t (&o)[16]) {
    const typename D::P p = D::prep(c, r, row, j);
#pragma unroll
    for (int i = 0; i < 8; i++) D::part(c, r, p, j, i, o[2 * i], o[2 * i + 1]);
}

// The whole sub-block by byte conversions (v_cvt_f32_ubyte) and f2h2, whose
// operands the compiler does not see through: more instructions than part(),
// the same bits.  The 16-token tiles wait on memory rather than on
// instruction issue, and for these formats some of them are faster this way
// (sk16_serial in gguf_gemm.hip).
template <typename D>
struct SerialDeq;
template <>
struct SerialDeq<GG<DQ4_K>> {
    DEV static void deq(const GG<DQ4_K>::Ctx&, const DQ4_K::Raw& r, int j, uint32_t (&o)[16]) {
        uint32_t sc0, m0, sc1, m1;
        q4k_scales(r.h, (j & 7) >> 1, sc0, m0, sc1, m1);
        const bool hi = j & 1;
        const float ds = h2f(r.h.x & 0xffffu) * (float)(hi ? sc1 : sc0), mm = h2f(r.h.x >> 16) * (float)(hi ? m1 : m0);
        const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        const int sh = hi ? 4 : 0;
#pragma unroll
        for (int i = 0; i < 8; i++) bytes_affine((q[i] >> sh) & 0x0F0F0F0Fu, ds, -mm, o[2 * i], o[2 * i + 1]);
    }
};
template <>
struct SerialDeq<GG<DQ5_K>> {
    DEV static void deq(const GG<DQ5_K>::Ctx&, const DQ5_K::Raw& r, int j, uint32_t (&o)[16]) {
        const int s = j & 7;
        uint32_t sc0, m0, sc1, m1;
        q4k_scales(r.h, s >> 1, sc0, m0, sc1, m1);
        const bool hi = s & 1;
        const float ds = h2f(r.h.x & 0xffffu) * (float)(hi ? sc1 : sc0), mm = h2f(r.h.x >> 16) * (float)(hi ? m1 : m0);
        const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        const uint32_t h[8] = {r.qh0.x, r.qh0.y, r.qh0.z, r.qh0.w, r.qh1.x, r.qh1.y, r.qh1.z, r.qh1.w};
        const int sh = hi ? 4 : 0;
#pragma unroll
        for (int i = 0; i < 8; i++)
            bytes_affine(((q[i] >> sh) & 0x0F0F0F0Fu) | (((h[i] >> s) & 0x01010101u) << 4), ds, -mm, o[2 * i],
                         o[2 * i + 1]);
    }
};
template <>
struct SerialDeq<GG<DIQ4_XS>> {
    DEV static void deq(const GG<DIQ4_XS>::Ctx&, const DIQ4_XS::Raw& r, int j, uint32_t (&o)[16]) {
        const float dl = iq4xs_dl(r.hdr, j & 7);
        const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            bytes_affine(iq4nl_bytes(q[i] & 0x0F0F0F0Fu) ^ 0x80808080u, dl, -128.f * dl, o[2 * i], o[2 * i + 1]);
            bytes_affine(iq4nl_bytes((q[i] >> 4) & 0x0F0F0F0Fu) ^ 0x80808080u, dl, -128.f * dl, o[8 + 2 * i],
                         o[8 + 2 * i + 1]);
        }
    }
};
template <>
struct SerialDeq<DNF4> {
    DEV static void deq(const DNF4::Ctx& c, const DNF4::Raw& r, int, uint32_t (&o)[16]) {
        const uint32_t w[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const uint32_t byte = (w[i] >> (8 * b)) & 0xFFu;
                o[4 * i + b] = f2h2(c.code[byte >> 4] * r.a, c.code[byte & 0xFu] * r.a);
            }
    }
};

// D::init with the codebook for DNF4, nothing for the others
template <typename D>
DEV void fmt_init(const typename D::Ctx& c, const GemmExt& e) {
    if constexpr (std::is_same<D, DNF4>::value) D::init(c, e.qmap);
    else D::init(c);
}

// Newton-Schulz phase launches on 128 x 128 tiles (gfx950): the operations of ns_phase_kernel for
// launches whose 256 x 256 tiles would leave most of the chip idle or spend it on padding.
//
// A 256 x 256 tile holds a CU for K / 32 * ~0.45 us plus about 14 us of launch, prologue and epilogue. A group of
// mid-size matrices has fewer of them than CUs (48 matrices of 384 x 1536: 144 in a symmetric
// product, of which 384 -> 512 padding is 44%), so its 18 dependent launches wait for one tile's
// latency each. Here a block of 256 threads computes 128 x 128, two blocks to a CU: four times the
// tiles, a quarter of the work and of the staging in each, no padding at multiples of 128. The price
// is LDS traffic: each wave's 64 x 64 reads 1 KB of fragments per MFMA, the whole 128 B per clock
// of a CU at the full MFMA rate, so on launches that fill the chip anyway the 256 x 256 engine is
// faster (plan_tiles in thorn_abi.hip chooses one side for all launches of a plan).
//
// The data layout is ns_phase_kernel's: s x s matrices as packed upper triangles of 256 x 256 blocks
// (SqPanel) with whole symmetric diagonal blocks. Of a diagonal block's four tiles the upper three
// are computed; the off-diagonal one is also stored transposed.
//
// Main loop: a ring of S stages of LDS (16 KB each, A and B by direct loads S - 1 K tiles ahead), one
// barrier per K tile of 32; the epilogue's tile (and the C term, loaded before the first K tile) has
// 32 KB of its own. Two kernels: 4 waves of 64 x 64 and S = 3, 80 KB, two blocks to a CU, each filling
// the other's waits, for launches of more than 256 tiles; 8 waves of 64 x 32 and S = 8, 160 KB, for
// launches that give a CU at most one block anyway, where two waves to a SIMD hide each other's LDS reads
// (a 1024 x 2048 matrix's products: 21.5 us with 4 waves and 64 KB in flight, 17.5 with 4 waves and 112 KB,
// 16 with 8 waves; a 257 x 257 matrix's, two thirds of it launch latency: 8.4, 9.2 and 8).
#pragma once
#include "ns_kernels.hip"

namespace thorn {

template <int STAGES, int WAVES>
struct T128 {
    static constexpr int BM = 128, BK = 32, S = STAGES;
    static constexpr int NW = WAVES, NT = 64 * WAVES;
    static constexpr int WN = NW / 2, NB = 4 / WN;           // waves across, 32-column blocks of each
    static constexpr int N = 2 * NB;                         // blocks of a wave
    static constexpr int OP_BYTES = BM * BK * 2;             // one operand's stage
    static constexpr int STAGE_BYTES = 2 * OP_BYTES;
    static constexpr int LOADS = 2 * OP_BYTES / 1024 / NW;   // direct loads per wave and K tile
    static constexpr int TILE = BM * BM * 2;                 // the epilogue's tile, before the stages
    static constexpr int SMEM = TILE + S * STAGE_BYTES;
    static_assert(LOADS * NW == 16 && SMEM <= 160 * 1024 && (S - 2) * LOADS < 63, "LDS, vmcnt");
    // this wave's rows and columns of the tile
    __device__ static __forceinline__ int a0(int wave) { return wave / WN * 64; }
    __device__ static __forceinline__ int b0(int wave) { return wave % WN * (32 * NB); }
};
constexpr int kT128 = 128;
typedef T128<3, 4> T128Two;   // two blocks to a CU
typedef T128<8, 8> T128One;   // one

// Byte offset of (row r, column c) of the epilogue's tile: 256-byte rows, 16-byte chunk k of row r
// at position k ^ (r & 15).
__device__ __forceinline__ int t128_off(int r, int c) {
    return r * 256 + ((((c >> 3) ^ (r & 15)) << 4) | ((c & 7) << 1));
}

// The C term's tile into the epilogue's: 32 pieces of 1 KB (four rows), 32 / NW a wave.
template <class T>
__device__ __forceinline__ void t128_load_c(const TileC& c, int m0, int n0, uint32_t lds0, int wave, int lane) {
    const u32x4 rsrc = sgpr_rsrc(c.ptr, c.ptr ? static_cast<uint32_t>(int64_t(c.rows) * c.ld * 2) : 0u);
    const uint32_t step = static_cast<uint32_t>(32 * c.ld);   // bytes of 16 rows, which share the swizzle
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 128 / T::NW * wave + 4 * j + (lane >> 4);
        const int col = n0 + 8 * ((lane & 15) ^ (row & 15));
        const uint32_t o = col < c.ld ? static_cast<uint32_t>((int64_t(m0 + row) * c.ld + col) * 2) : kOutOfRange;
#pragma unroll
        for (int h = 0; h < 8 / T::NW; ++h)
            asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(o + h * step), "s"(rsrc),
                         "{m0}"(lds0 + (32 / T::NW * wave + 4 * h + j) * 1024)
                         : "memory");
    }
}

// The operands' loaders.
template <class T>
struct Loads128 {
    typedef OperandDma<kT128, T::NW> Dma;
    Dma a, b;

    // Direct loads of K tile t (tiles in order; past the end zeros) into the stage at LDS address `at`
    // (this wave's share).
    template <bool AK, bool BK>
    __device__ __forceinline__ void issue(int t, uint32_t at) {
        if (a.switches(t) || b.switches(t)) {
            asm volatile("");
            a.begin_tile(t);
            b.begin_tile(t);
        }
        if constexpr (!AK || !BK) {
            if (t % 8 == 0 && t > 0) {
                asm volatile("");
                if (!AK && t < a.k0) a.next_panel();
                if (!BK && t < b.k0) b.next_panel();
            }
        }
#pragma unroll
        for (int q = 0; q < Dma::PER_WAVE; ++q) a.issue(q, at + q * 1024);
#pragma unroll
        for (int q = 0; q < Dma::PER_WAVE; ++q) b.issue(q, at + T::OP_BYTES + q * 1024);
    }
};

// K tiles [lo, hi) in one pair of layouts; acc[NB x + y]: the wave's 32 x 32 block (x, y), transposed
// as in mfma_phase. at: the stage of tile lo (bytes). `on`: the wave has blocks to compute.
template <class T, bool AK, bool BK>
__device__ __forceinline__ void t128_segment(int lo, int hi, bool on, const char* stages, int& at, int a0, int b0,
                                             Loads128<T>& ld, uint32_t m0w, floatx16 (&acc)[T::N]) {
    const int lane = threadIdx.x & 63;
    constexpr int LAST = (T::S - 1) * T::STAGE_BYTES;
    for (int kt = lo; kt < hi; ++kt) {
        // this wave's loads of tile kt have landed (those of the S - 2 tiles after it may be in flight);
        // after the barrier every wave's have, and all have read tile kt - 1, whose stage is refilled
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((T::S - 2) * T::LOADS) : "memory");
        ld.template issue<AK, BK>(kt + T::S - 1, m0w + (at == 0 ? LAST : at - T::STAGE_BYTES));
        const char* st = stages + at;
        at = at == LAST ? 0 : at + T::STAGE_BYTES;
        if (!on) continue;
        half8 a[2][2], b[2][T::NB];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int x = 0; x < 2; ++x) a[ks][x] = frag<128, AK>(st, a0 + 32 * x, ks, lane);
#pragma unroll
            for (int y = 0; y < T::NB; ++y) b[ks][y] = frag<128, BK>(st + T::OP_BYTES, b0 + 32 * y, ks, lane);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < T::NB; ++y) {
                    floatx16& d = acc[T::NB * x + y];
                    d = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[ks][y], a[ks][x], d, 0, 0, 0);
                }
    }
}

// acc = A B over KT K tiles for this wave's blocks of the tile at (m0, n0), C's tile loaded into the
// epilogue's. Layouts switch at a_k0 <= b_k0 as in gemm_tile. Ends with every load landed and a
// barrier.
template <class T>
__device__ __forceinline__ void t128_gemm(const Operand& A, const Operand& B, int m0, int n0, int KT, int a_k0,
                                          int b_k0, const TileC& ct, bool on, floatx16 (&acc)[T::N], char* smem) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int q = 0; q < T::N; ++q) acc[q] = floatx16{};
    Loads128<T> ld;
    ld.a.init(A, m0, wave, lane, a_k0, KT);
    ld.b.init(B, n0, wave, lane, b_k0, KT);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(smem));
    const uint32_t m0w = lds0 + T::TILE + wave * Loads128<T>::Dma::PER_WAVE * 1024;
    t128_load_c<T>(ct, m0 - ct.r0, n0 - ct.c0, lds0, wave, lane);
#pragma unroll
    for (int t = 0; t < T::S - 1; ++t) ld.template issue<true, true>(t, m0w + t * T::STAGE_BYTES);   // (no panel begins here)
    const int a0 = T::a0(wave), b0 = T::b0(wave);
    const int k1 = a_k0 < KT ? a_k0 : KT;
    const int k2 = b_k0 < k1 ? k1 : (b_k0 < KT ? b_k0 : KT);
    int at = 0;
    const char* const stages = smem + T::TILE;
    t128_segment<T, false, false>(0, k1, on, stages, at, a0, b0, ld, m0w, acc);
    t128_segment<T, true, false>(k1, k2, on, stages, at, a0, b0, ld, m0w, acc);
    t128_segment<T, true, true>(k2, KT, on, stages, at, a0, b0, ld, m0w, acc);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Stages val(r, c, a), the final f16 values of row r, columns c .. c + 3, from their accumulators (see
// stage_f16). On a diagonal tile only the blocks on and above the diagonal are staged, with their
// transposes below it, so the staged tile is exactly symmetric.
template <class T, class Val>
__device__ __forceinline__ void t128_stage(floatx16 (&acc)[T::N], char* smem, bool diag, bool on, Val val) {
    if (!on) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int a0 = T::a0(wave), b0 = T::b0(wave);
    const int lr = lane & 31, lc = 4 * (lane >> 5);
    static_for<0, T::N>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int rb = a0 + 32 * (q / T::NB), cb = b0 + 32 * (q % T::NB);
        if (diag && cb < rb) return;
        const int r = rb + lr;
        half4 h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = cb + lc + 8 * e;
            h[e] = val(r, c, floatx4{acc[q][4 * e], acc[q][4 * e + 1], acc[q][4 * e + 2], acc[q][4 * e + 3]});
            opaque(h[e]);   // one rounding for both copies, as in stage_f16
            *reinterpret_cast<half4*>(smem + t128_off(r, c)) = h[e];
        }
        if (!diag) return;
        // a block on the diagonal is whole before the transposes of its upper elements replace the
        // lower ones (a wave's LDS writes complete in order)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = cb + lc + 8 * e + i;
                if (c > r) *reinterpret_cast<_Float16*>(smem + t128_off(c, r)) = h[e][i];
            }
    });
}

// fn(it, r, c8, h) over this thread's row chunks: staged row r = NT / 16 it + tid / 16, columns c8 ..
// c8 + 7, c8 = 8 (tid % 16).
template <class T, class Fn>
__device__ __forceinline__ void t128_rows(const char* smem, Fn fn) {
    const int tr = threadIdx.x >> 4, c8 = 8 * (threadIdx.x & 15);
#pragma unroll
    for (int it = 0; it < 2048 / T::NT; ++it) {
        const int r = T::NT / 16 * it + tr;
        fn(it, r, c8, *reinterpret_cast<const half8v*>(smem + t128_off(r, c8)));
    }
}

// The staged tile to rows [0, rows) at o.ptr (rows below the matrix's end), columns n0 - c0 ...
template <class T>
__device__ __forceinline__ void t128_store(const char* smem, _Float16* out, int64_t ld, int rows, int n0) {
    const int nr = rows < kT128 ? rows : kT128;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(out, 0, static_cast<int>(nr * ld * 2), 0x00020000);
    const int tr = threadIdx.x >> 4, c8 = 8 * (threadIdx.x & 15);
    const uint32_t base = n0 + c8 < ld ? static_cast<uint32_t>((tr * ld + n0 + c8) * 2) : kOutOfRange;
    const uint32_t step = static_cast<uint32_t>(T::NT / 8 * ld);
    t128_rows<T>(smem, [&](int it, int, int, const half8v& h) { buf_store8<2>(rs, base + it * step, h); });
}

// The staged tile's transpose to out (row stride ld), whose rows are the tile's columns (`rows` of them
// valid) and whose columns c0 .. c0 + 127 are its rows (see sym_put_mirror for the lanes).
template <class T>
__device__ __forceinline__ void t128_store_mirror(const char* smem, _Float16* out, int64_t ld, int rows, int c0) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int grp = lane >> 4, j = lane & 15;
    const uint32_t lds0 = lds_address(smem);
#pragma unroll
    for (int it = 0; it < 32 / T::NW; ++it) {
        const int cb = 16 * (8 / T::NW * wave + (it >> 2)), r0 = 32 * (it & 3) + 8 * grp;
        const int col = cb + 4 * (j & 3);
        const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(lds0 + t128_off(r0 + (j >> 2), col)));
        const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(lds0 + t128_off(r0 + 4 + (j >> 2), col)));
        const half4 l4 = __builtin_bit_cast(half4, lo), h4 = __builtin_bit_cast(half4, hi);
        const half8v h{l4[0], l4[1], l4[2], l4[3], h4[0], h4[1], h4[2], h4[3]};
        if (cb + j < rows) stg_nt<half8v>(out + int64_t(cb + j) * ld + c0 + r0, h);
    }
}

// The tile (m0, n0) of a packed s x s result (m0 <= n0): into its panel, and transposed where it is
// the upper one of a diagonal block's two off-diagonal tiles.
template <class T>
__device__ __forceinline__ void t128_store_packed(const char* smem, _Float16* base, const OrthoMat& M, int m0, int n0) {
    const int b = m0 / 256, in = m0 % 256;
    const SqPanel p = sq_panel(M.s, M.lds, b);
    t128_store<T>(smem, base + p.off + in * p.ld, p.ld, p.rows - in, n0 - 256 * b);
    if (n0 / 256 == b && n0 != m0)
        t128_store_mirror<T>(smem, base + p.off + 128 * p.ld, p.ld, p.rows - 128, 0);
}

// Epilogue of a symmetric tile: out = f16(alpha acc + beta C) (see sym_store).
template <class T>
__device__ __forceinline__ void t128_sym(const OrthoMat& M, const NsOp& op, floatx16 (&acc)[T::N], bool on, int m0, int n0,
                                         char* smem) {
    const bool diag = m0 == n0;
    float alpha = op.alpha;
    if (op.kind == kOpGram) {
        const float osc = op.first ? M.scal[kScalX0Scale] : 1.f;
        alpha = osc * osc;
    }
    _Float16* const out = op.kind == kOpGram ? M.gram : sym_buf(M, op.osel);
    if (op.kind == kOpSym && op.csel >= 0) {
        const float beta = op.beta;
        t128_stage<T>(acc, smem, diag, on, [&](int r, int c, const floatx4& a) {
            const half4 cv = *reinterpret_cast<const half4*>(smem + t128_off(r, c));
            half4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                h[e] = static_cast<_Float16>(fmaf(beta, static_cast<float>(cv[e]), alpha * a[e]));
            return h;
        });
    } else {
        t128_stage<T>(acc, smem, diag, on, [&](int, int, const floatx4& a) {
            return half4{(_Float16)(alpha * a[0]), (_Float16)(alpha * a[1]), (_Float16)(alpha * a[2]),
                         (_Float16)(alpha * a[3])};
        });
    }
    lds_barrier();
    t128_store_packed<T>(smem, out, M, m0, n0);
    if (op.kind == kOpSym && op.osel2 >= 0) {   // Q = Z + a I
        if (diag) {
            lds_barrier();
            const int r = threadIdx.x;
            if (r < kT128) {
                _Float16& z = *reinterpret_cast<_Float16*>(smem + t128_off(r, r));
                z = m0 + r < M.s ? static_cast<_Float16>(static_cast<float>(z) + op.dual_add) : z;
            }
            lds_barrier();
        }
        t128_store_packed<T>(smem, sym_buf(M, op.osel2), M, m0, n0);
    }
}

// Epilogue of an update tile (see update_finish): the next iterate, u' and its row sums, or p.
// tj: the tile's column, rows of rowsqpart. (No sums of p^2: plans with decouple_md keep 256 x 256 tiles.)
template <class T>
__device__ __forceinline__ void t128_update(const OrthoMat& M, const NsOp& op, floatx16 (&acc)[T::N], int m0, int n0,
                                            int tj, char* smem) {
    const int rows = M.rows, cols = M.cols, ldx = M.ldx, flags = M.flags;
    const float osc = op.first ? M.scal[kScalX0Scale] : 1.f;
    _Float16* const xout = op.xsel == kXA ? M.xb : M.xa;
    const bool direct = op.final_iter && !(flags & kFlagPNN);
    const bool vec = flags & kFlagVec4, bf = flags & kFlagBf16;
    const int tr = threadIdx.x >> 4, c8 = 8 * (threadIdx.x & 15);
    const bool apply_full = direct && vec && !bf && m0 + kT128 <= rows && n0 + kT128 <= cols;
    float* const p = M.p;
    // a whole tile's p is requested before the staging
    constexpr int ITERS = 2048 / T::NT;
    float4 pv[ITERS][2];
    if (apply_full) {
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const float* pp = p + int64_t(m0 + T::NT / 16 * it + tr) * cols + n0 + c8;
            pv[it][0] = ldg<float4>(pp);
            pv[it][1] = ldg<float4>(pp + 4);
        }
    }
    if (op.csel >= 0) {
        const float bx = op.beta * osc;
        t128_stage<T>(acc, smem, false, true, [&](int r, int c, const floatx4& a) {
            const half4 xv = *reinterpret_cast<const half4*>(smem + t128_off(r, c));
            half4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(fmaf(bx, static_cast<float>(xv[e]), osc * a[e]));
            return h;
        });
    } else {
        t128_stage<T>(acc, smem, false, true, [&](int, int, const floatx4& a) {
            return half4{(_Float16)(a[0] * osc), (_Float16)(a[1] * osc), (_Float16)(a[2] * osc), (_Float16)(a[3] * osc)};
        });
    }
    lds_barrier();
    if (!direct) t128_store<T>(smem, xout + int64_t(m0) * ldx, ldx, rows - m0, n0);
    if (!op.final_iter) return;
    if (!direct) {   // row sums of u'^2: 16 consecutive lanes hold a row
        float* const rowsq = M.rowsqpart + int64_t(tj) * rows;
        t128_rows<T>(smem, [&](int, int r, int, const half8v& h) {
            float t = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = static_cast<float>(h[e]);
                t += f * f;
            }
            t = m0 + r < rows && n0 + c8 < ldx ? t : 0.f;
            t += dpp_mov<0xB1>(t);
            t += dpp_mov<0x4E>(t);
            t += dpp_mov<0x141>(t);
            t += dpp_mov<0x140>(t);
            if (c8 == 0 && m0 + r < rows) stg<float>(rowsq + m0 + r, t);
        });
        return;
    }
    const bool apply = (flags & kFlagApply) != 0;
    const float eta = (flags & kFlagMagma) ? M.eta * ldg<float>(M.magma_s) : M.eta, wd = M.wd;
    auto step1 = [&](float x, float u) {
        const float q = cautious_step(x, u, eta, wd);
        return apply ? q : x;
    };
    auto step8 = [&](float (&v)[8], const half8v& h) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = step1(v[e], static_cast<float>(h[e]));
    };
    if (apply_full) {
        t128_rows<T>(smem, [&](int it, int r, int, const half8v& h) {
            float v[8] = {pv[it][0].x, pv[it][0].y, pv[it][0].z, pv[it][0].w,
                          pv[it][1].x, pv[it][1].y, pv[it][1].z, pv[it][1].w};
            step8(v, h);
            float* pp = p + int64_t(m0 + r) * cols + n0 + c8;
            stg<float4>(pp, make_float4(v[0], v[1], v[2], v[3]));
            stg<float4>(pp + 4, make_float4(v[4], v[5], v[6], v[7]));
        });
    } else {
        auto rows_of = [&](auto fn) { t128_rows<T>(smem, [&](int, int r, int c, const half8v& h) { fn(r, c, h); }); };
        auto at = [&](int r, int c) { return reinterpret_cast<const _Float16*>(smem + t128_off(r, c)); };
        if (bf) update_edge<true, kT128>(rows_of, at, p, m0, n0, rows, cols, vec, apply, step1, step8);
        else update_edge<false, kT128>(rows_of, at, p, m0, n0, rows, cols, vec, apply, step1, step8);
    }
}

// ns_phase_kernel's operations on 128 x 128 tiles: tile number `local` of a symmetric result counts
// its upper-triangle tiles row by row, of an update column by column.
template <class T>
__global__ __launch_bounds__(T::NT, 2) void ns_phase128_kernel(const OrthoMat* __restrict__ mats, TaskList t0,
                                                                   NsOp op0, TaskList t1, NsOp op1, int t1_first) {
    __shared__ __attribute__((aligned(1024))) char smem[T::SMEM];
    int b;
    const bool later = t1_first ? xcd_split(blockIdx.x, t1.total, t0.total, b)
                                : xcd_split(blockIdx.x, t0.total, t1.total, b);
    const bool second = t1_first ? !later : later;
    const TaskList& tl = second ? t1 : t0;
    const NsOp& op = second ? op1 : op0;
    if (op.kind == kOpNone) return;
    const int2 task = *reinterpret_cast<const int2*>(tl.map + 2 * b);
    const OrthoMat& M = mats[task.x];
    const int local = task.y;

    const int KTs = (M.s + T::BK - 1) / T::BK;
    int ti, tj, KT, a_k0, b_k0;
    Operand A, B;
    TileC ct{nullptr, 0, 0, 0, 0};
    if (op.kind == kOpUpdate) {
        const int tm = (M.rows + kT128 - 1) / kT128;
        ti = local % tm;
        tj = local / tm;
        const Operand X = iterate_operand(M, op.xsel), Q = square_operand(sym_buf(M, op.qsel), M);
        KT = KTs;
        A = M.tall ? X : Q;
        B = M.tall ? Q : X;
        a_k0 = M.tall ? 0 : ti / 2 * 8;
        b_k0 = M.tall ? tj / 2 * 8 : KT;
        if (op.csel >= 0) ct = TileC{X.ptr, M.ldx, M.rows, 0, 0};
    } else {
        tri_decode(local, (M.s + kT128 - 1) / kT128, ti, tj);
        if (op.kind == kOpGram) {
            A = B = iterate_operand(M, op.xsel);
            KT = (M.l + T::BK - 1) / T::BK;
            a_k0 = b_k0 = M.tall ? KT : 0;
        } else {
            A = square_operand(sym_buf(M, op.asel), M);
            B = square_operand(sym_buf(M, op.bsel), M);
            KT = KTs;
            a_k0 = ti / 2 * 8;
            b_k0 = tj / 2 * 8;
            if (op.csel >= 0) {
                const SqPanel p = sq_panel(M.s, M.lds, ti / 2);
                ct = TileC{sym_buf(M, op.csel) + p.off, p.ld, p.rows, ti / 2 * 256, ti / 2 * 256};
            }
        }
    }
    const int m0 = ti * kT128, n0 = tj * kT128;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const bool update = op.kind == kOpUpdate;
    // a diagonal tile's lower left is its mirror
    const bool on = update || ti != tj || T::a0(wave) < T::b0(wave) + 32 * T::NB;
    floatx16 acc[T::N];
    t128_gemm<T>(A, B, m0, n0, KT, a_k0, b_k0, ct, on, acc, smem);
    if (update) t128_update<T>(M, op, acc, m0, n0, tj, smem);
    else t128_sym<T>(M, op, acc, on, m0, n0, smem);
}

}  // namespace thorn

// Newton-Schulz for small matrices (short side s <= 256): one launch runs the whole schedule of
// every small matrix of a group (gfx950).
//
// The grouped 256 x 256-tile launches of ns_kernels.hip give a small matrix one tile per phase, so
// its 18 phases cost 18 launch latencies. Here each small matrix gets a cluster of 1024-thread
// workgroups (thin ones, s <= 128: as many as their columns need, below; above, enough for the s x s
// products in 64 x 64 super-tiles and the s x l updates in 128 x 128 ones to take one round each, at
// most 16), placed on one XCD
// (block map), that runs every operation of the schedule in turn, 32 x 32 output tiles
// dealt to its 16 * C waves, with a barrier between operations (SmallSync). The
// operands stay in the L2-resident workspace, each s x s result and each iterate also stored
// transposed, so that every MFMA fragment, of A or of B, is one 16-byte load of a K-contiguous row.
// Products are computed whole (no mirroring of a symmetric result), and every output is rounded to
// f16 once from f16(beta C + alpha A B), as the reference's eager baddbmm does (thorn.py:338-343),
// so on small matrices the iteration tracks the reference's f16 trajectory closely.
//
// Workspace of a small matrix (all f16, padded to multiples of 32 with zeros that stay zero):
//   xw[2], xwt[2]: the iterate in the wide orientation (s_p x l_p) and transposed (l_p x s_p),
//     two slots; the iterate of a tall parameter is the transpose of its rows (thorn.py:629-630);
//   sq[4], sqt[4]: R, Z, QA, QB (s_p x s_p) and their transposes.
// The first iterate is written into xw[0] and xwt[0] by ortho_cast_kernel;
// u' goes to xa in the parameter's orientation, with the per-row partial sums of u'^2 that the
// per-row normalization needs.
//
// A plan whose matrices all take this path (none with decouple_md, Magma or an Adam step, every
// one applied this step) runs its whole step as ns_small_kernel<true>: each cluster also does, for
// its own matrix, the work of ortho_pre_kernel (momentum, tile partials of ||u||^2),
// ortho_norm_kernel (the norm) and ortho_cast_kernel (the first iterate) before the schedule, and
// of ortho_rowstats_kernel and ortho_pnn_apply_kernel (the update of p) after it: one launch in
// place of six, two more cluster barriers. The elementwise parts keep those kernels' tiles
// (TileMap), thread layouts and summation orders (each 256-thread quarter of a workgroup takes one
// tile at a time; the norm, the row statistics and the apply are the same device functions), so
// every value is bit for bit the one the separate launches give.
#include "ns_kernels.hip"
#include "update_kernels.hip"

namespace thorn {

constexpr int kSmallMaxS = 256;        // short side of the matrices this path takes
constexpr int kSmallMaxOps = 64;       // operations per schedule
constexpr int kSmallThreads = 1024;    // 16 waves per workgroup
constexpr int kSmallWaves = kSmallThreads / 64;

struct SmallOp {
    int8_t kind;     // kOpGram, kOpSym, kOpUpdate
    int8_t a, b, c;  // sym: A, B, C buffers (c < 0: none); update: a = Q buffer, c >= 0: + beta X
    int8_t o, o2;    // sym: output buffer, dual output (Q = out + dual I) or -1
    int8_t xsel;     // gram, update: iterate slot read (the update writes the other one)
    int8_t fin;      // update: the last one (writes u')
    float alpha, beta, dual;
};

struct SmallSchedule {
    SmallOp op[2][kSmallMaxOps];   // [0] square matrices (plain quintic), [1] the others (Gram)
    int32_t n[2];
};

// Barrier of the C workgroups of one matrix, on one word of the workspace: the arrival count in
// bits 0-15 and the generation in bits 16-31. A member arrives by adding 1 and learns the
// generation from the value it gets back; the last one to arrive (count C - 1 before its add) adds
// 2^16 - C, which clears the count and advances the generation in one atomic, and the others poll
// the word until the generation moves. Agent-scope release on arrival and acquire on departure.
// The wait is bounded: a cluster whose members are not all resident cannot hang the GPU; after
// `spin` polls (each a 64-cycle sleep) it sets *err and goes on. Should a member that gave up
// waiting arrive at the next barrier first, its arrival stays in the count (the last arrival
// subtracts C, it does not store 0), so every launch, whose members each arrive once at every
// barrier, leaves the count at 0.
__device__ __forceinline__ bool cluster_last(unsigned old, int C) { return (old & 0xFFFFu) == unsigned(C - 1); }
__device__ __forceinline__ void cluster_poll(unsigned* w, unsigned old, int* err, int spin) {
    int it = 0;
    while ((__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 16) == (old >> 16)) {
        if (it++ >= spin) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

__device__ __forceinline__ void cluster_barrier(int* bar, int C, int* err, int spin) {
    __syncthreads();
    if (C > 1 && threadIdx.x == 0) {
        unsigned* w = reinterpret_cast<unsigned*>(bar);
        const unsigned old = __hip_atomic_fetch_add(w, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (cluster_last(old, C)) {
            __hip_atomic_fetch_add(w, (1u << 16) - unsigned(C), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            cluster_poll(w, old, err, spin);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
    }
    __syncthreads();
}

// The same barrier for a cluster whose workgroups all run on one XCD, so that they share its L2,
// which is then the point where their stores meet: each wave's stores are complete in the L2
// before the arrival (vmcnt(0)), and after the departure the caches between the CU and the L2
// are invalidated together with the L2's clean lines (buffer_inv sc1), so the loads that follow
// read what the other members stored. The L2 is not written back (buffer_wbl2 sc1), as the
// agent-scope barrier does it for other XCDs. (Invalidating the CU's L1 alone, buffer_inv sc0, as
// LLVM's gfx942 model does for a workgroup split over CUs, left stale operands in one sequence
// whose members shared the XCD but not a shader engine.) The word is accessed exactly as there
// (the same atomics and polling loads).
__device__ __forceinline__ void cluster_barrier_xcd(int* bar, int C, int* err, int spin) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (C > 1 && threadIdx.x == 0) {
        unsigned* w = reinterpret_cast<unsigned*>(bar);
        const unsigned old = __hip_atomic_fetch_add(w, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (cluster_last(old, C))
            __hip_atomic_fetch_add(w, (1u << 16) - unsigned(C), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
            cluster_poll(w, old, err, spin);
        asm volatile("buffer_inv sc1\n\ts_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
}

// The XCD (XCC) this workgroup runs on.
__device__ __forceinline__ int xcc_id() {
    unsigned x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
    return static_cast<int>(x & 0xF);
}

// A cluster's barriers. At the start each member stores its XCC id in the barrier's words; the
// first barrier is agent scope, after which each member reads all the ids, and when they are equal
// (the launch placed the cluster on one XCD: block b runs on XCD b mod 8 up to a fixed offset, and
// the block map gives a cluster's members one residue) every later barrier is the XCD-local one.
// The placement is a dispatch order, not a guarantee, so the ids decide: with members on two XCDs
// every barrier stays agent scope. (The ids ride on the first barrier the kernel needs anyway; a
// barrier of their own at the start cost one more agent-scope round.)
struct SmallSync {
    int* bar;   // the barrier word, an unused word, then one XCC id per member
    int* err;
    int C, spin;
    bool local, ids;   // ids: the XCC ids are read after the next (agent-scope) barrier
    // xcd: XCD-local barriers allowed (thorn_ortho_set_small_xcd_barriers; with 0 every barrier is
    // agent scope)
    __device__ __forceinline__ SmallSync(int* bar_, int member, int C_, int* err_, int spin_, bool xcd)
        : bar(bar_), err(err_), C(C_), spin(spin_), local(false), ids(C_ > 1 && xcd) {
        if (ids && threadIdx.x == 0) bar[2 + member] = xcc_id();
    }
    __device__ __forceinline__ void wait() {
        if (local) {
            cluster_barrier_xcd(bar, C, err, spin);
            return;
        }
        cluster_barrier(bar, C, err, spin);
        if (ids) {
            bool same = true;
            for (int i = 1; i < C; ++i) same = same && bar[2 + i] == bar[2];
            local = __builtin_amdgcn_readfirstlane(same ? 1 : 0) != 0;
            ids = false;
        }
    }
};
constexpr int kSmallBarWords = 2 + 16;   // the largest cluster has 16 members

// Operand panels in LDS: a super-tile of up to 128 x 128 outputs (up to 16 tiles of 32 x 32, one
// per wave) is computed from K chunks of 32: rows [M0, M0+SM) of A and [N0, N0+SN) of BT, 64
// bytes each, in the K-major stage layout of the large-matrix GEMM (chunk c of row r at
// r * 64 + (c ^ ((r >> 2) & 3)) * 16: 16 lanes reading rows r..r+15 at one chunk cover all banks).
// A ring of kSmallStages stages is filled by direct global-to-LDS loads, one 1 KB load per wave
// per chunk (its 64 lanes fill 64 consecutive 16-byte slots: lane slot s holds the chunk whose
// swizzled position is s), kSmallStages - 1 chunks ahead of the MFMAs. Two chunks in flight are
// as fast as three (5.4 against 5.5 us per 256 x 256 x 256 product), and seven are slower (6.7 us):
// the loop's time per chunk follows the LDS traffic of its 16 waves' fragment reads (64 KB per
// chunk for a 128 x 128 super-tile) more than the loads' latency. Between products the ring holds
// the waves' epilogue staging tiles (and, in the fused step, the first iterate's transposes).
constexpr int kSmallStages = 3;
constexpr int kSmallStageBytes = 2 * 128 * 64;   // A rows [0, 128), then BT rows [0, 128)

// This wave's direct loads except the newest n (0 <= n <= kSmallStages - 2, wave-uniform) are
// complete, then the block barrier.
__device__ __forceinline__ void wait_loads_barrier(int n) {
    switch (n) {
        case 0: asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); break;
        case 1: asm volatile("s_waitcnt vmcnt(1)\n\ts_barrier" ::: "memory"); break;
        case 2: asm volatile("s_waitcnt vmcnt(2)\n\ts_barrier" ::: "memory"); break;
        case 3: asm volatile("s_waitcnt vmcnt(3)\n\ts_barrier" ::: "memory"); break;
        case 4: asm volatile("s_waitcnt vmcnt(4)\n\ts_barrier" ::: "memory"); break;
        case 5: asm volatile("s_waitcnt vmcnt(5)\n\ts_barrier" ::: "memory"); break;
        default: asm volatile("s_waitcnt vmcnt(6)\n\ts_barrier" ::: "memory"); break;
    }
}
static_assert(kSmallStages - 2 <= 6, "wait_loads_barrier covers 0 .. kSmallStages - 2");

// The C term of a wave's tile in LDS (kCTileBytes per wave): its 32 rows of C^T (rows n0..,
// columns m0..m0+31), 64 bytes each, chunk c of row r at r * 64 + (c ^ ((r >> 2) & 3)) * 16,
// filled by two direct loads (the 64 lanes of each fill 64 consecutive 16-byte slots); `ok` false
// loads `zero` instead. Requested just before the product's first chunks (eight-byte loads of the
// C^T rows into registers, 32 rows per instruction, had taken ~0.7 us more than the chunk alone;
// these two cost the first chunk little, and issued after the chunks they were still in flight
// when a short K loop ended).
constexpr int kCTileBytes = 32 * 64;
__device__ __forceinline__ void small_issue_c(uint32_t lds, const _Float16* CT, int64_t ldc, int m0, int n0, bool ok,
                                              const void* zero, int lane) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int r = 16 * h + (lane >> 2), c = (lane & 3) ^ ((r >> 2) & 3);
        const void* p = ok ? static_cast<const void*>(CT + int64_t(n0 + r) * ldc + m0 + 8 * c) : zero;
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"((const THORN_GLOBAL void*)p),
                     "{m0}"(lds + h * 1024)
                     : "memory");
    }
}

// This lane's C values of its tile from the LDS copy, in the accumulator layout: cv[g][e] is
// C[m0 + 8g + 4(lane / 32) + e][n0 + lane % 32].
__device__ __forceinline__ void small_read_c(half4 (&cv)[4], const char* ctile, int lane) {
    const int j = lane & 31;
#pragma unroll
    for (int g = 0; g < 4; ++g)
        cv[g] = *reinterpret_cast<const half4*>(ctile + j * 64 + ((g ^ ((j >> 2) & 3)) << 4) + 8 * (lane >> 5));
}

// acc (this wave's tile of the super-tile, if it has one) = A[M0.., 0:K] * B[0:K, N0..] with A
// row-major (lda) and B given by its transpose BT row-major (ldb), K a multiple of 32, every
// operand row inside the padded buffers (rows past sm / sn read `zero`). With CT, the wave's C
// tile (CT at m0, n0) is also loaded into `ctile` (small_issue_c). The whole workgroup calls it
// (barriers inside; the first one orders it after every wave's use of the staging tiles in the
// ring); on return every load has landed and the stages are free.
__device__ __forceinline__ floatx16 small_block(char* stages, const void* zero, const _Float16* A, int64_t lda,
                                                const _Float16* BT, int64_t ldb, int M0, int N0, int sm, int sn,
                                                int K, int wave, int lane, bool has_tile, int ti, int tj,
                                                uint32_t ctile, const _Float16* CT, int64_t ldc, int m0, int n0,
                                                unsigned tslot = 0, int q = 0) {
    floatx16 acc = {};
    const int nk = K / 32;
    const int slot = wave * 64 + lane, part = slot >> 9, r = (slot >> 2) & 127;
    const int c = (slot & 3) ^ ((r >> 2) & 3);
    const bool ok = part == 0 ? r < sm : r < sn;
    // a wave whose 16 rows all lie past sm / sn (an edge super-tile) loads nothing: its waits then
    // pass at once
    const bool loads = 16 * (wave & 7) < (part == 0 ? sm : sn);
    const char* src = reinterpret_cast<const char*>(part == 0 ? A + int64_t(M0 + r) * lda : BT + int64_t(N0 + r) * ldb) +
                      16 * c;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(stages)) + wave * 1024;
    auto issue = [&](int t) {
        if (!loads) return;
        const void* p = ok ? static_cast<const void*>(src + int64_t(t) * 64) : zero;
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"((const THORN_GLOBAL void*)p),
                     "{m0}"(lds0 + (t % kSmallStages) * kSmallStageBytes)
                     : "memory");
    };
    __syncthreads();
    // the C loads first: they return before chunk 0 (loads return in order), so no wait covers
    // them alone
    if (CT) small_issue_c(ctile, CT, ldc, m0, n0, has_tile, zero, lane);
    const int pre = nk < kSmallStages - 1 ? nk : kSmallStages - 1;
    for (int t = 0; t < pre; ++t) issue(t);
    for (int kc = 0; kc < nk; ++kc) {
        // this wave's loads of chunk kc have landed (the ones issued after it may still be in
        // flight); after the barrier every wave's have, and nobody reads stage (kc - 1) % S any
        // more, which then receives chunk kc + S - 1
        const int ahead = nk - 1 - kc < kSmallStages - 2 ? nk - 1 - kc : kSmallStages - 2;
        wait_loads_barrier(ahead);
        if (kc == 0) ts_op(tslot, q, 3);
        if (kc + kSmallStages - 1 < nk) issue(kc + kSmallStages - 1);
        if (has_tile) {
            const char* st = stages + (kc % kSmallStages) * kSmallStageBytes;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const half8 a = frag<128, true>(st, 32 * ti, ks, lane);
                const half8 b = frag<128, true>(st + kSmallStageBytes / 2, 32 * tj, ks, lane);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0);
            }
        }
    }
    ts_op(tslot, q, 4);
    __syncthreads();   // every wave is done with the stages (the last wait was vmcnt(0): the C loads too)
    return acc;
}

// The wave's 32 x 32 f16 staging tile: row-major, rows of 34 halves.
constexpr int kStageLd = 34;

// Lanes of one wave hand values to each other through the staging tile: every LDS access before
// this point is complete, and (a compiler memory barrier) none is moved across it or served from
// a value loaded before it. Without it the compiler may reuse a value it already loaded, since a
// write by another lane is not visible to a single thread's program order.
__device__ __forceinline__ void wave_lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Stages f16(alpha * acc + beta * C) of tile (m0, n0), C from small_read_c (HAS_C).
template <bool HAS_C>
__device__ __forceinline__ void small_stage(const floatx16& acc, _Float16* stage, float alpha, float beta,
                                            const half4 (&cv)[4], int lane) {
    const int j = lane & 31;
    wave_lds_sync();   // the previous tile's reads of the staging are done
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int i0 = 8 * g + 4 * (lane >> 5);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float t = alpha * acc[4 * g + e];
            if (HAS_C) t += beta * static_cast<float>(cv[g][e]);
            stage[(i0 + e) * kStageLd + j] = static_cast<_Float16>(t);
        }
    }
    wave_lds_sync();   // the whole tile is staged before any lane reads it
}

// Stores the staged tile to out (row-major, ld) at (m0, n0) and its transpose to outT (ldt) at
// (n0, m0): 16-byte chunks, 2 + 2 per lane. Tiles lie inside the padded buffers.
__device__ __forceinline__ void small_store(const _Float16* stage, _Float16* out, int64_t ld, _Float16* outT,
                                            int64_t ldt, int m0, int n0, int lane) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int ch = lane + 64 * q, r = ch >> 2, c8 = (ch & 3) * 8;
        half8 h, t;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            h[e] = stage[r * kStageLd + c8 + e];
            t[e] = stage[(c8 + e) * kStageLd + r];
        }
        stg<half8>(out + int64_t(m0 + r) * ld + n0 + c8, h);
        stg<half8>(outT + int64_t(n0 + r) * ldt + m0 + c8, t);
    }
}

// u' (f16) in the parameter's orientation into xa, from the staged tile (m0, n0) of the wide
// iterate (s_p x l_p); per-row partial sums of u'^2 into rowsqpart[tile column][row] for
// per-row-normalized matrices. Element (i, j) of the wide iterate is parameter element (i, j)
// (wide or square) or (j, i) (tall).
__device__ __forceinline__ void small_store_final(const _Float16* stage, const OrthoMat& M, int m0, int n0, int lane) {
    const bool tall = M.tall;
    const int prow0 = tall ? n0 : m0, pcol0 = tall ? m0 : n0;   // the tile in the parameter's orientation
    auto at = [&](int pr, int pc) { return tall ? stage[pc * kStageLd + pr] : stage[pr * kStageLd + pc]; };
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int ch = lane + 64 * q, r = ch >> 2, c8 = (ch & 3) * 8;
        if (prow0 + r < M.rows && pcol0 + c8 < M.ldx) {
            half8 h;
#pragma unroll
            for (int e = 0; e < 8; ++e) h[e] = at(r, c8 + e);
            stg<half8>(M.xa + int64_t(prow0 + r) * M.ldx + pcol0 + c8, h);
        }
    }
    if ((M.flags & kFlagPNN) && lane < 32 && prow0 + lane < M.rows) {
        float t = 0.f;
        for (int c = 0; c < 32; ++c) {
            const float f = static_cast<float>(at(lane, c));
            t += f * f;
        }
        M.rowsqpart[int64_t(pcol0 >> 5) * M.rows + prow0 + lane] = t;
    }
}

// A member with at most kKeepRounds rounds of elementwise tiles keeps u in registers between the fused
// prologue's two passes, and requests p of that many rounds before the row scales are computed.
constexpr int kKeepRounds = 3;

// -------------------------------------------------------------------------------------------------
// Thin matrices: short side s <= 128. A workgroup's LDS holds R, Z and Q (s x s, row-major, 16 bytes of
// padding per row) and its columns of the iterate, so between the first iterate and u' nothing goes
// through memory but a cluster's Gram matrices: every member runs the whole chain of s x s products itself,
// the same one in each, and member i owns the 32-column blocks [nb0, nb1) of the iterate, whose update Q X
// needs no other member's columns. A Gram matrix's elements are one MFMA chain over K each, as in the
// schedule through the L2 (partial sums of the members' columns would give other last bits): the members of a
// cluster deal its 32 x 32 tiles among them (thin_gram). A cluster meets at its Gram matrices and at the end,
// not at each of the 18 operations. Bound by latency: a product
// of two s x s matrices takes 0.6 us (s <= 32) to 2 us (s = 128) against 7-8 with both operands and the result in
// the L2, a Gram matrix of 16 x 3072 6 us (192 dependent MFMAs of 64 cycles) against 30, its update 3.7 against 60
// (two of 16 waves, through both orientations in memory). Step of 3072 x 16 71 us against 554, of 128 x 384 84
// against 156; the launch over 224 adapters of rank 16 78 us against 580.
// -------------------------------------------------------------------------------------------------
constexpr int kThinMaxS = 128, kThinMaxCluster = 16;
constexpr int kThinLds = 159 * 1024;
__host__ __device__ constexpr int thin_square_bytes(int T) { return 32 * T * (64 * T + 16); }
// the squares, or the ring that a cluster's Gram matrices go through
__host__ __device__ constexpr int thin_base(int T) { return 3 * thin_square_bytes(T) > 16384 ? 3 * thin_square_bytes(T) : 16384; }
// columns of the iterate (a multiple of 32) that fit beside them: s rows, and one of zeros for the rows
// that pad s to 32 T
__host__ __device__ __forceinline__ int thin_columns(int s) {
    const int T = (s + 31) / 32, rows = s < 32 * T ? s + 1 : s;
    return ((kThinLds - thin_base(T)) / rows - 16) / 64 * 32;
}
// Members of a matrix's cluster: as many as its columns need, and at least one per kKeepRounds rounds of
// elementwise tiles; 0: more than a cluster has.
__host__ __device__ __forceinline__ int thin_cluster(int s, int l, int64_t tiles) {
    const int lp = (l + 31) / 32 * 32, cols = thin_columns(s);
    const int64_t by_cols = (lp + cols - 1) / cols, by_tiles = (tiles + 4 * kKeepRounds - 1) / (4 * kKeepRounds);
    if (by_cols > kThinMaxCluster) return 0;
    return static_cast<int>(by_tiles < by_cols ? by_cols : by_tiles < kThinMaxCluster ? by_tiles : kThinMaxCluster);
}
// A member's iterate columns in LDS: element (i, j), j from the member's first column, at `at(i) + 2 j`.
struct ThinX {
    int base, ldx, s, nb0, nb1;   // bytes; 32-column blocks
    __device__ __forceinline__ ThinX(const OrthoMat& M, const SmallView& V, int member, int C)
        : base(thin_base(V.sp / 32)), s(M.s) {
        const int nt = V.lp / 32, per = (nt + C - 1) / C;
        nb0 = min(nt, member * per);
        nb1 = min(nt, nb0 + per);
        ldx = 64 * per + 16;
    }
    __device__ __forceinline__ int at(int i) const { return base + min(i, s) * ldx; }   // row s: zeros
};

// Zeros in the row behind the matrix and in the columns that pad it, before the iterate is written.
__device__ __forceinline__ void thin_clear(const OrthoMat& M, const SmallView& V, const ThinX& X, char* lds) {
    const int cols = 32 * (X.nb1 - X.nb0), valid = max(0, min(cols, M.l - 32 * X.nb0));
    if (M.s < V.sp)
        for (int j = threadIdx.x; j < cols / 2; j += kSmallThreads)
            *reinterpret_cast<unsigned*>(lds + X.at(M.s) + 4 * j) = 0u;
    for (int e = threadIdx.x; e < M.s * (cols - valid); e += kSmallThreads)
        *reinterpret_cast<_Float16*>(lds + X.at(e / (cols - valid)) + 2 * (valid + e % (cols - valid))) = _Float16(0.f);
}

// The member's columns of the first iterate from slot 0 of the workspace (after thin_clear, whose zeros
// it does not touch; a barrier before the iterate is read).
__device__ __forceinline__ void thin_load(const OrthoMat& M, const SmallView& V, const ThinX& X, char* lds) {
    const int per = 4 * (X.nb1 - X.nb0), total = M.s * per;   // 16-byte chunks
    constexpr int U = 4;
    for (int k0 = threadIdx.x; k0 < total; k0 += U * kSmallThreads) {
        half8 x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * kSmallThreads, r = k / per, c = 32 * X.nb0 + 8 * (k - r * per);
            if (k < total) x[u] = ldg<half8>(V.xw(0) + int64_t(r) * V.lp + c);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * kSmallThreads, r = k / per, c = 8 * (k - r * per), left = M.l - 32 * X.nb0 - c;
            if (k >= total) continue;
            if (left >= 8) {
                *reinterpret_cast<half8*>(lds + X.at(r) + 2 * c) = x[u];
            } else {
                for (int e = 0; e < left; ++e) *reinterpret_cast<_Float16*>(lds + X.at(r) + 2 * (c + e)) = x[u][e];
            }
        }
    }
}

// MFMA fragments: rows whose row r starts at LDS byte row0 (its 8 halves of k16 step ks for this half of
// the wave), and columns t0.. of k rows by two transposing reads (the lane's k row and the fourth after it).
__device__ __forceinline__ half8 thin_row_frag(const char* lds, int row0, int ks, int lane) {
    return *reinterpret_cast<const half8*>(lds + row0 + 32 * ks + 16 * (lane >> 5));
}
__device__ __forceinline__ half8 thin_col_frag(uint32_t lds0, int row_lo, int row_hi, int t0, int lane) {
    const int c = 2 * (t0 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3));
    const half4 lo = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(lds0 + row_lo + c)));
    const half4 hi = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(lds0 + row_hi + c)));
    return half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// Four consecutive results alpha * acc + beta * c of a product, one rounding to f16 each.
template <bool HAS_C>
__device__ __forceinline__ half4 thin_round(const floatx16& acc, int g, float alpha, float beta, const half4& c) {
    half4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float t = alpha * acc[4 * g + e];
        if (HAS_C) t += beta * static_cast<float>(c[e]);
        h[e] = static_cast<_Float16>(t);
    }
    return h;
}

// R = X X^T of a cluster's iterate, from the workspace (slot 0) into the workspace's R: the 32 x 32 tiles on and
// above the diagonal dealt over the members, then over a member's waves, the panel rows that they need streamed
// by all waves through a ring of stages of 64 columns in the place of the squares (A and B are one panel), one
// barrier a stage, a stage's fragments read while the one before it is multiplied. Ends with this wave's stores
// issued. Bound by the chain of dependent MFMAs, 64 cycles each: 0.2 us a
// stage; the step of 108 x 3711 (15 members) 136 us, of 16 x 60000 464, against 893 and 3370 through the L2.
template <int T>
__device__ __forceinline__ void thin_gram(const OrthoMat& M, const SmallView& V, int member, int C, char* lds) {
    constexpr int SP = 32 * T, STAGE = 128 * SP, MAX = thin_base(T) / STAGE, S = MAX < 6 ? MAX : 6, TRI = T * (T + 1) / 2;
    static_assert(S >= 3 && 4 * T <= kSmallWaves && TRI <= kSmallWaves, "ring, loads, tiles");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    unsigned need = 0;   // 32-row blocks
    int ti = 0, tj = 0;
    bool has = false;
    for (int k = member, w = 0; k < TRI; k += C, ++w) {
        int i, j;
        tri_decode(k, T, i, j);
        need |= 1u << i | 1u << j;
        if (w == wave) has = true, ti = 32 * i, tj = 32 * j;
    }
    if (need == 0) return;
    // this wave's piece of a stage: 16 rows of one of its two chunks of 32 columns
    const int chunk = wave / (2 * T), r0 = 16 * (wave % (2 * T)), r = r0 + (lane >> 2);
    const bool loads = wave < 4 * T && (need >> (r0 / 32) & 1u);
    const char* const src = reinterpret_cast<const char*>(V.xw(0) + int64_t(r) * V.lp + 32 * chunk) +
                            16 * ((lane & 3) ^ ((r >> 2) & 3));
    const uint32_t to = __builtin_amdgcn_readfirstlane(lds_address(lds)) + chunk * (64 * SP) + 64 * r0;
    // Loads past the end read zeros, so that every stage has as many and the waits are constants.
    const void* const zero = M.zero;
    const int width = r < M.s ? V.lp - 32 * chunk : 0;   // (the rows that pad s: zeros)
    int col = 0;
    auto issue = [&](int at) {   // the next stage, into the place at byte `at`
        if (loads) {
            const void* p = col < width ? static_cast<const void*>(src + 2 * int64_t(col)) : zero;
            asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"((const THORN_GLOBAL void*)p), "{m0}"(to + at)
                         : "memory");
        }
        col += 64;
    };
    half8 a[2][4], b[2][4];
    auto fetch = [&](int s, int at) {   // this wave's fragments of the stage there
        if (!has) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[s][i] = frag<128, true>(lds + at + i / 2 * (64 * SP), ti, i % 2, lane);
            b[s][i] = frag<128, true>(lds + at + i / 2 * (64 * SP), tj, i % 2, lane);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    floatx16 acc = {};
    int at = 0;   // of the stage that is multiplied, then refilled
    auto step = [&](int s, int k0) {   // columns k0 .. k0 + 63
        // the next stage has landed, and every wave has this one in registers
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S - 2) : "memory");
        issue(at);
        at = at == (S - 1) * STAGE ? 0 : at + STAGE;
        fetch(s ^ 1, at);
        if (!has || k0 >= V.lp) return;
#pragma unroll
        for (int i = 0; i < 2; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[s][i], a[s][i], acc, 0, 0, 0);
        if (k0 + 32 >= V.lp) return;
#pragma unroll
        for (int i = 2; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[s][i], a[s][i], acc, 0, 0, 0);
    };
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the squares are free; counts start at 0
#pragma unroll
    for (int k = 0; k < S; ++k) issue(k * STAGE);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(S - 1) : "memory");
    fetch(0, 0);
    for (int k0 = 0; k0 < V.lp; k0 += 128) {
        step(0, k0);
        step(1, k0 + 64);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    if (!has) return;
    _Float16* const R = V.sq(kBufR);
    const int lr = lane & 31, lc = 4 * (lane >> 5);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const half4 h = thin_round<false>(acc, g, 1.f, 0.f, half4{});
        stg<half4>(R + (ti + lr) * SP + tj + 8 * g + lc, h);
        if (ti == tj) continue;   // (a diagonal tile is symmetric as computed)
#pragma unroll
        for (int e = 0; e < 4; ++e) stg<_Float16>(R + (tj + 8 * g + lc + e) * SP + ti + lr, h[e]);
    }
}

// Sum of the squares of 32 consecutive elements in order, as the schedule through the L2 adds them: lane l of the
// lower half of the wave holds elements 8 g + 0 .. 3 in h[g], lane l + 32 elements 8 g + 4 .. 7; both get it.
__device__ __forceinline__ float thin_sum_squares(const half4 (&h)[4]) {
    float t = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {   // (what the other half of the wave adds meanwhile is dropped)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float f = static_cast<float>(h[g][e]);
                t += f * f;
            }
            // low, high: the value of the wave's lower and upper half in both (the builtin's second result comes
            // back as its first with this compiler)
            float low = t, high = t;
            asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(low), "+v"(high));
            t = half == 0 ? low : high;
        }
    }
    return t;
}

// The schedule of one matrix with s_p = 32 T, its first iterate in LDS. Accumulators are transposed
// products (B^T A^T): lane l has row (l & 31) of a 32 x 32 tile, columns 8 g + 4 (l / 32) + 0..3 in
// registers 4 g + 0..3.
template <int T>
__device__ __forceinline__ void thin_schedule(const OrthoMat& M, const SmallView& V, const SmallOp* ops, int nops,
                                              int member, int C, char* lds, SmallSync& sync, unsigned tslot) {
    constexpr int SP = 32 * T, LDQ = 2 * SP + 16, SQ = thin_square_bytes(T), TILES = T * T;
    static_assert(TILES <= kSmallWaves, "a wave per tile");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds));
    const ThinX X(M, V, member, C);
    // this wave's tile of an s x s product
    const int ti = 32 * (wave % TILES / T), tj = 32 * (wave % T);
    const bool has = wave < TILES;
    // Where each of R, Z, QA, QB is (a byte each: an array indexed by the operation would go to memory).
    // A product replaces its C term in place (R Z is made from R, and the next R from R Z; Q from Q), but
    // Z has a place of its own, and a Q that starts anew another.
    unsigned places = 0x02020100u;
    auto at = [&](int buf) { return static_cast<int>(places >> (8 * buf) & 3u) * SQ; };
    auto move = [&](int buf, int place) { places = (places & ~(255u << (8 * buf))) | unsigned(place / SQ) << (8 * buf); };

    for (int q = 0; q < nops; ++q) {
        const SmallOp op = ops[q];
        // opaque per operation: the compiler otherwise keeps every operation's per-lane addresses in
        // registers over the whole schedule (150 spilled)
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, lr = lane & 31, lc = 4 * (lane >> 5);
        const int kr = 8 * (lane >> 5) + ((lane & 15) >> 2);   // k row of a transposing read
        ts_op(tslot, q, 0);
        if (op.kind == kOpGram) {
            move(kBufR, 0);
            if (C > 1) {
                if (q > 0) sync.wait();   // every member's columns of the iterate (the first one's are there)
                thin_gram<T>(M, V, member, C, lds);
                sync.wait();
                constexpr int PER = SP / 8;   // 16-byte chunks of a row
                for (int k = tid; k < SP * PER; k += kSmallThreads)
                    *reinterpret_cast<half8*>(lds + k / PER * LDQ + 16 * (k % PER)) = ldg<half8>(V.sq(kBufR) + 8 * k);
            } else if (has) {
                floatx16 acc = {};
                const int ra = X.at(ti + lr), rb = X.at(tj + lr), nks = 2 * (X.nb1 - X.nb0);
                // four steps of 16 columns are read while the four before them are multiplied
                half8 a[2][4], b[2][4];
                auto fetch = [&](int s, int k0) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int ks = min(k0 + i, nks - 1);
                        a[s][i] = thin_row_frag(lds, ra, ks, lane);
                        b[s][i] = thin_row_frag(lds, rb, ks, lane);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                auto multiply = [&](int s, int k0) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (k0 + i < nks) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[s][i], a[s][i], acc, 0, 0, 0);
                };
                fetch(0, 0);
                for (int k0 = 0; k0 < nks; k0 += 8) {
                    fetch(1, k0 + 4);
                    multiply(0, k0);
                    fetch(0, k0 + 8);
                    multiply(1, k0 + 4);
                }
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<half4*>(lds + (ti + lr) * LDQ + 2 * (tj + 8 * g + lc)) =
                        thin_round<false>(acc, g, 1.f, 0.f, half4{});
            }
            __syncthreads();
        } else if (op.kind == kOpSym) {   // out = alpha A B + beta C over the squares
            const int A = at(op.a), B = at(op.b), Cs = at(op.c);
            if (op.o != kBufZ) move(op.o, Cs);
            const int out = at(op.o), here = (ti + lr) * LDQ + 2 * (tj + lc);
            half4 h[4];
            if (has) {
                floatx16 acc = {};
#pragma unroll
                for (int ks = 0; ks < 2 * T; ++ks) {
                    const int k = B + (16 * ks + kr) * LDQ;
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(thin_col_frag(lds0, k, k + 4 * LDQ, tj, lane),
                                                                 thin_row_frag(lds, A + (ti + lr) * LDQ, ks, lane), acc, 0, 0, 0);
                }
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    h[g] = thin_round<true>(acc, g, op.alpha, op.beta, *reinterpret_cast<const half4*>(lds + Cs + here + 16 * g));
            }
            __syncthreads();   // every operand is read
            if (has) {
#pragma unroll
                for (int g = 0; g < 4; ++g) *reinterpret_cast<half4*>(lds + out + here + 16 * g) = h[g];
                if (op.o2 >= 0) {   // Q = out + dual I
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (ti + lr == tj + 8 * g + lc + e && ti + lr < M.s)
                                h[g][e] = static_cast<_Float16>(static_cast<float>(h[g][e]) + op.dual);
                        *reinterpret_cast<half4*>(lds + 2 * SQ + here + 16 * g) = h[g];
                    }
                }
            }
            if (op.o2 >= 0) move(op.o2, 2 * SQ);
            __syncthreads();
        } else {   // X' = Q X (+ beta X) on this member's columns, 32 of them per wave at a time, in place
            const int Q = at(op.a);
            for (int b = X.nb0 + wave; b < X.nb1; b += kSmallWaves) {
                const int j0 = 32 * (b - X.nb0), n0 = 32 * b;
                half8 x[2 * T];
#pragma unroll
                for (int ks = 0; ks < 2 * T; ++ks) x[ks] = thin_col_frag(lds0, X.at(16 * ks + kr), X.at(16 * ks + kr + 4), j0, lane);
                if (!op.fin || !M.tall) {
                    // rows of X' (a lane 4 consecutive columns): the next iterate, or u' of a wide parameter
#pragma unroll 1
                    for (int t = 0; t < T; ++t) {
                        const int row = 32 * t + lr;
                        floatx16 acc = {};
#pragma unroll
                        for (int ks = 0; ks < 2 * T; ++ks)
                            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[ks], thin_row_frag(lds, Q + row * LDQ, ks, lane), acc, 0, 0, 0);
                        half4 h[4];
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const int c = 8 * g + lc;
                            half4* const px = reinterpret_cast<half4*>(lds + X.at(row) + 2 * (j0 + c));
                            h[g] = op.c >= 0 ? thin_round<true>(acc, g, 1.f, op.beta, *px)
                                             : thin_round<false>(acc, g, 1.f, 0.f, half4{});
                            if (row >= M.s) continue;
                            if (op.fin) stg<half4>(M.xa + int64_t(row) * M.ldx + n0 + c, h[g]);
                            else *px = h[g];
                            // for the cluster's next Gram matrix (its last one's readers have met since)
                            if (!op.fin && C > 1) stg<half4>(V.xw(0) + int64_t(row) * V.lp + n0 + c, h[g]);
                        }
                        if (op.fin && (M.flags & kFlagPNN)) {
                            const float sq = thin_sum_squares(h);
                            if (lane < 32 && row < M.s) M.rowsqpart[int64_t(n0 >> 5) * M.rows + row] = sq;
                        }
                    }
                } else {
                    // u' of a tall parameter, whose rows are the iterate's columns: a lane has one of them,
                    // 4 consecutive elements
                    const int row = n0 + lr;
#pragma unroll 1
                    for (int t = 0; t < T; ++t) {
                        floatx16 acc = {};
#pragma unroll
                        for (int ks = 0; ks < 2 * T; ++ks)
                            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(thin_row_frag(lds, Q + (32 * t + lr) * LDQ, ks, lane), x[ks],
                                                                         acc, 0, 0, 0);
                        half4 h[4];
#pragma unroll
                        for (int g = 0; g < 4; ++g) {   // (a tall matrix is not square: no beta X)
                            h[g] = thin_round<false>(acc, g, 1.f, 0.f, half4{});
                            if (row < M.rows) stg<half4>(M.xa + int64_t(row) * M.ldx + 32 * t + 8 * g + lc, h[g]);
                        }
                        if (M.flags & kFlagPNN) {
                            const float sq = thin_sum_squares(h);
                            if (lane < 32 && row < M.rows) M.rowsqpart[int64_t(t) * M.rows + row] = sq;
                        }
                    }
                }
            }
            __syncthreads();
        }
        ts_op(tslot, q, 1);
        ts_op(tslot, q, 2);
    }
    sync.wait();   // every member's u' and row sums
}

// The fused step's prologue and epilogue: a workgroup's four 256-thread quarters take elementwise
// tiles 4 member + q, then 4 (member + C) + q, ... of the matrix.
constexpr int kQuarter = 256;
static_assert(kSmallThreads == 4 * kQuarter, "four quarters of a workgroup");

// First iterate of elementwise tile t by one quarter: the values of small_x0; the orientation in which
// the tile's columns are contiguous stored directly, the other through the quarter's LDS transpose `tt`
// (a row per column of the tile, holding its R = 4096 / 2^lw rows, R + 8 halves apart) as 16-byte chunks
// of 8 rows (rows past the matrix, inside the padded side, receive zeros). All quarters call it the same
// number of times (block barriers); `active`: t is a tile of the matrix.
constexpr int kX0Halves = 256 * 24;   // the largest transpose: 256 columns of 16 rows
static_assert(4 * kX0Halves * 2 <= kSmallStages * kSmallStageBytes, "four transposes in the ring");
// KEEP: u as momentum_tile gave it.
template <bool BF, bool KEEP>
__device__ __forceinline__ void small_x0_tile(const OrthoMat& M, const SmallView& V, int t, int t256, bool active,
                                              float denom, _Float16* tt, const float (&u)[16]) {
    const TileMap tm(M, t, t256);
    const int R = 4096 >> tm.lw, pitch = R + 8;   // the tile's rows
    _Float16* const direct = M.tall ? V.xwt(0) : V.xw(0);   // row r of the parameter, contiguous
    const int ldd = M.tall ? V.sp : V.lp;
    _Float16* const tpose = M.tall ? V.xw(0) : V.xwt(0);    // column c of the parameter, contiguous
    const int ldt = M.tall ? V.lp : V.sp;                   // (also the padded number of rows)
    if (active) {
        const float beta1 = M.beta1;
        const bool vec = KEEP && (M.flags & kFlagVec4);     // the elements that u belongs to
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int r = vec ? tm.vrow(k / 4) : tm.erow(k), c = vec ? tm.vcol() + k % 4 : tm.ecol(k);
            _Float16 x = _Float16(0.f);
            if (r < M.rows && c < M.cols) {
                x = (_Float16)((KEEP ? u[k] : u_of<BF>(M, r, c, beta1)) / denom);
                direct[int64_t(r) * ldd + c] = x;
            }
            tt[(c - tm.c0) * pitch + r - tm.row0] = x;
        }
    }
    lds_barrier();   // (not the stores)
    if (active) {
        const int per = R / 8;
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) {
            const int chunk = t256 + kQuarter * h2, cl = chunk / per, h = chunk % per;
            if (tm.c0 + cl < M.cols && tm.row0 + 8 * h < ldt)
                stg<half8>(tpose + int64_t(tm.c0 + cl) * ldt + tm.row0 + 8 * h,
                           *reinterpret_cast<const half8*>(tt + cl * pitch + 8 * h));
        }
    }
    lds_barrier();   // the transpose is read before the next round writes it
}

// Before the schedule: the momentum and the tile partials of ||u||^2 (momentum_tile, as
// ortho_pre_kernel makes them), a cluster barrier, the norm and, in member 0, the matrix's
// scalars, the first iterate f16(u / (||u|| + 1e-8)) and its padding, a cluster barrier.
// A thin matrix of one workgroup leaves its first iterate in LDS; returns whether it did.
template <bool BF, bool KEEP>
__device__ __forceinline__ bool small_fused_prologue_as(const OrthoMat& M, const SmallView& V, int member, int C,
                                                        float* red, char* stages, SmallSync& sync) {
    const int q = threadIdx.x / kQuarter, t256 = threadIdx.x % kQuarter;
    const int ntiles = M.mom_tiles_r * M.mom_tiles_c, per = 4 * C;
    float u[KEEP ? kKeepRounds : 1][16];
    float* const quads = reinterpret_cast<float*>(stages) + 64 * q;
    auto norm_round = [&](int t0, float (&ur)[16]) {
        const int t = t0 + 4 * member + q;
        // (barriers for LDS alone: the moments' stores drain behind them; 4 us a round when waited for)
        lds_barrier();   // the previous round's quads are read
        if (t < ntiles) momentum_tile<BF, !KEEP>(M, t, t256, false, ur, quads);
        lds_barrier();
        if (t < ntiles) tile_partials(M, t, t256, false, quads);
    };
    // (the same trip count in every quarter: barriers)
    if constexpr (KEEP) {
#pragma unroll
        for (int r = 0; r < kKeepRounds; ++r)
            if (r * per < ntiles) norm_round(r * per, u[r]);
    } else {
        for (int t0 = 0; t0 < ntiles; t0 += per) norm_round(t0, u[0]);
    }
    sync.wait();
    const float s = norm_partials(M, red);
    if (member == 0 && threadIdx.x == 0) norm_write_scales(M, s);
    const float denom = norm_denom(s);
    const bool thin = M.flags & kFlagThin;
    if constexpr (KEEP) {
        if (thin && C == 1) {
            const ThinX X(M, V, 0, 1);
            thin_clear(M, V, X, stages);
#pragma unroll
            for (int r = 0; r < kKeepRounds; ++r) {
                const int t = r * per + q;
                if (t >= ntiles) continue;
                const TileMap tm(M, t, t256);
                const bool vec = M.flags & kFlagVec4;
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    const int row = vec ? tm.vrow(k / 4) : tm.erow(k), c = vec ? tm.vcol() + k % 4 : tm.ecol(k);
                    if (row >= M.rows || c >= M.cols) continue;
                    *reinterpret_cast<_Float16*>(stages + X.at(M.tall ? c : row) + 2 * (M.tall ? row : c)) =
                        (_Float16)(u[r][k] / denom);
                }
            }
            __syncthreads();
            return true;
        }
    }
    if (member == 0 && !thin) small_x0_padding(M, V, threadIdx.x, kSmallThreads);
    if (member == 0 && thin && M.l < V.lp)   // (what thin_gram reads of it)
        for (int e = threadIdx.x; e < M.s * (V.lp - M.l); e += kSmallThreads)
            V.xw(0)[int64_t(e / (V.lp - M.l)) * V.lp + M.l + e % (V.lp - M.l)] = _Float16(0.f);
    _Float16* const tt = reinterpret_cast<_Float16*>(stages) + q * kX0Halves;
    auto x0_round = [&](int t0, const float (&ur)[16]) {
        const int t = t0 + 4 * member + q;
        small_x0_tile<BF, KEEP>(M, V, t < ntiles ? t : 0, t256, t < ntiles, denom, tt, ur);
    };
    if constexpr (KEEP) {
#pragma unroll
        for (int r = 0; r < kKeepRounds; ++r)
            if (r * per < ntiles) x0_round(r * per, u[r]);
    } else {
        for (int t0 = 0; t0 < ntiles; t0 += per) x0_round(t0, u[0]);
    }
    sync.wait();
    return false;
}

template <bool BF>
__device__ __forceinline__ bool small_fused_prologue(const OrthoMat& M, const SmallView& V, int member, int C,
                                                     float* red, char* stages, SmallSync& sync) {
    if (M.mom_tiles_r * M.mom_tiles_c <= kKeepRounds * 4 * C)
        return small_fused_prologue_as<BF, true>(M, V, member, C, red, stages, sync);
    return small_fused_prologue_as<BF, false>(M, V, member, C, red, stages, sync);
}

// After the schedule (its last barrier has made every member's u' and row sums visible): gamma and
// the row scales s_i of per-row-normalized matrices (every member computes them, into LDS while
// the rows fit, else into the matrix's rowscale, the same values from each; member 0 also stores
// gamma, as ortho_rowstats_kernel does), then p's update on this member's tiles.
constexpr int kFusedMaxScaleRows = kSmallStages * kSmallStageBytes / 4;
static_assert(kFusedMaxScaleRows * 4 + kSmallThreads * 4 <= kThinLds);
template <bool BF>
__device__ __forceinline__ void small_fused_apply(const OrthoMat& M, int member, int C, float* red, char* stages) {
    const int q = threadIdx.x / kQuarter, t256 = threadIdx.x % kQuarter;
    const bool pnn = M.flags & kFlagPNN;
    float* const sc = reinterpret_cast<float*>(stages);
    const bool staged = M.rows <= kFusedMaxScaleRows;
    const int ntiles = M.mom_tiles_r * M.mom_tiles_c, t0 = 4 * member + q, per = 4 * C;
    // p of the member's first kKeepRounds rounds, in flight while the row scales are computed
    float x[kKeepRounds][16];
#pragma unroll
    for (int r = 0; r < kKeepRounds; ++r)
        if (t0 + r * per < ntiles) tile_load<BF>(M, TileMap(M, t0 + r * per, t256), M.p, x[r]);
    float* const rows = reinterpret_cast<float*>(stages + kThinLds) - kSmallThreads;   // past sc
    const float gamma = pnn ? pnn_gamma(M, red, rows, staged ? sc : M.rowscale) : 1.f;   // its block_sum syncs them
    if (pnn && member == 0 && threadIdx.x == 0) M.scal[kScalGamma] = gamma;
    auto scale = [&](int row) { return staged ? sc[row] : ldg<float>(M.rowscale + row); };
#pragma unroll
    for (int r = 0; r < kKeepRounds; ++r)
        if (t0 + r * per < ntiles) pnn_apply_p<BF>(M, t0 + r * per, t256, M.xa, gamma, scale, x[r]);
    for (int t = t0 + kKeepRounds * per; t < ntiles; t += per) {
        tile_load<BF>(M, TileMap(M, t, t256), M.p, x[0]);
        pnn_apply_p<BF>(M, t, t256, M.xa, gamma, scale, x[0]);
    }
}

// One launch: the schedule of every small matrix in the task list, whose block map gives each block
// its matrix and its place in the matrix's cluster (thorn_ortho_fill_table gives a cluster's blocks
// one residue mod 8, so that they run on one XCD). err: set when a cluster barrier times out.
// Each operation's output is cut into super-tiles of 64 x 64 or 128 x 128 (the size that takes
// fewer rounds over the cluster, 64 on a tie) dealt to the cluster's workgroups; within one, wave
// w takes the 32 x 32 tile (w % (SM/32), w / (SM/32)).
// FUSED: the plan's whole step (small_fused_prologue, the schedule, small_fused_apply).
template <bool FUSED>
__global__ __launch_bounds__(kSmallThreads) void ns_small_kernel(const OrthoMat* __restrict__ mats, TaskList tl,
                                                                 SmallSchedule sc, int* err, int spin,
                                                                 int xcd_barriers) {
    // the ring's stages and the waves' C tiles (small_issue_c), or a thin matrix's squares
    constexpr int kRing = kSmallStages * kSmallStageBytes, kCTiles = kSmallWaves * kCTileBytes;
    __shared__ __attribute__((aligned(1024))) char stages[kRing + kCTiles > kThinLds ? kRing + kCTiles : kThinLds];
    char* const cbuf = stages + kRing;
    __shared__ float red[kSmallWaves];
    static_assert(kSmallWaves * 32 * kStageLd * 2 <= kSmallStages * kSmallStageBytes, "staging tiles in the ring");
    // the block map: (matrix, member | C << 8), or matrix -1 for a block that has no work
    const int mat = tl.map[2 * blockIdx.x];
    if (mat < 0) return;
    const int mc = tl.map[2 * blockIdx.x + 1];
    const OrthoMat& M = mats[mat];
    const int member = mc & 255, C = mc >> 8;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    _Float16* const stage = reinterpret_cast<_Float16*>(stages) + wave * 32 * kStageLd;
    const char* const ctile = cbuf + wave * kCTileBytes;
    const uint32_t ctile_lds = __builtin_amdgcn_readfirstlane(lds_address(ctile));
    const SmallView V = small_view(M);
    SmallSync sync(M.small_bar, member, C, err, spin, xcd_barriers != 0);
    const int set = M.rows == M.cols ? 0 : 1;
    const unsigned tslot = ts_begin();
    bool x0_in_lds = false;
    if constexpr (FUSED) {
        if (M.flags & kFlagBf16) x0_in_lds = small_fused_prologue<true>(M, V, member, C, red, stages, sync);
        else x0_in_lds = small_fused_prologue<false>(M, V, member, C, red, stages, sync);
    }
    ts_point(tslot, 1);

    const int thin = M.flags & kFlagThin ? V.sp / 32 : 0;
    if (thin) {
        if (!x0_in_lds) {
            const ThinX X(M, V, member, C);
            thin_clear(M, V, X, stages);
            thin_load(M, V, X, stages);
            __syncthreads();
        }
        // a case for each number of 32 x 32 tiles of s
        if (thin == 1) thin_schedule<1>(M, V, sc.op[set], sc.n[set], member, C, stages, sync, tslot);
        else if (thin == 2) thin_schedule<2>(M, V, sc.op[set], sc.n[set], member, C, stages, sync, tslot);
        else if (thin == 3) thin_schedule<3>(M, V, sc.op[set], sc.n[set], member, C, stages, sync, tslot);
        else thin_schedule<4>(M, V, sc.op[set], sc.n[set], member, C, stages, sync, tslot);
    }
    const int nops = thin ? 0 : sc.n[set];
    for (int q = 0; q < nops; ++q) {
        const SmallOp op = sc.op[set][q];
        ts_op(tslot, q, 0);
        ts_op(tslot, q, 1);   // kept by a workgroup with no super-tile in this operation
        // output rows x cols and the operands of this operation
        const int orows = V.sp, ocols = op.kind == kOpUpdate ? V.lp : V.sp;
        const _Float16 *A, *BT, *CT = nullptr;
        int64_t lda, ldb;
        int K;
        if (op.kind == kOpGram) {          // R = X X^T, K = l
            A = BT = V.xw(op.xsel);
            lda = ldb = V.lp;
            K = V.lp;
        } else if (op.kind == kOpSym) {    // out = alpha A B + beta C
            A = V.sq(op.a);
            BT = V.sqt(op.b);
            lda = ldb = V.sp;
            K = V.sp;
            if (op.c >= 0) CT = V.sqt(op.c);
        } else {                           // X' = Q X (+ beta X), K = s
            A = V.sq(op.a);
            BT = V.xwt(op.xsel);
            lda = ldb = V.sp;
            K = V.sp;
            if (op.c >= 0) CT = V.xwt(op.xsel);
        }
        // super-tiles of 64 x 64 when they take no more rounds over the cluster than 128 x 128 ones
        // (a quarter of the K-loop work per workgroup), else 128 x 128
        const int r64 = (orows + 63) / 64 * ((ocols + 63) / 64), r128 = (orows + 127) / 128 * ((ocols + 127) / 128);
        const int TS = (r64 + C - 1) / C <= (r128 + C - 1) / C ? 64 : 128;
        const int SM = min(orows, TS), SN = min(ocols, TS);
        const int SR = (orows + TS - 1) / TS, SC = (ocols + TS - 1) / TS;
        const int tm = SM / 32;
        const bool has_tile = wave < tm * (SN / 32);
        const int ti = has_tile ? wave % tm : 0, tj = has_tile ? wave / tm : 0;
        for (int st = member; st < SR * SC; st += C) {
            const int M0 = TS * (st % SR), N0 = TS * (st / SR);
            const int sm = min(SM, orows - M0), sn = min(SN, ocols - N0);
            const bool mine = has_tile && 32 * ti < sm && 32 * tj < sn;
            const int m0 = M0 + 32 * ti, n0 = N0 + 32 * tj;
            // every C^T has s_p columns
            const floatx16 acc = small_block(stages, M.zero, A, lda, BT, ldb, M0, N0, sm, sn, K, wave, lane, mine,
                                             ti, tj, ctile_lds, CT, V.sp, m0, n0, tslot, q);
            ts_op(tslot, q, 1);
            if (!mine) continue;
            half4 cv[4] = {};
            if (CT) small_read_c(cv, ctile, lane);
            const float alpha = op.kind == kOpSym ? op.alpha : 1.f;
            if (CT) small_stage<true>(acc, stage, alpha, op.beta, cv, lane);
            else small_stage<false>(acc, stage, alpha, op.beta, cv, lane);
            if (op.kind == kOpGram) {
                small_store(stage, V.sq(kBufR), V.sp, V.sqt(kBufR), V.sp, m0, n0, lane);
            } else if (op.kind == kOpSym) {
                small_store(stage, V.sq(op.o), V.sp, V.sqt(op.o), V.sp, m0, n0, lane);
                if (op.o2 >= 0) {
                    wave_lds_sync();
                    if (m0 == n0 && lane < 32 && m0 + lane < M.s) {
                        _Float16& z = stage[lane * kStageLd + lane];
                        z = static_cast<_Float16>(static_cast<float>(z) + op.dual);
                    }
                    wave_lds_sync();
                    small_store(stage, V.sq(op.o2), V.sp, V.sqt(op.o2), V.sp, m0, n0, lane);
                }
            } else if (op.fin) {
                small_store_final(stage, M, m0, n0, lane);
            } else {
                const int xo = 1 - op.xsel;
                small_store(stage, V.xw(xo), V.lp, V.xwt(xo), V.sp, m0, n0, lane);
            }
        }
        ts_op(tslot, q, 2);
        sync.wait();
    }
    ts_point(tslot, 2);
    if constexpr (FUSED) {
        if (M.flags & kFlagBf16) small_fused_apply<true>(M, member, C, red, stages);
        else small_fused_apply<false>(M, member, C, red, stages);
    }
    // kind 4 (small), fused flag, the member and the matrix's index in the plan
    ts_end(tslot, 4ull | (FUSED ? 16ull : 0ull) | (static_cast<unsigned long long>(member) << 8) |
                      (static_cast<unsigned long long>(mat) << 20));
}

}  // namespace thorn

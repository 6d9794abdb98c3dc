// The library's internal matmul call (csrc/kernels.h) for the tests: the trainer alone gives it windows, long reductions,
// a capped scratch or shared operands, and the public entry points cannot. Host code only; built beside the library.
#include "gemm_split.h"
#include "kernels.h"

using namespace dllm_hip;

// Mirrored field by field by tests/matmul_calls.py. Pointers are device memory; 0 stands for none.
struct MatmulCall {
    const float *A, *B, *Bt;
    float* C;
    int64_t a_kind, lda, ldb, ldbt, ldc, I, J, L;
    const int64_t* seg;
    int64_t nseg, seg_max;
    const float *bias, *addsrc;
    const int* addrow;
    const float *addend, *weight, *rowscale;
    float* partial;
    int64_t partial_cap;
    void* scratch;
    int64_t cap;
    float* bt_transpose;
    int64_t share, ready;
    uint32_t* stat;
};

static GemmCall call_of(const MatmulCall& m) {
    GemmCall g;
    g.Af = m.A;
    g.a_kind = static_cast<int>(m.a_kind);
    g.lda = m.lda;
    g.B = m.B;
    g.ldb = m.ldb;
    g.Bt = m.Bt;
    g.ldbt = m.ldbt;
    g.C = m.C;
    g.ldc = m.ldc;
    g.I = m.I;
    g.J = m.J;
    g.l1 = m.L;
    g.seg = m.seg;
    g.nseg = static_cast<int>(m.nseg);
    g.seg_max = m.seg_max;
    g.bias = m.bias;
    g.addsrc = m.addsrc;
    g.ld_add = m.J;
    g.seg_addrow = m.addrow;
    g.seg_addend = m.addend;
    g.ld_seg_add = m.J;
    g.seg_weight = m.weight;
    g.seg_rowscale = m.rowscale;
    g.seg_partial = m.partial;
    g.seg_partial_cap = m.partial_cap;
    g.split_scratch = m.scratch;
    g.split_cap = static_cast<size_t>(m.cap);
    g.bt_transpose = m.bt_transpose;
    g.split_share = static_cast<int>(m.share);
    g.split_ready = m.ready != 0;
    g.split_stat = m.stat;
    return g;
}

extern "C" {

// Rows per block on the int8 path: I when the call runs there whole, 0 when it runs on FP64.
int64_t matmul_rows(const MatmulCall* m) { return gemm_split_rows(call_of(*m)); }

// Whether its windows run in parallel there.
int matmul_parallel(const MatmulCall* m) { return split_plan(call_of(*m)).parallel; }

// Scratch bytes for the whole call.
int64_t matmul_bytes(const MatmulCall* m) { return static_cast<int64_t>(split_gemm_bytes(call_of(*m))); }

// The call's row blocks in order: each one's rows, its rows on the int8 path, and whether it takes B's split as made.
int64_t matmul_blocks(const MatmulCall* m, int64_t most, int64_t* rows, int64_t* on_int8, int64_t* ready) {
    const GemmCall g = call_of(*m);
    const int64_t n = gemm_split_rows(g);
    int64_t k = 0;
    for (int64_t i0 = 0; n > 0 && i0 < g.I && k < most; i0 += n, ++k) {
        const GemmCall b = gemm_split_block(g, n, i0);
        rows[k] = b.I;
        on_int8[k] = gemm_split_rows(b);
        ready[k] = b.split_ready;
    }
    return k;
}

// Whether the call, having handed back `tiles` and recomputed `chains` outputs, lost time on the int8 path.
int matmul_lost(const MatmulCall* m, uint32_t tiles, uint32_t chains) {
    return gemm_split_lost(gemm_split_cost(call_of(*m)), SplitDone{tiles, chains});
}

int matmul_run(const MatmulCall* m, hipStream_t stream) { return launch_gemm(call_of(*m), stream); }

}  // extern "C"

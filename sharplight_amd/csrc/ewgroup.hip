// Fused elementwise groups: a chain of elementwise nodes of one output shape evaluated per element in one
// launch, optionally with the row norm before it (a norm whose output only the group reads) or after it (a
// norm of one of the group's values) -- the reference lowerer's fused elementwise unit and its NormHead /
// NormTail folds (src/Sharplight.Shaders/Lowering/GraphLowerer.Fusion.cs:88-285; the generated kernels of
// ElementwiseCodegen.cs and RowNormKernelSource.cs:75-106).
//
// The group arrives as a small program (slhip_ew_program): inputs are loaded into registers 0 .. n_inputs-1,
// then each op writes its destination register; each op is the f32 arithmetic of the standalone op (ew_ops.hpp), its
// result rounded to the node's output type when that is not f32 -- so the group computes bit for bit what the
// nodes compute one launch at a time. Only the registers some reader outside the group needs are stored.
//
// Flat form (no norm): a wave takes 256 consecutive elements of one row, four per lane; every input is
// fetched before any op runs. The op codes are wave-uniform, so the interpreter's dispatch runs on the scalar
// unit while the vector unit does the arithmetic on four values per lane.
// Row form (a norm head or tail): a wave per row, two passes over it in 256-element steps: pass 1 sums the
// squares of the norm's operand (the head's input, or the tail's register after running the group, whose
// outputs it stores); pass 2 runs the group with the normalized head (and stores its outputs), or runs it
// again to normalize the tail register into y. The row's second read hits the cache.
//
// Generated form (the default): the interpreter dispatches every op of every element step on the scalar unit,
// which costs several times the arithmetic. So the first run of a program (per device, shape and types)
// generates a kernel for it -- straight-line HIP calling the same per-element functions (ewg_core.hpp) with
// the op codes, input modes and types as constants -- compiles it with hipRTC for the device's architecture
// and caches it; later runs launch it. The row form of the generated kernel keeps the norm's operand in
// registers between the passes (rows up to 4096 values), so a tail group reads its inputs and runs its ops
// once. It is compiled without floating-point contraction, so each node's result is rounded as the node
// alone rounds it. SLHIP_EWG_JIT=0 (or a failed compile) keeps the interpreter.
#include "common.hpp"
#include "ewg_core.hpp"

#include <hip/hiprtc.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>
#include <string>
#include <unordered_map>

// the text of the headers the generated kernels include (generated by the build from the sources)
#include "ewg_jit_sources.inc"

namespace slhip {

constexpr int kEwgRegs = SLHIP_EW_MAX_REGS;

struct EwgArgs {
    slhip_ew_program p;
    int64_t rows, cols;
    int pow_special[SLHIP_EW_MAX_OPS];  // Pow with a per-row or scalar exponent: the reference's special forms
};

// The register file: sixteen named four-value registers read and written through switches on the (wave-
// uniform) index, which keeps them in VGPRs -- an array indexed at run time would live in scratch memory.
struct Regs {
    f4v r0, r1, r2, r3, r4, r5, r6, r7, r8, r9, r10, r11, r12, r13, r14, r15;
#define SLHIP_EWG_CASES(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15)
    __device__ __forceinline__ f4v get(int i) const
    {
        switch (i) {
#define SLHIP_EWG_GET(k) case k: return r##k;
            SLHIP_EWG_CASES(SLHIP_EWG_GET)
#undef SLHIP_EWG_GET
        default: return r0;
        }
    }
    __device__ __forceinline__ void set(int i, f4v v)
    {
        switch (i) {
#define SLHIP_EWG_SET(k) case k: r##k = v; break;
            SLHIP_EWG_CASES(SLHIP_EWG_SET)
#undef SLHIP_EWG_SET
        default: break;
        }
    }
#undef SLHIP_EWG_CASES
};
static_assert(kEwgRegs == 16, "the register file has sixteen registers");

// Four values of input i at row r, columns c .. c + 3 (the input's mode and type are wave-uniform).
__device__ __forceinline__ f4v fetch4(const slhip_ew_input& in, int64_t r, int64_t c, int64_t cols)
{
#define SLHIP_EWG_FETCH(M)                                                                                             \
    if (in.mode == M) {                                                                                                \
        if (in.dtype == SLHIP_F32) return fetch4_t<M, SLHIP_F32>(in.data, r, c, cols);                                 \
        if (in.dtype == SLHIP_BF16) return fetch4_t<M, SLHIP_BF16>(in.data, r, c, cols);                               \
        return fetch4_t<M, SLHIP_F16>(in.data, r, c, cols);                                                            \
    }
    SLHIP_EWG_FETCH(SLHIP_EWI_ROW)
    SLHIP_EWG_FETCH(SLHIP_EWI_COL)
    SLHIP_EWG_FETCH(SLHIP_EWI_SCALAR)
    SLHIP_EWG_FETCH(SLHIP_EWI_FULL)
#undef SLHIP_EWG_FETCH
    return f4v{0.0f, 0.0f, 0.0f, 0.0f};
}

__device__ __forceinline__ void store4(void* p, int dt, int64_t off, f4v v)
{
    if (dt == SLHIP_F32) store4_t<SLHIP_F32>(p, off, v);
    else if (dt == SLHIP_BF16) store4_t<SLHIP_BF16>(p, off, v);
    else store4_t<SLHIP_F16>(p, off, v);
}

// The ops of the program on the registers.
__device__ __forceinline__ void run_ops(const EwgArgs& a, Regs& R)
{
    for (int k = 0; k < a.p.n_ops; k++) {  // uniform
        const slhip_ew_op& o = a.p.ops[k];
        f4v r = o.kind == SLHIP_EWK_BINARY ? bin4(o.op, R.get(o.a), R.get(o.b), a.pow_special[k] != 0)
                                           : un4(o.op, R.get(o.a), o.p0, o.p1);
        if (o.round != SLHIP_F32) r = round4(o.round, r);
        R.set(o.dst, r);
    }
}

__device__ __forceinline__ void fetch_inputs(const EwgArgs& a, int64_t r, int64_t c, Regs& R)
{
    for (int i = 0; i < a.p.n_inputs; i++) R.set(i, fetch4(a.p.inputs[i], r, c, a.cols));
}

__device__ __forceinline__ void store_outputs(const EwgArgs& a, int64_t r, int64_t c, const Regs& R)
{
    for (int j = 0; j < a.p.n_outputs; j++) {
        const slhip_ew_output& o = a.p.outputs[j];
        store4(o.data, o.dtype, r * a.cols + c, R.get(o.reg));
    }
}

// Flat form: wave w of the grid takes row w / spans, elements 256 (w % spans) + 4 lane .. + 3.
__global__ __launch_bounds__(256) void ewg_flat(EwgArgs a, int64_t spans)
{
    const int64_t w = static_cast<int64_t>(blockIdx.x) * 4 + wave_id();
    if (w >= a.rows * spans) return;
    const int64_t r = w / spans;
    int64_t c = (w - r * spans) * 256 + 4 * (threadIdx.x & 63);
    c = c < a.cols ? c : a.cols - 4;  // lanes past the row's end redo its last vector
    Regs R{};
    fetch_inputs(a, r, c, R);
    run_ops(a, R);
    store_outputs(a, r, c, R);
}

// Row form: one wave per row (see the file comment).
__global__ __launch_bounds__(256) void ewg_row(EwgArgs a)
{
    const int64_t r = static_cast<int64_t>(blockIdx.x) * 4 + wave_id();
    if (r >= a.rows) return;
    const int lane = threadIdx.x & 63;
    const bool head = a.p.head.kind != 0;
    const slhip_ew_norm& nm = head ? a.p.head : a.p.tail;
    Regs R{};
    // pass 1: the sum of squares of the norm's operand (tail: after the group, whose outputs are stored now)
    float q = 0.0f;
    for (int64_t c0 = 0; c0 < a.cols; c0 += 256) {
        int64_t c = c0 + 4 * lane;
        const bool own = c < a.cols;
        c = own ? c : a.cols - 4;
        fetch_inputs(a, r, c, R);
        if (!head) {
            run_ops(a, R);
            store_outputs(a, r, c, R);
        }
        const float s = sumsq4(R.get(nm.reg));
        q += own ? s : 0.0f;
    }
    q = wave_sum(q);
    // RowOp (src/Sharplight.Cpu/RowOp.cs:63-84): scale = 1 / sqrt(sum / n + eps), L2Norm 1 / sqrt(sum + eps)
    const float scale = nm.kind == SLHIP_EWN_L2 ? 1.0f / sqrtf(q + nm.eps) : 1.0f / sqrtf(q / static_cast<float>(a.cols) + nm.eps);
    // pass 2
    for (int64_t c0 = 0; c0 < a.cols; c0 += 256) {
        int64_t c = c0 + 4 * lane;
        c = c < a.cols ? c : a.cols - 4;
        fetch_inputs(a, r, c, R);
        float wv[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        if (nm.w) {
            const float4 t = *reinterpret_cast<const float4*>(nm.w + c);
            wv[0] = t.x; wv[1] = t.y; wv[2] = t.z; wv[3] = t.w;
        }
        if (head) {
            f4v h = R.get(nm.reg);
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = round_to(nm.dtype_y, (h[e] * scale) * wv[e]);
            R.set(nm.reg, h);
            run_ops(a, R);
            store_outputs(a, r, c, R);
        } else {
            run_ops(a, R);
            const f4v t = R.get(nm.reg);
            f4v y;
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = (t[e] * scale) * wv[e];
            store4(nm.y, nm.dtype_y, r * a.cols + c, y);
        }
    }
}

static int check_program(const slhip_ew_program* p, int64_t rows, int64_t cols)
{
    if (!p) return fail(SLHIP_ERR_INVALID, "ew_program: null program");
    if (rows < 0 || cols < 0) return fail(SLHIP_ERR_INVALID, "ew_program: negative shape");
    if (p->n_inputs < 1 || p->n_inputs > SLHIP_EW_MAX_INPUTS || p->n_ops < 0 || p->n_ops > SLHIP_EW_MAX_OPS ||
        p->n_outputs < 0 || p->n_outputs > SLHIP_EW_MAX_OUTPUTS)
        return fail(SLHIP_ERR_INVALID, "ew_program: %d inputs (1..%d), %d ops (0..%d), %d outputs (0..%d)", p->n_inputs,
                    SLHIP_EW_MAX_INPUTS, p->n_ops, SLHIP_EW_MAX_OPS, p->n_outputs, SLHIP_EW_MAX_OUTPUTS);
    const int nreg = SLHIP_EW_MAX_REGS;
    auto dt_ok = [](int d) { return d == SLHIP_F32 || d == SLHIP_BF16 || d == SLHIP_F16; };
    for (int i = 0; i < p->n_inputs; i++) {
        const slhip_ew_input& in = p->inputs[i];
        if (!in.data || !dt_ok(in.dtype) || in.mode < SLHIP_EWI_FULL || in.mode > SLHIP_EWI_SCALAR)
            return fail(SLHIP_ERR_INVALID, "ew_program: input %d is incomplete", i);
        if (in.mode == SLHIP_EWI_FULL || in.mode == SLHIP_EWI_ROW) {
            const uintptr_t al = in.dtype == SLHIP_F32 ? 16 : 8;
            if (reinterpret_cast<uintptr_t>(in.data) % al != 0)
                return fail(SLHIP_ERR_UNSUPPORTED, "ew_program: input %d is not %d-byte aligned", i, static_cast<int>(al));
        }
    }
    for (int k = 0; k < p->n_ops; k++) {
        const slhip_ew_op& o = p->ops[k];
        if (o.kind != SLHIP_EWK_BINARY && o.kind != SLHIP_EWK_UNARY) return fail(SLHIP_ERR_INVALID, "ew_program: op %d kind", k);
        if (o.a < 0 || o.a >= nreg || (o.kind == SLHIP_EWK_BINARY && (o.b < 0 || o.b >= nreg)) || o.dst < 0 || o.dst >= nreg)
            return fail(SLHIP_ERR_INVALID, "ew_program: op %d register out of range", k);
        if (o.kind == SLHIP_EWK_BINARY ? (o.op < SLHIP_BIN_ADD || o.op > SLHIP_BIN_FMOD)
                                       : (o.op < 0 || o.op > SLHIP_UN_IS_INF))
            return fail(SLHIP_ERR_INVALID, "ew_program: op %d code %d", k, o.op);
        if (!dt_ok(o.round)) return fail(SLHIP_ERR_INVALID, "ew_program: op %d rounding type", k);
    }
    for (int j = 0; j < p->n_outputs; j++) {
        const slhip_ew_output& o = p->outputs[j];
        if (!o.data || !dt_ok(o.dtype) || o.reg < 0 || o.reg >= nreg)
            return fail(SLHIP_ERR_INVALID, "ew_program: output %d is incomplete", j);
        if (reinterpret_cast<uintptr_t>(o.data) % (o.dtype == SLHIP_F32 ? 16 : 8) != 0)
            return fail(SLHIP_ERR_UNSUPPORTED, "ew_program: output %d is misaligned", j);
    }
    if (p->head.kind && p->tail.kind) return fail(SLHIP_ERR_INVALID, "ew_program: a norm head or a norm tail, not both");
    const slhip_ew_norm& nm = p->head.kind ? p->head : p->tail;
    if (nm.kind) {
        if (nm.kind != SLHIP_EWN_RMS && nm.kind != SLHIP_EWN_L2) return fail(SLHIP_ERR_INVALID, "ew_program: norm kind");
        if (p->head.kind && (nm.reg < 0 || nm.reg >= p->n_inputs || p->inputs[nm.reg].mode != SLHIP_EWI_FULL))
            return fail(SLHIP_ERR_INVALID, "ew_program: the norm head normalizes a full-shape input register");
        if (p->tail.kind && (nm.reg < 0 || nm.reg >= nreg || !nm.y || !dt_ok(nm.dtype_y)))
            return fail(SLHIP_ERR_INVALID, "ew_program: the norm tail is incomplete");
        if (p->head.kind && !dt_ok(nm.dtype_y)) return fail(SLHIP_ERR_INVALID, "ew_program: the norm head's type");
        if (nm.w && reinterpret_cast<uintptr_t>(nm.w) % 16 != 0) return fail(SLHIP_ERR_UNSUPPORTED, "ew_program: norm weight misaligned");
        if (p->tail.kind && reinterpret_cast<uintptr_t>(nm.y) % (nm.dtype_y == SLHIP_F32 ? 16 : 8) != 0)
            return fail(SLHIP_ERR_UNSUPPORTED, "ew_program: norm output misaligned");
    } else if (p->n_outputs == 0) {
        return fail(SLHIP_ERR_INVALID, "ew_program: nothing to store");
    }
    if (cols % 4 != 0) return fail(SLHIP_ERR_UNSUPPORTED, "ew_program: rows of %lld values (a multiple of 4 is required)",
                                   static_cast<long long>(cols));
    return SLHIP_OK;
}

// The reference's special Pow forms apply when the exponent is one value along the row (BinaryOp.Apply).
static void set_pow_special(EwgArgs& a)
{
    for (int k = 0; k < a.p.n_ops; k++) {
        const slhip_ew_op& o = a.p.ops[k];
        a.pow_special[k] = o.kind == SLHIP_EWK_BINARY && o.op == SLHIP_BIN_POW && o.b < a.p.n_inputs &&
                           (a.p.inputs[o.b].mode == SLHIP_EWI_COL || a.p.inputs[o.b].mode == SLHIP_EWI_SCALAR);
    }
}

// ---- generated kernels ------------------------------------------------------------------------------

// Register values of the generated row form kept across its two passes: rows up to this many 256-value steps.
constexpr int kJitKeepSteps = 16;

// Whether a program is of the row form with its norm's operand kept in registers: it gets two kernels, ewg_jit and
// ewg_jit_stream, which loads the full-shape inputs (each read once) and stores the norm's result with the streaming policy.
static bool jit_streams(const EwgArgs& a)
{
    return (a.p.head.kind != SLHIP_EWN_NONE || a.p.tail.kind != SLHIP_EWN_NONE) && (a.cols + 255) / 256 <= kJitKeepSteps;
}

// The streaming kernel is for launches that the caches cannot hold anyway; memory-bound either way. Rows of 4096 f32, two
// inputs, sum and norm stored, us plain / streaming: 33 MB 13.7 / 15.8, 67 MB 17.8 / 19.2, 134 MB 26.5 / 25.5, 201 MB 45.7 /
// 35.9, 268 MB 58 / 49.6, 403 MB 90 / 75, 537 MB 101.9 / 89 on buffers that rotate; on the same
// buffers in every pass 107 / 105, where the caches serve the plain loads a part of the last pass. Streaming the group's own outputs
// too loses (537 MB rotating 101), and so do two bodies in one kernel (105). The flat form is level everywhere.
constexpr int64_t kJitStreamBytes = 144ll << 20;

static bool jit_large(const EwgArgs& a)
{
    auto size = [](int dt) { return dt == SLHIP_F32 ? 4 : 2; };
    int64_t per = a.p.tail.kind ? size(a.p.tail.dtype_y) : 0;
    for (int i = 0; i < a.p.n_inputs; i++)
        if (a.p.inputs[i].mode == SLHIP_EWI_FULL) per += size(a.p.inputs[i].dtype);
    for (int k = 0; k < a.p.n_outputs; k++) per += size(a.p.outputs[k].dtype);
    return a.rows > kJitStreamBytes / (per * a.cols);  // per > 0: a row form has a full input or an output
}

static std::string fbits(float v)
{
    uint32_t u;
    memcpy(&u, &v, 4);
    char b[48];
    snprintf(b, sizeof b, "__uint_as_float(0x%08xu)", u);
    return b;
}

static const char* mode_name(int m)
{
    return m == SLHIP_EWI_ROW ? "SLHIP_EWI_ROW" : m == SLHIP_EWI_COL ? "SLHIP_EWI_COL" : m == SLHIP_EWI_SCALAR ? "SLHIP_EWI_SCALAR" : "SLHIP_EWI_FULL";
}

static const char* dt_name(int d) { return d == SLHIP_BF16 ? "SLHIP_BF16" : d == SLHIP_F16 ? "SLHIP_F16" : "SLHIP_F32"; }

// The source of the kernel for program p over rows of `cols` values (see the file comment). Every shape
// and code is a literal; the pointers and the row count are the arguments (EwgJitArgs).
static std::string jit_source(const EwgArgs& a)
{
    const slhip_ew_program& p = a.p;
    const bool head = p.head.kind != SLHIP_EWN_NONE, tail = p.tail.kind != SLHIP_EWN_NONE;
    const slhip_ew_norm& nm = head ? p.head : p.tail;
    std::string s;
    char b[512];
    auto add = [&](const char* fmt, auto... v) {
        snprintf(b, sizeof b, fmt, v...);
        s += b;
    };
    const int nv = static_cast<int>((a.cols + 255) / 256);
    const bool keep = nv <= kJitKeepSteps;
    const bool once = jit_streams(a);
    const char* end = once ? "}\nextern \"C\" __global__ __launch_bounds__(256) void ewg_jit(EwgJitArgs a) { body<false>(a); }\n"
                             "extern \"C\" __global__ __launch_bounds__(256) void ewg_jit_stream(EwgJitArgs a) { body<true>(a); }\n"
                           : "}\n";
    s += "#include \"ewg_core.hpp\"\nusing namespace slhip;\n";
    add("constexpr int64_t COLS = %lld;\n", static_cast<long long>(a.cols));
    auto fetch = [&](int i, const char* dst) {
        add("    %s = fetch4_t<%s, %s, %s>(a.in[%d], r, c, COLS);\n", dst, mode_name(p.inputs[i].mode), dt_name(p.inputs[i].dtype),
            once && p.inputs[i].mode == SLHIP_EWI_FULL ? "STREAM" : "false", i);
    };
    auto ops = [&]() {
        for (int k = 0; k < p.n_ops; k++) {
            const slhip_ew_op& o = p.ops[k];
            if (o.kind == SLHIP_EWK_BINARY)
                add("    R%d = bin4(%d, R%d, R%d, %s);\n", o.dst, o.op, o.a, o.b, a.pow_special[k] ? "true" : "false");
            else
                add("    R%d = un4(%d, R%d, %s, %s);\n", o.dst, o.op, o.a, fbits(o.p0).c_str(), fbits(o.p1).c_str());
            if (o.round != SLHIP_F32) add("    R%d = round4(%s, R%d);\n", o.dst, dt_name(o.round), o.dst);
        }
    };
    auto stores = [&]() {
        for (int j = 0; j < p.n_outputs; j++)
            add("    store4_t<%s>(a.out[%d], r * COLS + c, R%d);\n", dt_name(p.outputs[j].dtype), j, p.outputs[j].reg);
    };
    s += once ? "template <bool STREAM>\n__device__ __forceinline__ void body(const EwgJitArgs& a)\n{\n"
              : "extern \"C\" __global__ __launch_bounds__(256) void ewg_jit(EwgJitArgs a)\n{\n";
    s += "    f4v R0, R1, R2, R3, R4, R5, R6, R7, R8, R9, R10, R11, R12, R13, R14, R15;\n";
    if (!head && !tail) {
        const int64_t spans = (a.cols + 255) / 256;
        add("    const int64_t wv = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);\n"
            "    if (wv >= a.rows * %lld) return;\n"
            "    const int64_t r = wv / %lld;\n"
            "    int64_t c = (wv - r * %lld) * 256 + 4 * (threadIdx.x & 63);\n"
            "    c = c < COLS ? c : COLS - 4;\n",
            static_cast<long long>(spans), static_cast<long long>(spans), static_cast<long long>(spans));
        for (int i = 0; i < p.n_inputs; i++) {
            char d[8];
            snprintf(d, sizeof d, "R%d", i);
            fetch(i, d);
        }
        ops();
        stores();
        s += end;
        return s;
    }
    s += "    const int64_t r = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);\n"
         "    if (r >= a.rows) return;\n"
         "    const int lane = threadIdx.x & 63;\n";
    add("    constexpr int NV = %d;\n", nv);
    if (keep) s += "    f4v keep[NV];\n";
    s += "    float q = 0.0f;\n"
         "#pragma unroll\n"
         "    for (int v = 0; v < NV; v++) {\n"
         "    int64_t c = static_cast<int64_t>(v) * 256 + 4 * lane;\n"
         "    const bool own = c < COLS;\n"
         "    c = own ? c : COLS - 4;\n";
    if (head) {
        fetch(nm.reg, "R0");
        if (keep) s += "    keep[v] = R0;\n";
        s += "    q += own ? sumsq4(R0) : 0.0f;\n";
    } else {
        for (int i = 0; i < p.n_inputs; i++) {
            char d[8];
            snprintf(d, sizeof d, "R%d", i);
            fetch(i, d);
        }
        ops();
        stores();
        if (keep) add("    keep[v] = R%d;\n", nm.reg);
        add("    q += own ? sumsq4(R%d) : 0.0f;\n", nm.reg);
    }
    s += "    }\n    q = wave_sum(q);\n";
    if (nm.kind == SLHIP_EWN_L2) add("    const float scale = 1.0f / sqrtf(q + %s);\n", fbits(nm.eps).c_str());
    else add("    const float scale = 1.0f / sqrtf(q / static_cast<float>(COLS) + %s);\n", fbits(nm.eps).c_str());
    s += "#pragma unroll\n"
         "    for (int v = 0; v < NV; v++) {\n"
         "    int64_t c = static_cast<int64_t>(v) * 256 + 4 * lane;\n"
         "    c = c < COLS ? c : COLS - 4;\n";
    s += nm.w ? "    const float4 w4 = *reinterpret_cast<const float4*>(a.w + c);\n    const f4v wv = f4v{w4.x, w4.y, w4.z, w4.w};\n"
              : "    const f4v wv = f4v{1.0f, 1.0f, 1.0f, 1.0f};\n";
    if (head) {
        for (int i = 0; i < p.n_inputs; i++) {
            if (i == nm.reg) continue;
            char d[8];
            snprintf(d, sizeof d, "R%d", i);
            fetch(i, d);
        }
        if (keep) add("    R%d = keep[v];\n", nm.reg);
        else fetch(nm.reg, ("R" + std::to_string(nm.reg)).c_str());
        add("    for (int e = 0; e < 4; e++) R%d[e] = round_to(%s, (R%d[e] * scale) * wv[e]);\n", nm.reg, dt_name(nm.dtype_y), nm.reg);
        ops();
        stores();
    } else {
        if (keep) {
            s += "    const f4v t = keep[v];\n";
        } else {
            for (int i = 0; i < p.n_inputs; i++) {
                char d[8];
                snprintf(d, sizeof d, "R%d", i);
                fetch(i, d);
            }
            ops();
            add("    const f4v t = R%d;\n", nm.reg);
        }
        s += "    f4v yv;\n    for (int e = 0; e < 4; e++) yv[e] = (t[e] * scale) * wv[e];\n";
        add("    store4_t<%s, %s>(a.y, r * COLS + c, yv);\n", dt_name(nm.dtype_y), once ? "STREAM" : "false");
    }
    s += "    }\n";
    s += end;
    return s;
}

struct JitEntry {
    hipModule_t mod = nullptr;
    hipFunction_t fn = nullptr, stream = nullptr;  // stream: the row form's second kernel
    bool failed = false;
};
static std::mutex g_jit_mu;
static std::unordered_map<std::string, JitEntry> g_jit;  // key: device, then the source

// SLHIP_EWG_JIT=0 runs the interpreter (read at every run, so that a test can take both paths).
static bool jit_enabled()
{
    const char* e = getenv("SLHIP_EWG_JIT");
    return !e || atoi(e) != 0;
}

// The generated kernel for this program on the current device, or null (compile failed, or disabled: the
// interpreter runs).
static hipFunction_t jit_kernel(const EwgArgs& a, bool capturing)
{
    if (!jit_enabled()) return nullptr;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    auto pick = [&](const JitEntry& e) { return e.stream && jit_large(a) ? e.stream : e.fn; };
    const std::string src = jit_source(a);
    const std::string key = std::to_string(dev) + "\n" + src;
    std::lock_guard<std::mutex> lock(g_jit_mu);
    auto it = g_jit.find(key);
    if (it != g_jit.end()) return it->second.failed ? nullptr : pick(it->second);
    // not under stream capture (loading a module is not a capturable operation): the interpreter runs this
    // launch, the kernel is made on the next uncaptured one (or ahead of time, ew_program_prepare)
    if (capturing) return nullptr;
    JitEntry& e = g_jit[key];
    e.failed = true;
    hipDeviceProp_t props;
    if (hipGetDeviceProperties(&props, dev) != hipSuccess) return nullptr;
    std::string arch = props.gcnArchName;
    arch = arch.substr(0, arch.find(':'));
    const std::string arch_opt = "--offload-arch=" + arch;
    const char* opts[] = {arch_opt.c_str(), "-O3", "-std=c++17", "-ffp-contract=off",
                          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
    hiprtcProgram prog;
    if (hiprtcCreateProgram(&prog, src.c_str(), "ewg_jit.hip", kJitHeaderCount, kJitHeaderSources, kJitHeaderNames) != HIPRTC_SUCCESS)
        return nullptr;
    const hiprtcResult cr = hiprtcCompileProgram(prog, static_cast<int>(sizeof opts / sizeof opts[0]), opts);
    if (cr != HIPRTC_SUCCESS) {
        size_t n = 0;
        hiprtcGetProgramLogSize(prog, &n);
        std::string log(n, '\0');
        if (n) hiprtcGetProgramLog(prog, &log[0]);
        fprintf(stderr, "sharplight_hip: compiling a fused elementwise group failed (%s); the interpreter runs it\n%s\n",
                hiprtcGetErrorString(cr), log.c_str());
        hiprtcDestroyProgram(&prog);
        return nullptr;
    }
    size_t n = 0;
    hiprtcGetCodeSize(prog, &n);
    std::string code(n, '\0');
    hiprtcGetCode(prog, &code[0]);
    hiprtcDestroyProgram(&prog);
    if (hipModuleLoadData(&e.mod, code.data()) != hipSuccess || hipModuleGetFunction(&e.fn, e.mod, "ewg_jit") != hipSuccess ||
        (jit_streams(a) && hipModuleGetFunction(&e.stream, e.mod, "ewg_jit_stream") != hipSuccess)) {
        fprintf(stderr, "sharplight_hip: loading a fused elementwise group's kernel failed; the interpreter runs it\n");
        return nullptr;
    }
    e.failed = false;
    return pick(e);
}

static int jit_launch(hipFunction_t fn, const EwgArgs& a, hipStream_t st)
{
    EwgJitArgs j{};
    for (int i = 0; i < a.p.n_inputs; i++) j.in[i] = a.p.inputs[i].data;
    for (int k = 0; k < a.p.n_outputs; k++) j.out[k] = a.p.outputs[k].data;
    const slhip_ew_norm& nm = a.p.head.kind ? a.p.head : a.p.tail;
    j.w = nm.kind ? nm.w : nullptr;
    j.y = a.p.tail.kind ? a.p.tail.y : nullptr;
    j.rows = a.rows;
    const bool row_form = a.p.head.kind || a.p.tail.kind;
    const int64_t blocks = row_form ? (a.rows + 3) / 4 : (a.rows * ((a.cols + 255) / 256) + 3) / 4;
    if (blocks > 0x7FFFFFFF) return fail(SLHIP_ERR_UNSUPPORTED, "ew_program: grid too large");
    void* args[] = {&j};
    const hipError_t e = hipModuleLaunchKernel(fn, static_cast<unsigned>(blocks), 1, 1, 256, 1, 1, 0, st, args, nullptr);
    if (e != hipSuccess) return hip_fail(e, "hipModuleLaunchKernel(ewg_jit)");
    return SLHIP_OK;
}

// Makes (compiles and loads) the generated kernel of a program ahead of its first run, on the current
// device: the provider does so when it compiles a segment, so that a segment recorded into a graph later
// still launches it. The pointers in the program do not matter, nor does the row count.
int ew_program_prepare(const slhip_ew_program* prog, int64_t cols)
{
    const int st = check_program(prog, 1, cols);
    if (st != SLHIP_OK) return st;
    if (cols == 0) return SLHIP_OK;
    EwgArgs a{};
    a.p = *prog;
    a.rows = 1;
    a.cols = cols;
    set_pow_special(a);
    jit_kernel(a, false);
    return SLHIP_OK;
}

}  // namespace slhip

using namespace slhip;

extern "C" SLHIP_API int slhip_ew_program_run(const slhip_ew_program* prog, int64_t rows, int64_t cols, slhip_stream stream)
{
    const int st = check_program(prog, rows, cols);
    if (st != SLHIP_OK) return st;
    if (rows == 0 || cols == 0) return SLHIP_OK;
    EwgArgs a{};
    a.p = *prog;
    a.rows = rows;
    a.cols = cols;
    set_pow_special(a);
    hipStream_t s = to_stream(stream);
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cs) != hipSuccess) cs = hipStreamCaptureStatusNone;
    if (hipFunction_t fn = jit_kernel(a, cs != hipStreamCaptureStatusNone)) return jit_launch(fn, a, s);
    if (prog->head.kind || prog->tail.kind) {
        if (rows > 0x7FFFFFFFLL * 4) return fail(SLHIP_ERR_UNSUPPORTED, "ew_program: too many rows");
        ewg_row<<<dim3(static_cast<unsigned>((rows + 3) / 4)), 256, 0, s>>>(a);
        return check_launch("ewg_row");
    }
    const int64_t spans = (cols + 255) / 256;
    const int64_t blocks = (rows * spans + 3) / 4;
    if (blocks > 0x7FFFFFFF) return fail(SLHIP_ERR_UNSUPPORTED, "ew_program: grid too large");
    ewg_flat<<<dim3(static_cast<unsigned>(blocks)), 256, 0, s>>>(a, spans);
    return check_launch("ewg_flat");
}

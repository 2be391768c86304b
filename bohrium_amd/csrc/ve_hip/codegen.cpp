#include "codegen.hpp"

#include <bohrium/jitk/fuser.hpp>

#include <algorithm>
#include <cmath>
#include <functional>
#include <cstring>
#include <map>
#include <sstream>
#include <stdexcept>

namespace bohrium {
namespace vehip {

using jitk::Block;
using jitk::InstrPtr;
using jitk::LoopB;

const char *strategy_name(Strategy s) {
    switch (s) {
        case Strategy::MAP: return "map";
        case Strategy::FULL_REDUCE: return "reduce";
        case Strategy::SCAN: return "scan";
        case Strategy::SERIAL: return "serial";
        case Strategy::ROW_REDUCE: return "row";
        case Strategy::SEG_REDUCE: return "seg";
    }
    return "?";
}

const char *hip_type(bh_type t) {
    switch (t) {
        case bh_type::BOOL: return "bool";
        case bh_type::INT8: return "int8_t";
        case bh_type::INT16: return "int16_t";
        case bh_type::INT32: return "int32_t";
        case bh_type::INT64: return "int64_t";
        case bh_type::UINT8: return "uint8_t";
        case bh_type::UINT16: return "uint16_t";
        case bh_type::UINT32: return "uint32_t";
        case bh_type::UINT64: return "uint64_t";
        case bh_type::FLOAT32: return "float";
        case bh_type::FLOAT64: return "double";
        case bh_type::COMPLEX64: return "bh_c64";
        case bh_type::COMPLEX128: return "bh_c128";
        case bh_type::R123: return "uint64_t";
    }
    throw std::runtime_error("hip_type(): unknown type");
}

bool divides_by_power_of_two(const bh_instruction &i) {
    if (i.opcode != BH_DIVIDE || i.operand.size() != 3 || !i.operand[2].isConstant()) return false;
    int e = 0;
    if (i.constant.type == bh_type::FLOAT64 && i.operand_type(0) == bh_type::FLOAT64)
        return std::fabs(std::frexp(i.constant.value.float64, &e)) == 0.5 && std::abs(e - 1) <= 1022;
    if (i.constant.type == bh_type::FLOAT32 && i.operand_type(0) == bh_type::FLOAT32)
        return std::fabs(std::frexp(i.constant.value.float32, &e)) == 0.5 && std::abs(e - 1) <= 126;
    return false;
}

namespace {

// ------------------------------------------------------------------ helpers

bool sweeping_innermost_axis(const bh_instruction &i) {
    return bh_opcode_is_sweep(i.opcode) && i.sweep_axis() == i.operand[1].ndim - 1;
}

bool is_complex_op(const bh_instruction &i, int idx) { return bh_type_is_complex(i.operand_type(idx)); }

const char *cplx_prefix(bh_type t) { return t == bh_type::COMPLEX64 ? "make_c64" : "make_c128"; }

// Conversion with C99 assignment semantics.
std::string cast_expr(bh_type to, bh_type from, const std::string &e) {
    const bool cto = bh_type_is_complex(to), cfrom = bh_type_is_complex(from);
    if (!cto && !cfrom) return "((" + std::string(hip_type(to)) + ")(" + e + "))";
    if (cto && !cfrom) {
        const char *f = to == bh_type::COMPLEX64 ? "float" : "double";
        return std::string(cplx_prefix(to)) + "((" + f + ")(" + e + "), (" + f + ")0)";
    }
    if (cto && cfrom) {
        const char *f = to == bh_type::COMPLEX64 ? "float" : "double";
        return std::string(cplx_prefix(to)) + "((" + f + ")(" + e + ").real, (" + f + ")(" + e + ").imag)";
    }
    if (to == bh_type::BOOL) return "((" + e + ").real != 0 || (" + e + ").imag != 0)";
    return "((" + std::string(hip_type(to)) + ")(" + e + ").real)";
}

// Scalar body of one instruction; `ops` are the rendered operands in the
// reference's order (out, in1, in2, ...).  Semantics follow the reference's
// write_operation() for C99 (core/jitk/instruction.cpp:58-544).
std::string hip_operation(const bh_instruction &instr, const std::vector<std::string> &ops, bool math64) {
    std::ostringstream o;
    const auto &a = ops;
    auto bin = [&](const char *op) { o << a[0] << " = " << a[1] << " " << op << " " << a[2] << ";"; };
    auto un = [&](const char *fn, const char *cfn) {
        if (bh_type_is_complex(instr.operand_type(1)) && cfn != nullptr)
            o << a[0] << " = " << cfn << "(" << a[1] << ");";
        else
            o << a[0] << " = " << fn << "(" << a[1] << ");";
    };
    switch (instr.opcode) {
        case BH_BITWISE_AND: bin("&"); break;
        case BH_BITWISE_AND_REDUCE: o << a[0] << " = " << a[0] << " & " << a[1] << ";"; break;
        case BH_BITWISE_OR: bin("|"); break;
        case BH_BITWISE_OR_REDUCE: o << a[0] << " = " << a[0] << " | " << a[1] << ";"; break;
        case BH_BITWISE_XOR: bin("^"); break;
        case BH_BITWISE_XOR_REDUCE: o << a[0] << " = " << a[0] << " ^ " << a[1] << ";"; break;
        case BH_LOGICAL_NOT: o << a[0] << " = !" << a[1] << ";"; break;
        case BH_LOGICAL_OR: bin("||"); break;
        case BH_LOGICAL_OR_REDUCE: o << a[0] << " = " << a[0] << " || " << a[1] << ";"; break;
        case BH_LOGICAL_AND: bin("&&"); break;
        case BH_LOGICAL_AND_REDUCE: o << a[0] << " = " << a[0] << " && " << a[1] << ";"; break;
        case BH_LOGICAL_XOR: o << a[0] << " = !" << a[1] << " != !" << a[2] << ";"; break;
        case BH_LOGICAL_XOR_REDUCE: o << a[0] << " = !" << a[0] << " != !" << a[1] << ";"; break;
        case BH_LEFT_SHIFT: bin("<<"); break;
        case BH_RIGHT_SHIFT: bin(">>"); break;
        case BH_GREATER: bin(">"); break;
        case BH_GREATER_EQUAL: bin(">="); break;
        case BH_LESS: bin("<"); break;
        case BH_LESS_EQUAL: bin("<="); break;
        case BH_MAXIMUM: o << a[0] << " = " << a[1] << " > " << a[2] << " ? " << a[1] << " : " << a[2] << ";"; break;
        case BH_MAXIMUM_REDUCE:
            o << a[0] << " = " << a[0] << " > " << a[1] << " ? " << a[0] << " : " << a[1] << ";";
            break;
        case BH_MINIMUM: o << a[0] << " = " << a[1] << " < " << a[2] << " ? " << a[1] << " : " << a[2] << ";"; break;
        case BH_MINIMUM_REDUCE:
            o << a[0] << " = " << a[0] << " < " << a[1] << " ? " << a[0] << " : " << a[1] << ";";
            break;
        case BH_INVERT:
            if (instr.operand[0].base->dtype() == bh_type::BOOL)
                o << a[0] << " = !" << a[1] << ";";
            else
                o << a[0] << " = ~" << a[1] << ";";
            break;
        case BH_MOD:
            if (bh_type_is_float(instr.operand[0].base->dtype()))
                o << a[0] << " = fmod(" << a[1] << ", " << a[2] << ");";
            else
                o << a[0] << " = " << a[1] << " % " << a[2] << ";";
            break;
        case BH_REMAINDER: {
            const bh_type t = instr.operand[0].base->dtype();
            if (bh_type_is_float(t)) {
                o << a[0] << " = " << a[1] << " - floor(" << a[1] << " / " << a[2] << ") * " << a[2] << ";";
            } else if (bh_type_is_unsigned_integer(t)) {
                o << a[0] << " = " << a[1] << " % " << a[2] << ";";
            } else {  // Python/NumPy sign convention
                o << a[0] << " = ((" << a[1] << " > 0) == (" << a[2] << " > 0) || (" << a[1] << " % " << a[2]
                  << ") == 0) ? (" << a[1] << " % " << a[2] << ") : (" << a[1] << " % " << a[2] << ") + " << a[2]
                  << ";";
            }
            break;
        }
        case BH_RINT: un("rint", nullptr); break;
        case BH_EXP2: un("exp2", nullptr); break;
        case BH_EXPM1: un("expm1", nullptr); break;
        case BH_LOG1P: un("log1p", nullptr); break;
        case BH_ARCSIN: un("asin", nullptr); break;
        case BH_ARCCOS: un("acos", nullptr); break;
        case BH_ARCTAN: un("atan", nullptr); break;
        case BH_ARCTAN2: o << a[0] << " = atan2(" << a[1] << ", " << a[2] << ");"; break;
        case BH_ARCSINH: un("asinh", nullptr); break;
        case BH_ARCCOSH: un("acosh", nullptr); break;
        case BH_ARCTANH: un("atanh", nullptr); break;
        case BH_FLOOR: un("floor", nullptr); break;
        case BH_CEIL: un("ceil", nullptr); break;
        case BH_TRUNC: un("trunc", nullptr); break;
        case BH_LOG2: un("log2", nullptr); break;
        case BH_ISNAN:
        case BH_ISINF:
        case BH_ISFINITE: {
            const char *fn = instr.opcode == BH_ISNAN ? "isnan" : (instr.opcode == BH_ISINF ? "isinf" : "isfinite");
            const bh_type t = instr.operand_type(1);
            if (bh_type_is_complex(t)) {
                o << a[0] << " = " << fn << "((" << a[1] << ").real);";
            } else if (bh_type_is_float(t)) {
                o << a[0] << " = " << fn << "(" << a[1] << ");";
            } else {
                o << a[0] << " = " << (instr.opcode == BH_ISFINITE ? "true" : "false") << ";";
            }
            break;
        }
        case BH_CONJ: o << a[0] << " = bh_conj(" << a[1] << ");"; break;
        case BH_RANGE:
        case BH_RANDOM:
        case BH_GATHER:
        case BH_SCATTER: o << a[0] << " = " << a[1] << ";"; break;
        case BH_COND_SCATTER: o << "if (" << a[2] << ") { " << a[0] << " = " << a[1] << "; }"; break;
        case BH_SIN: un("sin", "bh_csin"); break;
        case BH_COS: un("cos", "bh_ccos"); break;
        case BH_TAN: un("tan", "bh_ctan"); break;
        case BH_SINH: un("sinh", "bh_csinh"); break;
        case BH_COSH: un("cosh", "bh_ccosh"); break;
        case BH_TANH: un("tanh", "bh_ctanh"); break;
        case BH_EXP: un(math64 && instr.operand_type(1) == bh_type::FLOAT64 ? "bh_exp64" : "exp", "bh_cexp"); break;
        case BH_ABSOLUTE: {
            const bh_type t = instr.operand_type(1);
            if (t == bh_type::BOOL || bh_type_is_unsigned_integer(t)) {
                o << a[0] << " = " << a[1] << ";";
            } else if (bh_type_is_float(t)) {
                o << a[0] << " = fabs(" << a[1] << ");";
            } else if (t == bh_type::INT64) {
                o << a[0] << " = llabs(" << a[1] << ");";
            } else if (bh_type_is_complex(t)) {
                o << a[0] << " = abs((int)(" << a[1] << ").real);";  // C99 cast of a complex to int
            } else {
                o << a[0] << " = abs((int)" << a[1] << ");";
            }
            break;
        }
        case BH_SQRT: un("sqrt", "bh_csqrt"); break;
        case BH_LOG: un(math64 && instr.operand_type(1) == bh_type::FLOAT64 ? "bh_log64" : "log", "bh_clog"); break;
        case BH_NOT_EQUAL: bin("!="); break;
        case BH_EQUAL: bin("=="); break;
        case BH_POWER:
            if (bh_type_is_complex(instr.operand_type(0))) {
                o << a[0] << " = bh_cpow(" << a[1] << ", " << a[2] << ");";
            } else if (bh_type_is_integer(instr.operand_type(0)) || instr.operand_type(0) == bh_type::BOOL) {
                o << a[0] << " = bh_pow_int((double) " << a[1] << ", (double)" << a[2] << ");";
            } else {
                o << a[0] << " = pow(" << a[1] << ", " << a[2] << ");";
            }
            break;
        case BH_ADD: bin("+"); break;
        case BH_ADD_REDUCE: o << a[0] << " += " << a[1] << ";"; break;
        case BH_ADD_ACCUMULATE: bin("+"); break;
        case BH_SUBTRACT: bin("-"); break;
        case BH_MULTIPLY: bin("*"); break;
        case BH_MULTIPLY_REDUCE: o << a[0] << " *= " << a[1] << ";"; break;
        case BH_MULTIPLY_ACCUMULATE: bin("*"); break;
        case BH_DIVIDE:
            if (bh_type_is_signed_integer(instr.operand[0].base->dtype())) {  // NumPy floor division
                o << a[0] << " = ((" << a[1] << " > 0) != (" << a[2] << " > 0) && (" << a[1] << " % " << a[2]
                  << ") != 0)?(" << a[1] << " / " << a[2] << " - 1):(" << a[1] << " / " << a[2] << ");";
            } else if (divides_by_power_of_two(instr)) {
                // x / 2^k is x * 2^-k to the last bit, and the reciprocal leaves the loop (an IEEE float64 division
                // is 11 instructions, one at a quarter of the rate; every uniform draw divides by 2^64)
                const char *t = instr.operand_type(0) == bh_type::FLOAT32 ? "float" : "double";
                o << a[0] << " = " << a[1] << " * ((" << t << ")1 / " << a[2] << ");";
            } else {
                bin("/");
            }
            break;
        case BH_IDENTITY:
            o << a[0] << " = " << cast_expr(instr.operand_type(0), instr.operand_type(1), a[1]) << ";";
            break;
        case BH_LOG10:
            if (bh_type_is_complex(instr.operand_type(0))) {
                const bh_type t = instr.operand_type(0);
                o << a[0] << " = bh_clog(" << a[1] << ") / " << cplx_prefix(t) << "(log(10.0f), 0);";
            } else {
                o << a[0] << " = log10(" << a[1] << ");";
            }
            break;
        case BH_REAL: o << a[0] << " = bh_creal(" << a[1] << ");"; break;
        case BH_IMAG: o << a[0] << " = bh_cimag(" << a[1] << ");"; break;
        case BH_SIGN: {
            const bh_type t = instr.operand_type(0);
            if (bh_type_is_complex(t)) {
                const char *ft = t == bh_type::COMPLEX64 ? "float" : "double";
                o << "{ " << ft << " re_ = (" << a[1] << ").real, im_ = (" << a[1] << ").imag; " << a[0] << " = "
                  << cplx_prefix(t) << "(re_ == 0 ? ((im_ > 0) - (0 > im_)) : ((re_ > 0) - (0 > re_)), 0); }";
            } else {
                o << a[0] << " = ((" << a[1] << " > 0) - (0 > " << a[1] << "));";
            }
            break;
        }
        default:
            throw std::runtime_error(std::string("hip engine: instruction not supported: ") +
                                     bh_opcode_text(instr.opcode));
    }
    return o.str();
}

// The binary operator of a reduction/accumulate as an expression of (x, y).
std::string combine_expr(bh_opcode op, const std::string &x, const std::string &y) {
    switch (op) {
        case BH_ADD_REDUCE:
        case BH_ADD_ACCUMULATE: return "(" + x + " + " + y + ")";
        case BH_MULTIPLY_REDUCE:
        case BH_MULTIPLY_ACCUMULATE: return "(" + x + " * " + y + ")";
        case BH_MINIMUM_REDUCE: return "(" + x + " < " + y + " ? " + x + " : " + y + ")";
        case BH_MAXIMUM_REDUCE: return "(" + x + " > " + y + " ? " + x + " : " + y + ")";
        case BH_LOGICAL_AND_REDUCE: return "(" + x + " && " + y + ")";
        case BH_LOGICAL_OR_REDUCE: return "(" + x + " || " + y + ")";
        case BH_LOGICAL_XOR_REDUCE: return "(!" + x + " != !" + y + ")";
        case BH_BITWISE_AND_REDUCE: return "(" + x + " & " + y + ")";
        case BH_BITWISE_OR_REDUCE: return "(" + x + " | " + y + ")";
        case BH_BITWISE_XOR_REDUCE: return "(" + x + " ^ " + y + ")";
        default: throw std::runtime_error("combine_expr(): not a sweep");
    }
}

std::string literal(const bh_constant &c) {
    std::ostringstream s;
    c.write_literal(s);
    return s.str();
}

// A view key that ignores size-1 dimensions (which never change an address).
struct VKey {
    const bh_base *base;
    int64_t start;
    std::vector<std::pair<int64_t, int64_t> > dims;
    bool operator<(const VKey &o) const {
        if (base != o.base) return base < o.base;
        if (start != o.start) return start < o.start;
        return dims < o.dims;
    }
};
VKey vkey(const bh_view &v) {
    VKey k{v.base, v.start, {}};
    for (int64_t d = 0; d < v.ndim; ++d)
        if (v.shape[d] > 1) k.dims.emplace_back(v.shape[d], v.stride[d]);
    return k;
}

// Key of an offset-and-strides argument group: views with equal start and strides share it.
typedef std::pair<int64_t, std::vector<int64_t> > OSKey;
OSKey oskey(const bh_view &v) { return {v.start, std::vector<int64_t>(v.stride.begin(), v.stride.end())}; }

struct Scope {
    const Scope *parent = nullptr;
    std::set<const bh_base *> tmps;
    std::set<VKey> srep;
    // Scalar-replaced reduction outputs declared by this scope and stored when it closes.
    std::vector<std::pair<const bh_view *, int64_t> > wb;
    // Temporaries that stand for an accumulator of an enclosing skeleton (collapsed reductions).
    std::map<const bh_base *, std::string> alias;
    // Input views already loaded into a register of this name (unrolled grid-stride groups).
    std::map<VKey, std::string> preload;
    const std::string *preloadOf(const bh_view &v) const {
        if (!preload.empty()) {
            auto it = preload.find(vkey(v));
            if (it != preload.end()) return &it->second;
        }
        return parent ? parent->preloadOf(v) : nullptr;
    }
    bool isTmp(const bh_base *b) const { return tmps.count(b) || (parent && parent->isTmp(b)); }
    bool isSrep(const bh_view &v) const { return srep.count(vkey(v)) || (parent && parent->isSrep(v)); }
    const std::string *aliasOf(const bh_base *b) const {
        auto it = alias.find(b);
        if (it != alias.end()) return &it->second;
        return parent ? parent->aliasOf(b) : nullptr;
    }
    bool isArray(const bh_view &v) const { return !(isTmp(v.base) || isSrep(v) || aliasOf(v.base)); }
    bool isDeclared(const bh_view &v) const { return isTmp(v.base) || isSrep(v); }
};

void indent(std::ostringstream &o, int n) { o << std::string(n * 2, ' '); }

// ------------------------------------------------------------------ writer

// Results are stored past the caches (non-temporal) when the kernel's arrays together fill the 256 MB last-level cache:
// they would not stay there anyway, and what is kept out of it stays for the input's next reader.  Measured, cached ->
// non-temporal: 200 sweeps of the 8192^2 float32 stencil 23.9 -> 22.1 ms; where three kernels read one 197 MB array before
// the result is stored, row statistics 156 -> 126 us and column statistics 176 -> 147 us; x*2+1 into 256 MiB 105 -> 83 us,
// into 144 MiB 52 -> 45, into 128 (256 with its input) 42.8 -> 40.3, and with the result's maximum taken next 68 -> 67;
// running counts of 22e6 float32 (255 MiB) 96 -> 85.  Below the limit the two are level: of 17e6 (195 MiB) 78 and 81, int16 -> float32
// into 152 MiB 38.2 and 37.9.
// Only where they pay, which the same measurements bound:
//  - the lanes store neighbouring pieces of at most 16 bytes.  y[::8] = s*2 into 1 GiB 516 -> 1666 us with
//    non-temporal stores, g.T[...] = q*2 4.5 -> 12.3 ms, 1 GiB of bool -> int64 354 -> 712 us at 32 bytes a lane, but
//    238 -> 190 at 16;
//  - rows of the written view, where it is not contiguous, that hold a wave's store (64 lanes of 16 bytes);
//  - the kernel reads at least an eighth of what it stores.  400 MiB written and nothing read: 72 -> 96 us.
constexpr int64_t kStreamBytes = 240ll << 20;
constexpr int64_t kStreamStore = 128ll << 20;  // (a smaller result beside large inputs stays for its reader)
constexpr int64_t kStreamRead = 8;
constexpr int64_t kStreamRow = 64 * 16;

// Bytes of the base that a view reaches (broadcast axes count once).
int64_t reached_bytes(const bh_view &v) {
    int64_t n = bh_type_size(v.base->dtype());
    for (int64_t d = 0; d < v.ndim; ++d)
        if (v.stride[d] != 0) n *= v.shape[d];
    return n;
}

struct KernelParam {
    std::string type;  // value type: "double *", "int64_t", ...
    std::string name;
    bool is_ptr;
};

// ---- MAP over tiles: read-only views whose contiguous axis is not the innermost loop's (transposed
// operands).  In the flat walk each of a wave's lanes reads such a view one row apart: 64 requests of
// a cache line for 64 elements, bound by the L2 request rate.  Here a workgroup takes a T x T tile of
// the two axes, copies the transposed views' tile through LDS with its lanes along their contiguous
// axis, and computes with its lanes along the innermost axis (a row of T + 1 elements in LDS, so
// neither direction conflicts).  Measured on 4096^2 float32: a.T * 1 64.4 -> 29.0 us (4.6 TB/s),
// (a + a.T) * 0.5 70.1 -> 36.8 us.
struct TiledForm {
    int64_t q = -1;  // the axis along which the transposed views are contiguous
    std::vector<const bh_view *> views;
    int side = 0;    // T
};

// Tiled from 2^20 elements on, or where a transposed view has 6 MB, half as much again as one XCD's L2: below, the L2s
// hold the lines of the flat walk until their other elements are asked for, and a tile is two rounds of latency for one.
// Flat / tiled, device us: x + x.T float32 512^2 6.3 / 6.2, 724^2 6.8 / 9.4, 860^2 7.8 / 9.6, 1024^2 8.7 / 6.6, x + y.T 1300^2
// 15.2 / 12.8; four maps of which two are tiled float64 760^2 28.4 / 31.2, 960^2 36.3 / 29.1; x.T * 1.5 and x + x.T together
// complex128 512^2 13.2 / 14.1, 860^2 26.2 / 17.6.
constexpr uint64_t kTileMinItems = 1u << 20;
constexpr int64_t kTileMinBytes = 6 << 20;

TiledForm tiled_form(const std::vector<const LoopB *> &chain, uint64_t p, const std::vector<const bh_view *> &reads) {
    TiledForm f;
    if (p < 2) return f;
    uint64_t total = 1;
    for (uint64_t r = 0; r < p; ++r) total *= static_cast<uint64_t>(std::max<int64_t>(0, chain[r]->size));
    const int64_t a = static_cast<int64_t>(p) - 1;
    int bytes = 0;
    int64_t largest = 0;
    for (const bh_view *v : reads) {
        if (v->ndim <= a || v->hasSlide()) continue;
        if (v->stride[a] == 0 || std::abs(v->stride[a]) < 8) continue;
        int64_t q = -1;
        for (int64_t r = 0; r < a; ++r)
            if (std::abs(v->stride[r]) == 1) q = r;
        if (q < 0 || (f.q >= 0 && f.q != q)) continue;
        f.q = q;
        f.views.push_back(v);
        const int sz = bh_type_size(v->base->dtype());
        bytes += sz;
        largest = std::max(largest, reached_bytes(*v));
    }
    if (total < kTileMinItems && largest < kTileMinBytes) return TiledForm();
    if (f.views.empty() || chain[a]->size < 32 || chain[f.q]->size < 32) return TiledForm();
    f.side = 65 * 64 * bytes <= 40960 ? 64 : 32;
    while (33 * 32 * bytes > 65536) {
        bytes -= bh_type_size(f.views.back()->base->dtype());
        f.views.pop_back();
    }
    return f;
}

class Writer {
public:
    Writer(const LoopB &unit, const WriterConfig &cfg) : unit(unit), cfg(cfg) { collect(); }

    KernelPlan plan(Strategy s);

private:
    const LoopB &unit;
    const WriterConfig &cfg;
    KernelPlan kp;

    std::map<const bh_base *, int> bid;
    std::vector<const bh_base *> base_order;
    std::set<const bh_base *> always_array;
    std::set<bh_base *> temps;
    std::map<VKey, int> vid;
    std::map<OSKey, int> osid;
    std::vector<const bh_view *> os_views;
    // Sliding views get an offset argument of their own, re-read from (origin, operand) at launch.
    std::map<const bh_view *, std::pair<int64_t, int> > sliding_src;
    std::map<const LoopB *, int> lid;
    std::vector<const LoopB *> loops;
    std::vector<InstrPtr> const_instrs;
    std::vector<InstrPtr> const_params;  // one instruction per distinct constant: parameter c<j>
    std::map<int64_t, int> const_of_origin;
    std::set<const bh_base *> index_checked;  // bases needing their element count (gather/scatter)
    // Instructions a skeleton implements itself (collapsed reductions and their identities).
    std::set<const bh_instruction *> skip;
    // ROW_REDUCE: the inner loop whose iterations are spread over the 64 lanes of a wave.
    std::set<const LoopB *> lane_loops;  // loops strided by the lanes of a wave (row skeleton)
    bool fence_lanes = false;            // order the lanes' memory accesses after each lane loop
    // Instruction replaced by "store its input into `scan_sink`" in the scan skeleton.
    const bh_instruction *scan_instr = nullptr;
    std::string scan_sink;

    /* Launch-shape arguments of a skeleton (plan-time values passed as kernel arguments, so that the
     * source does not depend on the sizes). */
    std::vector<std::pair<std::string, int64_t> > shape_args;

    std::ostringstream body;
    // FULL_REDUCE, SEG_REDUCE: the main kernel's body while `body` holds the finalize's
    std::string main_body;

    void collect();
    int view_id(const bh_view &v) {
        auto it = vid.find(vkey(v));
        if (it != vid.end()) return it->second;
        const int id = static_cast<int>(vid.size());
        vid[vkey(v)] = id;
        return id;
    }
    int os_id(const bh_view &v) {
        if (v.hasSlide()) {
            OSKey k{INT64_MIN, {static_cast<int64_t>(reinterpret_cast<uintptr_t>(&v))}};
            auto it = osid.find(k);
            if (it != osid.end()) return it->second;
            const int id = static_cast<int>(os_views.size());
            osid[k] = id;
            os_views.push_back(&v);
            return id;
        }
        auto it = osid.find(oskey(v));
        if (it != osid.end()) return it->second;
        const int id = static_cast<int>(os_views.size());
        osid[oskey(v)] = id;
        os_views.push_back(&v);
        return id;
    }
    std::string name(const Scope &sc, const bh_view &v) {
        std::ostringstream s;
        if (const std::string *a = sc.aliasOf(v.base)) return *a;
        if (sc.isTmp(v.base)) {
            s << "t" << bid.at(v.base);
        } else if (sc.isSrep(v)) {
            s << "s" << bid.at(v.base) << "_" << view_id(v);
        } else {
            s << "a" << bid.at(v.base);
        }
        return s.str();
    }
    // Strides are part of the plan key, so views with equal strides share one parameter (and the
    // compiler one product i * stride for all of them, e.g. the five loads of a stencil).
    std::map<int64_t, int> stride_ids;
    std::vector<int64_t> stride_vals;
    int stride_id(int64_t stride) {
        auto it = stride_ids.find(stride);
        if (it != stride_ids.end()) return it->second;
        const int id = static_cast<int>(stride_vals.size());
        stride_ids[stride] = id;
        stride_vals.push_back(stride);
        return id;
    }
    std::string index(const bh_view &v, int hidden_axis = BH_MAXDIM, int off_axis = -1, int off = 0) {
        std::ostringstream s;
        const int k = os_id(v);
        s << "vo" << k;
        if (!v.is_scalar()) {
            // Strides are part of the plan key, so unit and zero strides are spelled out.
            for (int64_t d = 0; d < v.ndim; ++d) {
                int64_t t = d >= hidden_axis ? d + 1 : d;
                if (v.stride[d] == 0) continue;
                if (t == off_axis)
                    s << " + (i" << t << " + (i" << t << " == 0 ? 0 : " << off << "))";
                else
                    s << " + i" << t;
                if (v.stride[d] != 1) s << " * vs" << stride_id(v.stride[d]);
            }
        }
        return s.str();
    }
    std::string ref(const Scope &sc, const bh_view &v, int hidden_axis = BH_MAXDIM) {
        if (const std::string *p = sc.preloadOf(v)) return *p;
        std::string n = name(sc, v);
        if (sc.isArray(v)) n += "[" + index(v, hidden_axis) + "]";
        return n;
    }
    std::string const_ref(const bh_instruction &i) { return "c" + std::to_string(const_of_origin.at(i.origin_id)); }

    /* The rank that the lanes of a wave walk in the code being written (-1: one thread, or no such rank), and the
     * neighbouring elements of it that one lane owns. */
    int64_t lane_axis = -1;
    int lane_run = 1;
    /* Whether stores to `v` go past the caches (kStreamBytes). */
    bool streamed(const bh_view &v) const;
    void declare_scope(const LoopB &l, Scope &sc, int ind);
    void write_back(const LoopB &l, Scope &sc, int ind);
    void emit_block(const Block &b, Scope &sc, int ind);
    void emit_blocks(const LoopB &l, Scope &sc, int ind);
    void emit_body(const LoopB &l, const Scope *parent, int ind);
    void emit_instr(const bh_instruction &i, Scope &sc, int ind);

    /* One element of a grid-stride loop: `decode(ind)` derives the loop indices from f_,
     * `compute(ind, outer)` emits the body in a scope whose parent is `outer`. */
    struct Element {
        std::function<void(int)> decode;
        std::function<void(int, const Scope *)> compute;
        const LoopB *body_loop = nullptr;  // innermost loop whose read-only inputs may be preloaded
        const Scope *outer = nullptr;
        /* A 2-D iteration (i0 outer, i1 inner of this extent): without unrolling, the two indices
         * are advanced by the grid stride instead of being divided out of f_ for every element. */
        std::string inner;
        /* decode is i0 = f_ (one rank): an unrolled group of consecutive f_ touches consecutive
         * elements of every unit-stride view. */
        bool unit = false;
    };
    /* Grid-stride over [0, tot).  With `parts`, the range is cut into min(8, bh_nblk) contiguous
     * parts, part x walked by the workgroups b with b mod 8 = x (the workgroups one XCD runs), so a
     * stencil's neighbouring rows are read by the workgroups of one L2. */
    void grid_stride(const std::string &tot, int unroll, const Element &e);
    bool parts = false;
    /* A 2-D stencil's walk by column groups and row bands; false (nothing emitted) when the body is none.
     * Sets the number of thread tasks. */
    bool stencil_walk(const Element &e, const std::string &n0, const std::string &n1, int64_t s0, int64_t s1, int unroll,
                      int64_t *tasks);
    std::vector<const bh_view *> preloadable(const LoopB &l);
    void emit_map();
    void emit_map_tiled(const TiledForm &f, const std::vector<const LoopB *> &chain, uint64_t p, const Scope &ksc);
    void emit_row_reduce();
    void emit_seg_reduce();
    void emit_full_reduce();
    void emit_scan();
    void emit_serial();
    std::vector<KernelParam> parameters();
};

void Writer::collect() {
    std::vector<InstrPtr> all = jitk::allInstr(unit);
    for (const InstrPtr &i : all) {
        for (const bh_view &v : i->operand) {
            if (v.isConstant()) continue;
            if (!bid.count(v.base)) {
                bid[v.base] = static_cast<int>(bid.size());
                base_order.push_back(v.base);
            }
        }
        if (bh_opcode_is_accumulate(i->opcode)) {
            always_array.insert(i->operand[0].base);
        } else if (i->opcode == BH_GATHER) {
            always_array.insert(i->operand[1].base);
            index_checked.insert(i->operand[1].base);
        } else if (i->opcode == BH_SCATTER || i->opcode == BH_COND_SCATTER) {
            always_array.insert(i->operand[0].base);
            index_checked.insert(i->operand[0].base);
        }
        // (a sweep's constant is its axis: it shapes the loops and is no argument.  The fuser rewrites it
        // when it swaps axes, so shared with an equal constant it would be re-read from the flush as the
        // axis that the program named.)
        if (i->has_constant() && !bh_opcode_is_sweep(i->opcode)) const_instrs.push_back(i);
    }
    for (const bh_base *b : unit.getAllFrees()) {
        if (!bid.count(b)) {
            bid[b] = static_cast<int>(bid.size());
            base_order.push_back(b);
        }
    }
    std::sort(const_instrs.begin(), const_instrs.end(),
              [](const InstrPtr &a, const InstrPtr &b) { return a->origin_id < b->origin_id; });
    // Constants of equal type and value share one parameter (a loop body repeats 1.0, 0.5, its
    // coefficients ...; each parameter takes SGPRs, and past the SGPR budget the compiler spills them
    // to VGPR lanes and reads them back in every iteration).  The flush key records which constants
    // of a flush are equal, so a cached plan is reused only where the same ones are.
    for (size_t j = 0; j < const_instrs.size(); ++j) {
        const bh_constant &c = const_instrs[j]->constant;
        int id = -1;
        if (c.type != bh_type::R123) {
            for (size_t k = 0; k < const_params.size() && id < 0; ++k) {
                const bh_constant &d = const_params[k]->constant;
                if (d.type == c.type && std::memcmp(&d.value, &c.value, bh_type_size(c.type)) == 0)
                    id = static_cast<int>(k);
            }
        }
        if (id < 0) {
            id = static_cast<int>(const_params.size());
            const_params.push_back(const_instrs[j]);
        }
        const_of_origin[const_instrs[j]->origin_id] = id;
    }
    temps = unit.getAllTemps();
    std::set<bh_base *> non_temps = unit.getAllNonTemps();
    for (const bh_base *b : always_array) non_temps.insert(const_cast<bh_base *>(b));
    for (const InstrPtr &i : all)
        for (const bh_view &v : i->operand)
            if (!v.isConstant() && non_temps.count(v.base) &&
                std::find(kp.params.begin(), kp.params.end(), v.base) == kp.params.end())
                kp.params.push_back(v.base);
    for (const InstrPtr &i : all) {
        if (i->operand.empty() || i->operand[0].isConstant()) continue;
        if (non_temps.count(i->operand[0].base)) kp.written.insert(i->operand[0].base);
    }
    // Loop ids (pre-order) for the size arguments.
    std::vector<const LoopB *> stack{&unit};
    while (!stack.empty()) {
        const LoopB *l = stack.back();
        stack.pop_back();
        if (l->rank >= 0 && !lid.count(l)) {
            lid[l] = static_cast<int>(loops.size());
            loops.push_back(l);
        }
        for (auto it = l->_block_list.rbegin(); it != l->_block_list.rend(); ++it)
            if (!it->isInstr()) stack.push_back(&it->getLoop());
    }
    // Register every view's offset-and-stride group in instruction order.
    for (const InstrPtr &i : all) {
        for (size_t o = 0; o < i->operand.size(); ++o) {
            const bh_view &v = i->operand[o];
            if (v.isConstant()) continue;
            os_id(v);
            if (v.hasSlide()) sliding_src[&v] = {i->origin_id, static_cast<int>(o)};
        }
    }
}

bool Writer::streamed(const bh_view &v) const {
    if (lane_axis < 0 || v.ndim <= lane_axis || v.stride[lane_axis] != 1 || bh_type_is_complex(v.base->dtype())) return false;
    const int64_t size = bh_type_size(v.base->dtype());
    if (lane_run * size > 16) return false;
    if (!v.isContiguous() && v.shape[lane_axis] * size < kStreamRow) return false;
    // The kernel's arrays, by what it reaches of each.
    std::map<const bh_base *, int64_t> all, read;
    for (const InstrPtr &i : jitk::allInstr(unit)) {
        if (bh_opcode_is_system(i->opcode)) continue;
        for (size_t o = 0; o < i->operand.size(); ++o) {
            const bh_view &w = i->operand[o];
            if (w.isConstant() || std::find(kp.params.begin(), kp.params.end(), w.base) == kp.params.end()) continue;
            const int64_t n = reached_bytes(w);
            all[w.base] = std::max(all[w.base], n);
            if (o > 0) read[w.base] = std::max(read[w.base], n);
        }
    }
    int64_t total = 0, loaded = 0;
    for (const auto &b : all) total += b.second;
    for (const auto &b : read) loaded += b.second;
    const int64_t stored = reached_bytes(v);
    return total >= kStreamBytes && stored >= kStreamStore && loaded * kStreamRead >= stored;
}

void Writer::declare_scope(const LoopB &l, Scope &sc, int ind) {
    const std::set<bh_base *> local_tmps = l.getLocalTemps();
    for (const InstrPtr &i : jitk::allInstr(l)) {
        for (const bh_view &v : i->operand) {
            if (v.isConstant() || !local_tmps.count(v.base)) continue;
            if (sc.isDeclared(v) || always_array.count(v.base)) continue;
            sc.tmps.insert(v.base);
            indent(body, ind);
            body << hip_type(v.base->dtype()) << " t" << bid.at(v.base) << ";\n";
        }
    }
    for (const Block &b : l._block_list) {
        if (b.isInstr()) continue;
        for (const InstrPtr &i : jitk::allLocalInstr(b.getLoop())) {
            if (!(bh_opcode_is_reduction(i->opcode) && sweeping_innermost_axis(*i))) continue;
            const bh_view &v = i->operand[0];
            if (sc.isDeclared(v) || always_array.count(v.base)) continue;
            sc.srep.insert(vkey(v));
            sc.wb.emplace_back(&v, i->sweep_axis());
            indent(body, ind);
            body << hip_type(v.base->dtype()) << " s" << bid.at(v.base) << "_" << view_id(v) << ";\n";
        }
    }
}

// Store the scope's scalar-replaced reduction outputs once, after the loops that sweep them.
void Writer::write_back(const LoopB &, Scope &sc, int ind) {
    for (const auto &w : sc.wb) {
        const bh_view &v = *w.first;
        indent(body, ind);
        body << "a" << bid.at(v.base) << "[" << index(v, static_cast<int>(w.second)) << "] = s" << bid.at(v.base) << "_"
             << view_id(v) << ";\n";
    }
    sc.wb.clear();
}

void Writer::emit_block(const Block &b, Scope &sc, int ind) {
    if (b.isInstr()) {
        if (b.getInstr() != nullptr && !bh_opcode_is_system(b.getInstr()->opcode) && !skip.count(b.getInstr().get()))
            emit_instr(*b.getInstr(), sc, ind);
        return;
    }
    const LoopB &c = b.getLoop();
    const bool lanes = lane_loops.count(&c) != 0;
    if (lanes && fence_lanes) {
        indent(body, ind);
        body << "__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, \"workgroup\");\n";
    }
    indent(body, ind);
    if (lanes) {
        body << "for (int64_t i" << c.rank << " = lane_; i" << c.rank << " < n" << lid.at(&c) << "; i" << c.rank
             << " += 64) {\n";
    } else {
        body << "for (int64_t i" << c.rank << " = 0; i" << c.rank << " < n" << lid.at(&c) << "; ++i" << c.rank << ") {\n";
    }
    emit_body(c, &sc, ind + 1);
    indent(body, ind);
    body << "}\n";
    if (!lanes) return;
    if (fence_lanes) {
        // Elements written by one lane are read or overwritten by another (before and after every
        // lane loop): the wave's memory accesses so far complete before it goes on (the lanes share
        // one CU's L1).
        indent(body, ind);
        body << "__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, \"workgroup\");\n";
    }
    // Fold the lanes' partial reductions; every lane ends with the row's value.
    for (const InstrPtr &sw : c._sweeps) {
        const bh_view &v = sw->operand[0];
        const std::string var = ref(sc, v, static_cast<int>(sw->sweep_axis()));
        if (var.empty() || var[0] == 'a') throw std::logic_error("row skeleton: a reduction output is not in a register");
        const std::string T = hip_type(v.base->dtype());
        indent(body, ind);
        body << var << " = bh_wave_reduce(" << var << ", [](" << T << " x, " << T << " y) -> " << T << " { return "
             << combine_expr(sw->opcode, "x", "y") << "; });\n";
    }
}

void Writer::emit_blocks(const LoopB &l, Scope &sc, int ind) {
    for (const Block &b : l._block_list) emit_block(b, sc, ind);
}

void Writer::emit_body(const LoopB &l, const Scope *parent, int ind) {
    if (l.isSystemOnly()) return;
    Scope sc;
    sc.parent = parent;
    declare_scope(l, sc, ind);
    emit_blocks(l, sc, ind);
    write_back(l, sc, ind);
}

void Writer::emit_instr(const bh_instruction &instr, Scope &sc, int ind) {
    std::vector<std::string> ops;
    indent(body, ind);
    if (&instr == scan_instr) {
        body << scan_sink << " = " << ref(sc, instr.operand[1]) << ";\n";
        return;
    }
    if (instr.opcode == BH_RANGE) {
        ops.push_back(ref(sc, instr.operand[0]));
        ops.push_back("(" + index(instr.operand[0]) + ")");
    } else if (instr.opcode == BH_RANDOM) {
        ops.push_back(ref(sc, instr.operand[0]));
        const std::string c = const_ref(instr);
        ops.push_back("bh_random123(" + c + "_start, " + c + "_key, " + index(instr.operand[0]) + ")");
    } else if (instr.opcode == BH_GATHER) {
        // out[...] = in[in.start + idx[...]], with the index checked against the base.  No branch: an
        // index outside the base loads element 0 and marks bh_bad_, which raises the error flag when
        // the function ends; a body without branches keeps the loads of several elements in flight.
        const bh_view &in = instr.operand[1];
        const int k = os_id(in);
        const std::string out = ref(sc, instr.operand[0]);
        body << "{ const int64_t g_ = vo" << k << " + (int64_t)(" << ref(sc, instr.operand[2]) << "); "
             << "const bool ok_ = (uint64_t)g_ < (uint64_t)nb" << bid.at(in.base) << "; bh_bad_ |= !ok_; "
             << out << " = a" << bid.at(in.base) << "[ok_ ? g_ : (int64_t)0]; }\n";
        kp.uses_gather_flag = true;
        kp.uses_index_check = true;
        kp.uses_error_flag = true;
        return;
    } else if (instr.opcode == BH_SCATTER || instr.opcode == BH_COND_SCATTER) {
        const bh_view &out = instr.operand[0];
        const int k = os_id(out);
        body << "{ const int64_t g_ = vo" << k << " + (int64_t)(" << ref(sc, instr.operand[2]) << "); ";
        if (instr.opcode == BH_COND_SCATTER) body << "if (" << ref(sc, instr.operand[3]) << ") ";
        body << "{ if (g_ < 0 || g_ >= nb" << bid.at(out.base) << ") { atomicOr(bh_err, BH_ERR_INDEX); } else { a"
             << bid.at(out.base) << "[g_] = " << ref(sc, instr.operand[1]) << "; } } }\n";
        kp.uses_index_check = true;
        kp.uses_error_flag = true;
        return;
    } else if (bh_opcode_is_accumulate(instr.opcode)) {
        ops.push_back(ref(sc, instr.operand[0]));
        ops.push_back(name(sc, instr.operand[0]) + "[" +
                      index(instr.operand[0], BH_MAXDIM, instr.sweep_axis(), -1) + "]");
        ops.push_back(ref(sc, instr.operand[1]));
    } else {
        for (size_t o = 0; o < instr.operand.size(); ++o) {
            const bh_view &v = instr.operand[o];
            if (v.isConstant()) {
                ops.push_back(bh_opcode_is_sweep(instr.opcode) ? std::string() : const_ref(instr));
            } else if (o == 0 && bh_opcode_is_reduction(instr.opcode) && instr.operand[1].ndim > 1) {
                ops.push_back(ref(sc, v, instr.sweep_axis()));
            } else {
                ops.push_back(ref(sc, v));
            }
        }
    }
    const bh_view &out = instr.operand[0];
    if (sc.isArray(out) && !bh_opcode_is_sweep(instr.opcode) && instr.opcode != BH_COND_SCATTER && streamed(out)) {
        const std::string at = ops[0];
        ops[0] = "nt_";
        body << "{ " << hip_type(out.base->dtype()) << " nt_; " << hip_operation(instr, ops, cfg.math64)
             << " __builtin_nontemporal_store(nt_, &" << at << "); }\n";
        return;
    }
    body << hip_operation(instr, ops, cfg.math64) << "\n";
}

std::vector<KernelParam> Writer::parameters() {
    std::vector<KernelParam> params;
    auto lit = [&](const std::string &type, const std::string &name, const void *p, int size, int align) {
        params.push_back({type, name, false});
        ArgSpec a;
        a.kind = ArgSpec::LITERAL;
        a.bytes.assign(static_cast<const uint8_t *>(p), static_cast<const uint8_t *>(p) + size);
        a.size = size;
        a.align = align;
        kp.args.push_back(a);
    };
    for (bh_base *b : kp.params) {
        params.push_back({std::string(hip_type(b->dtype())) + " *", "a" + std::to_string(bid.at(b)), true});
        ArgSpec a;
        a.kind = ArgSpec::BASE_PTR;
        a.base = b;
        kp.args.push_back(a);
    }
    for (size_t k = 0; k < os_views.size(); ++k) {
        const bh_view &v = *os_views[k];
        lit("int64_t", "vo" + std::to_string(k), &v.start, 8, 8);
        auto src = sliding_src.find(&v);
        if (src != sliding_src.end()) {
            kp.args.back().view_origin = src->second.first;
            kp.args.back().view_operand = src->second.second;
        } else if (v.hasSlide()) {
            kp.reusable = false;
        }
    }
    for (size_t j = 0; j < stride_vals.size(); ++j) lit("int64_t", "vs" + std::to_string(j), &stride_vals[j], 8, 8);
    for (size_t j = 0; j < loops.size(); ++j) lit("int64_t", "n" + std::to_string(j), &loops[j]->size, 8, 8);
    for (const bh_base *b : index_checked) {
        const int64_t n = b->nelem();
        lit("int64_t", "nb" + std::to_string(bid.at(b)), &n, 8, 8);
    }
    for (const auto &a : shape_args) lit("int64_t", a.first, &a.second, 8, 8);
    for (size_t j = 0; j < const_params.size(); ++j) {
        const bh_constant &c = const_params[j]->constant;
        const std::string cn = "c" + std::to_string(j);
        if (c.type == bh_type::R123) {
            lit("uint64_t", cn + "_start", &c.value.r123.start, 8, 8);
            kp.args.back().const_origin = const_params[j]->origin_id;
            kp.args.back().const_part = 0;
            lit("uint64_t", cn + "_key", &c.value.r123.key, 8, 8);
            kp.args.back().const_origin = const_params[j]->origin_id;
            kp.args.back().const_part = 1;
        } else {
            const int size = bh_type_size(c.type);
            const int align = bh_type_is_complex(c.type) ? size / 2 : size;
            lit(hip_type(c.type), cn, &c.value, size, align);
            kp.args.back().const_origin = const_params[j]->origin_id;
        }
    }
    if (kp.uses_error_flag) {
        params.push_back({"unsigned int *", "bh_err", true});
        ArgSpec a;
        a.kind = ArgSpec::ERRFLAG_PTR;
        kp.args.push_back(a);
    }
    return params;
}

// ---- MAP: grid-stride over the flattened leading parallel ranks
// Input views of an innermost loop that can be loaded before any of its instructions run:
// reads of parameter arrays that no instruction of the loop writes (not gathered, scattered
// or accumulated).  Distinct views in first-use order.
std::vector<const bh_view *> Writer::preloadable(const LoopB &l) {
    std::set<const bh_base *> written;
    for (const InstrPtr &i : jitk::allInstr(l))
        if (!i->operand.empty() && !i->operand[0].isConstant()) written.insert(i->operand[0].base);
    std::vector<const bh_view *> out;
    std::set<VKey> seen;
    for (const InstrPtr &i : jitk::allInstr(l)) {
        if (bh_opcode_is_system(i->opcode) || i->opcode == BH_GATHER) continue;
        for (size_t o = 1; o < i->operand.size(); ++o) {
            const bh_view &v = i->operand[o];
            if (v.isConstant() || written.count(v.base) || always_array.count(v.base)) continue;
            if (std::find(kp.params.begin(), kp.params.end(), v.base) == kp.params.end()) continue;
            if (seen.insert(vkey(v)).second) out.push_back(&v);
        }
    }
    return out;
}

// Grid-stride loop over the flat index f_ in [0, tot).  With unroll > 1, full groups of
// `unroll` elements first load every read-only input of all of them into registers and then
// compute them, so a wave has all of its loads in flight at once; the remaining elements run one
// at a time.  A group is `unroll` consecutive elements on a one-rank walk without XCD parts (a
// unit-stride view's loads merge into wide loads), else `unroll` elements strided by the grid.

// Full reductions of at most this many elements can be one workgroup's (kernels of one code share it over their
// sizes; from here on the autotuner works on the main loop).
constexpr uint64_t kOneWorkgroupItems = 1u << 20;
// Full reductions with at most this many instructions in their loop count as light (half the grid).
constexpr size_t kLightReduceInstrs = 16;

namespace {
// A base read through two or more different views in `l` (a stencil: neighbouring elements of one
// array read at once).
bool shifted_reads(const LoopB &l) {
    std::map<const bh_base *, std::set<std::vector<int64_t> > > views;
    for (const InstrPtr &i : jitk::allInstr(l)) {
        for (size_t o = 1; o < i->operand.size(); ++o) {
            const bh_view &v = i->operand[o];
            if (v.isConstant()) continue;
            std::vector<int64_t> key{v.start, v.ndim};
            for (int64_t d = 0; d < v.ndim; ++d) {
                key.push_back(v.shape[d]);
                key.push_back(v.stride[d]);
            }
            auto &set = views[v.base];
            set.insert(key);
            if (set.size() > 1) return true;
        }
    }
    return false;
}
} // namespace

// ---- stencil walk of a 2-D iteration (i0 of s0, i1 of s1): neighbouring elements of one array read through
// several views.  Element by element each view is a load of its own (5 loads of 4 bytes and their index
// arithmetic per point of a 5-point stencil: about 60 VALU instructions, which bounded the sweep at half the
// copy rate).  Here a thread owns V neighbouring columns and walks down a band of rows with a window of the
// array in registers: every element of the band is loaded once per thread (16-byte loads of the V columns
// plus the side columns), and a group of `ur` rows is loaded before it is computed.  Measured on the 8192^2
// float32 5-point sweep with max|new - old|: 134 -> 103 us (4.0 -> 5.2 TB/s; a plain copy reaches 5.6), 200 sweeps
// 27.3 -> 21.3 ms (23.9 of them without the stores past the caches, kStreamBytes).
namespace {
// A window: the views of one base with equal strides, as offsets (row, column) from the first.
struct Window {
    const bh_view *first = nullptr;
    std::map<VKey, std::pair<int, int> > taps;
    std::vector<const bh_view *> views;
};

// Windows of the read-only views `reads` of a 2-D loop nest (two or more views each, unit column stride,
// offsets within 3 rows and 8 columns).
std::vector<Window> stencil_windows(const std::vector<const bh_view *> &reads) {
    std::vector<Window> out;
    for (const bh_view *v : reads) {
        if (v->ndim != 2 || v->stride[1] != 1 || v->hasSlide() || v->stride[0] < 16) continue;
        bool placed = false;
        for (Window &w : out) {
            if (w.first->base != v->base || w.first->stride[0] != v->stride[0]) continue;
            const int64_t s0 = v->stride[0], d = v->start - w.first->start;
            const int64_t dr = d >= 0 ? (d + s0 / 2) / s0 : -((-d + s0 / 2) / s0), dc = d - dr * s0;
            if (std::abs(dr) > 3 || std::abs(dc) > 8) continue;
            w.taps[vkey(*v)] = {static_cast<int>(dr), static_cast<int>(dc)};
            w.views.push_back(v);
            placed = true;
            break;
        }
        if (placed) continue;
        Window w;
        w.first = v;
        w.taps[vkey(*v)] = {0, 0};
        w.views.push_back(v);
        out.push_back(w);
    }
    out.erase(std::remove_if(out.begin(), out.end(), [](const Window &w) { return w.taps.size() < 2; }), out.end());
    return out;
}

// Fewer elements than this (2^20: 1024^2, 256 workgroups of single row groups) leave too few bands to fill the chip,
// and their arrays stay in the L2s, where the element walk's repeated loads are cheap.  Element walk / this, device us of
// the 5-point sum: float32 512^2 6.3 / 6.2, 1024^2 6.9 / 6.6, 1500^2 8.3 / 8.1, 4096^2 28.2 / 23.7; float64 512^2 6.4 / 6.4,
// 1024^2 8.5 / 7.0, 1500^2 12.2 / 9.8, 4096^2 61 / 45.
constexpr int64_t kStencilMinItems = 1 << 20;
} // namespace

bool Writer::stencil_walk(const Element &e, const std::string &n0, const std::string &n1, int64_t s0, int64_t s1,
                          int unroll, int64_t *tasks) {
    if (e.body_loop == nullptr || s0 * s1 < kStencilMinItems || s0 * s1 >= (1ll << 31) || s1 < 64) return false;
    const std::vector<const bh_view *> reads = preloadable(*e.body_loop);
    const std::vector<Window> wins = stencil_windows(reads);
    if (wins.empty()) return false;
    std::vector<const bh_view *> others;
    int widest = 1;
    for (const bh_view *v : reads) {
        widest = std::max(widest, bh_type_size(v->base->dtype()));
        bool in = false;
        for (const Window &w : wins) in |= w.taps.count(vkey(*v)) != 0;
        if (!in) others.push_back(v);
    }
    const int V = std::max(1, std::min(4, 16 / widest));
    const int UR = std::max(2, std::min(8, unroll));
    if (s1 / V < 16) return false;
    // Bands of up to 8 row groups, fewer when the bands would not give every CU 8 workgroups.
    const int64_t groups = s1 / V;
    int64_t H = 8 * UR;
    while (H > UR && ((s0 + H - 1) / H) * groups < 256ll * 8 * kp.block) H -= UR;
    shape_args.emplace_back("st_h", H);
    lane_axis = 1;
    lane_run = V;
    *tasks = (s0 + H - 1) / H * groups;

    // Columns of window k that row j of a row group needs: those of the taps that touch it.
    auto need = [&](const Window &w, int j) {
        std::set<int> c;
        for (const auto &t : w.taps)
            if (j - t.second.first >= 0 && j - t.second.first < UR)
                for (int v = 0; v < V; ++v) c.insert(t.second.second + v);
        return c;
    };
    auto reg = [](size_t k, int j, int c) {
        auto num = [](int x) { return (x < 0 ? "m" : "p") + std::to_string(std::abs(x)); };
        return "w" + std::to_string(k) + "_" + num(j) + "_" + num(c);
    };
    auto load = [&](int ind, size_t k, int j, int c, const std::string &row) {
        const bh_view &v = *wins[k].first;
        indent(body, ind);
        body << reg(k, j, c) << " = a" << bid.at(v.base) << "[vo" << os_id(v) << " + (" << row << " + " << j << ") * vs"
             << stride_id(v.stride[0]) << " + (c0_ + " << c << ")];\n";
    };
    body << "  const int64_t ng_ = " << n1 << " / " << V << ", nt_ = (" << n0 << " + st_h - 1) / st_h * ng_;\n";
    if (parts) {
        body << "  const unsigned px_ = bh_nblk < BH_XCDS ? bh_nblk : BH_XCDS;\n";
        body << "  const unsigned pw_ = bh_nblk / px_ + (bh_bid % px_ < bh_nblk % px_ ? 1u : 0u);\n";
        body << "  const int64_t pt_ = ((nt_ + px_ - 1) / px_ + BH_WG - 1) / BH_WG * BH_WG;\n";
        body << "  const int64_t p0_ = (int64_t)(bh_bid % px_) * pt_;\n";
        body << "  const int64_t pe_ = p0_ + pt_ < nt_ ? p0_ + pt_ : nt_;\n";
        body << "  const int64_t st_ = (int64_t)pw_ * BH_WG;\n";
        body << "  int64_t g_ = p0_ + (int64_t)(bh_bid / px_) * BH_WG + threadIdx.x;\n";
    } else {
        body << "  const int64_t pe_ = nt_, st_ = (int64_t)bh_nblk * BH_WG;\n";
        body << "  int64_t g_ = (int64_t)bh_bid * BH_WG + threadIdx.x;\n";
    }
    body << "  for (; g_ < pe_; g_ += st_) {\n";
    body << "    const int64_t b_ = (int64_t)((uint32_t)g_ / (uint32_t)ng_), c0_ = (g_ - b_ * ng_) * " << V << ";\n";
    body << "    int64_t r_ = b_ * st_h;\n    const int64_t re_ = r_ + st_h < " << n0 << " ? r_ + st_h : " << n0 << ";\n";
    body << "    if (r_ + " << UR << " <= re_) {\n";
    struct Span {
        int lo, hi;
    };
    std::vector<Span> span;
    for (size_t k = 0; k < wins.size(); ++k) {
        Span s{0, 0};
        for (const auto &t : wins[k].taps) {
            s.lo = std::min(s.lo, t.second.first);
            s.hi = std::max(s.hi, t.second.first);
        }
        span.push_back(s);
        const std::string T = hip_type(wins[k].first->base->dtype());
        // the rows that a group takes over from the one before it
        for (int j = s.lo; j < s.hi; ++j)
            for (int c : need(wins[k], j)) body << "      " << T << " " << reg(k, j, c) << ";\n";
        for (int j = s.lo; j < s.hi; ++j) {
            const std::set<int> have = need(wins[k], j + UR);
            for (int c : need(wins[k], j))
                if (have.count(c)) load(3, k, j, c, "r_");
        }
    }
    body << "      for (; r_ + " << UR << " <= re_; r_ += " << UR << ") {\n";
    for (size_t k = 0; k < wins.size(); ++k) {
        const std::string T = hip_type(wins[k].first->base->dtype());
        for (int j = span[k].hi; j < UR + span[k].hi; ++j)
            for (int c : need(wins[k], j)) body << "        " << T << " " << reg(k, j, c) << ";\n";
        for (int j = span[k].lo; j < UR + span[k].hi; ++j) {
            const std::set<int> have = j < span[k].hi ? need(wins[k], j + UR) : std::set<int>();
            for (int c : need(wins[k], j))
                if (!have.count(c)) load(4, k, j, c, "r_");
        }
    }
    auto ld = [&](size_t k, int u, int v) {
        return "ld" + std::to_string(k) + "_" + std::to_string(u) + "_" + std::to_string(v);
    };
    auto at = [&](int u, int v) {
        body << "        {\n          const int64_t i0 = r_ + " << u << ", i1 = c0_ + " << v << ";\n";
    };
    for (size_t k = 0; k < others.size(); ++k)
        for (int u = 0; u < UR; ++u)
            for (int v = 0; v < V; ++v)
                body << "        " << hip_type(others[k]->base->dtype()) << " " << ld(k, u, v) << ";\n";
    for (int u = 0; u < UR; ++u)
        for (int v = 0; v < V && !others.empty(); ++v) {
            at(u, v);
            for (size_t k = 0; k < others.size(); ++k) body << "          " << ld(k, u, v) << " = " << ref(*e.outer, *others[k]) << ";\n";
            body << "        }\n";
        }
    for (int u = 0; u < UR; ++u)
        for (int v = 0; v < V; ++v) {
            Scope pre;
            pre.parent = e.outer;
            for (size_t k = 0; k < others.size(); ++k) pre.preload[vkey(*others[k])] = ld(k, u, v);
            for (size_t k = 0; k < wins.size(); ++k)
                for (const auto &t : wins[k].taps)
                    pre.preload[t.first] = reg(k, u + t.second.first, v + t.second.second);
            at(u, v);
            e.compute(5, &pre);
            body << "        }\n";
        }
    for (size_t k = 0; k < wins.size(); ++k)
        for (int j = span[k].lo; j < span[k].hi; ++j) {
            const std::set<int> have = need(wins[k], j + UR);
            for (int c : need(wins[k], j))
                if (have.count(c)) body << "        " << reg(k, j, c) << " = " << reg(k, j + UR, c) << ";\n";
        }
    body << "      }\n    }\n";
    // the band's last rows, element by element
    body << "    for (; r_ < re_; ++r_)\n      for (int v_ = 0; v_ < " << V << "; ++v_) {\n        const int64_t i0 = r_, i1 = c0_ + v_;\n";
    e.compute(4, e.outer);
    body << "      }\n  }\n";
    if (V > 1) {
        // the columns past the last whole group
        body << "  const int64_t cr_ = " << n1 << " - ng_ * " << V << ";\n";
        body << "  if (cr_ > 0)\n    for (int64_t f_ = (int64_t)bh_bid * BH_WG + threadIdx.x; f_ < cr_ * " << n0
             << "; f_ += (int64_t)bh_nblk * BH_WG) {\n";
        body << "      const int64_t i0 = f_ / cr_, i1 = ng_ * " << V << " + (f_ - i0 * cr_);\n";
        e.compute(3, e.outer);
        body << "    }\n";
    }
    return true;
}

void Writer::grid_stride(const std::string &tot_in, int unroll, const Element &e) {
    std::string tot = tot_in;
    if (parts) {
        // Part x of X = min(8, bh_nblk) holds [x * pt_, (x + 1) * pt_); its workgroups are
        // b = x, x + X, ... (q_ or q_ + 1 of them), each taking every whole workgroup's worth in turn.
        body << "  const unsigned px_ = bh_nblk < BH_XCDS ? bh_nblk : BH_XCDS;\n";
        body << "  const unsigned pw_ = bh_nblk / px_ + (bh_bid % px_ < bh_nblk % px_ ? 1u : 0u);\n";
        body << "  const int64_t pt_ = ((" << tot << " + px_ - 1) / px_ + BH_WG - 1) / BH_WG * BH_WG;\n";
        body << "  const int64_t p0_ = (int64_t)(bh_bid % px_) * pt_;\n";
        body << "  const int64_t pe_ = p0_ + pt_ < " << tot << " ? p0_ + pt_ : " << tot << ";\n";
        body << "  const int64_t st_ = (int64_t)pw_ * BH_WG;\n";
        body << "  int64_t g_ = p0_ + (int64_t)(bh_bid / px_) * BH_WG + threadIdx.x;\n";
        tot = "pe_";
    } else {
        body << "  const int64_t st_ = (int64_t)bh_nblk * BH_WG;\n";
        body << "  int64_t g_ = (int64_t)bh_bid * BH_WG + threadIdx.x;\n";
    }
    lane_run = unroll > 1 && e.unit && !parts ? unroll : 1;
    if (lane_run > 1) {
        // Groups of `unroll` consecutive elements: group q_ is [q_ * unroll, q_ * unroll + unroll), the
        // groups are walked grid-stride, so a lane's loads of one unit-stride view are adjacent (the
        // compiler merges them into one wide load, e.g. 16 bytes for 4 floats) and a wave's lanes read
        // consecutive 4 * unroll-byte pieces.  The last tot % unroll elements go to the first threads.
        const std::vector<const bh_view *> reads =
            e.body_loop != nullptr ? preloadable(*e.body_loop) : std::vector<const bh_view *>();
        const std::string U = std::to_string(unroll);
        body << "  const int64_t g0_ = g_, ng_ = " << tot << " / " << U << ";\n";
        body << "  for (; g_ < ng_; g_ += st_) {\n";
        for (int u = 0; u < unroll; ++u)
            for (size_t k = 0; k < reads.size(); ++k)
                body << "    " << hip_type(reads[k]->base->dtype()) << " ld" << k << "_" << u << ";\n";
        for (int u = 0; u < unroll; ++u) {
            if (reads.empty()) break;
            body << "    {\n      const int64_t f_ = g_ * " << U << " + " << u << ";\n";
            e.decode(3);
            for (size_t k = 0; k < reads.size(); ++k)
                body << "      ld" << k << "_" << u << " = " << ref(*e.outer, *reads[k]) << ";\n";
            body << "    }\n";
        }
        for (int u = 0; u < unroll; ++u) {
            Scope pre;
            pre.parent = e.outer;
            for (size_t k = 0; k < reads.size(); ++k)
                pre.preload[vkey(*reads[k])] = "ld" + std::to_string(k) + "_" + std::to_string(u);
            body << "    {\n      const int64_t f_ = g_ * " << U << " + " << u << ";\n";
            e.decode(3);
            e.compute(3, &pre);
            body << "    }\n";
        }
        body << "  }\n";
        body << "  g_ = ng_ * " << U << " + g0_;\n";
        body << "  if (g_ < " << tot << ") {\n";
        body << "    const int64_t f_ = g_;\n";
        e.decode(2);
        e.compute(2, e.outer);
        body << "  }\n";
        return;
    }
    if (unroll > 1) {
        const std::vector<const bh_view *> reads =
            e.body_loop != nullptr ? preloadable(*e.body_loop) : std::vector<const bh_view *>();
        body << "  for (; g_ + " << unroll - 1 << " * st_ < " << tot << "; g_ += " << unroll << " * st_) {\n";
        for (int u = 0; u < unroll; ++u)
            for (size_t k = 0; k < reads.size(); ++k)
                body << "    " << hip_type(reads[k]->base->dtype()) << " ld" << k << "_" << u << ";\n";
        for (int u = 0; u < unroll; ++u) {
            if (reads.empty()) break;
            body << "    {\n      const int64_t f_ = g_ + " << u << " * st_;\n";
            e.decode(3);
            for (size_t k = 0; k < reads.size(); ++k)
                body << "      ld" << k << "_" << u << " = " << ref(*e.outer, *reads[k]) << ";\n";
            body << "    }\n";
        }
        for (int u = 0; u < unroll; ++u) {
            Scope pre;
            pre.parent = e.outer;
            for (size_t k = 0; k < reads.size(); ++k)
                pre.preload[vkey(*reads[k])] = "ld" + std::to_string(k) + "_" + std::to_string(u);
            body << "    {\n      const int64_t f_ = g_ + " << u << " * st_;\n";
            e.decode(3);
            e.compute(3, &pre);
            body << "    }\n";
        }
        body << "  }\n";
    }
    if (unroll <= 1 && !e.inner.empty()) {
        const std::string &n = e.inner;
        body << "  int64_t i0_ = g_ / " << n << ", i1_ = g_ - i0_ * " << n << ";\n";
        body << "  const int64_t sq_ = st_ / " << n << ", sr_ = st_ - sq_ * " << n << ";\n";
        body << "  for (; g_ < " << tot << "; g_ += st_) {\n";
        body << "    const int64_t i0 = i0_, i1 = i1_;\n";
        e.compute(2, e.outer);
        body << "    i1_ += sr_;\n    i0_ += sq_;\n    if (i1_ >= " << n << ") { i1_ -= " << n << "; ++i0_; }\n";
        body << "  }\n";
        return;
    }
    body << "  for (; g_ < " << tot << "; g_ += st_) {\n";
    body << "    const int64_t f_ = g_;\n";
    e.decode(2);
    e.compute(2, e.outer);
    body << "  }\n";
}

// The inner loop of a row reduction: the innermost parallel loop of `l0` holds only constant
// IDENTITY seeds of the reductions of one innermost sub-loop (and frees), and that sub-loop's
// sweeps are all reductions over its own rank.  Null when `l0` has another form.
// The loops a wave's 64 lanes stride when a block runs one wave per row: every loop directly
// inside the innermost leading parallel loop P (at least one with 32 or more iterations), whose own
// sweeps are reductions over their own, last axis; loops nested in them run inside one lane.  A base written by one of
// them is accessed by the others only through the identical view (so each element stays with the
// lane that wrote it), no reduction output is read inside its own loop or held in memory by an
// accumulate, gather or scatter, and P's own instructions are element-wise.  Empty: another form.
std::vector<const LoopB *> row_lane_loops(const LoopB &l0, bool *cross = nullptr) {
    if (cross != nullptr) *cross = false;
    const uint64_t p = std::max<uint64_t>(1, jitk::parallel_ranks(l0).first);
    const std::vector<const LoopB *> chain = jitk::get_first_loop_blocks(l0);
    if (chain.size() < p) return {};
    const LoopB &P = *chain[p - 1];
    std::vector<const LoopB *> loops;
    int64_t longest = 0;
    for (const Block &b : P._block_list) {
        if (b.isInstr()) {
            const InstrPtr &i = b.getInstr();
            if (bh_opcode_is_system(i->opcode)) continue;
            if (bh_opcode_is_sweep(i->opcode) || i->opcode == BH_GATHER || i->opcode == BH_SCATTER ||
                i->opcode == BH_COND_SCATTER)
                return {};
            continue;
        }
        const LoopB &C = b.getLoop();
        for (const InstrPtr &sw : C._sweeps)
            if (!bh_opcode_is_reduction(sw->opcode) || sw->sweep_axis() != C.rank ||
                sw->sweep_axis() != sw->operand[1].ndim - 1)
                return {};
        // (loops nested in C run in the lane that owns C's index, sweeps over their axes included)
        for (const InstrPtr &i : jitk::allInstr(C))
            if (i->opcode == BH_SCATTER || i->opcode == BH_COND_SCATTER) return {};
        loops.push_back(&C);
        longest = std::max(longest, C.size);
    }
    if (loops.empty() || longest < 32) return {};
    // Reduction outputs stay in registers: not read inside their loop, not an array of another kind.
    std::set<const bh_base *> red_outs;
    for (const LoopB *C : loops) {
        std::set<const bh_base *> outs;
        for (const InstrPtr &sw : C->_sweeps) outs.insert(sw->operand[0].base);
        for (const InstrPtr &i : jitk::allInstr(*C))
            for (size_t o = 1; o < i->operand.size(); ++o)
                if (!i->operand[o].isConstant() && outs.count(i->operand[o].base)) return {};
        red_outs.insert(outs.begin(), outs.end());
    }
    for (const InstrPtr &i : jitk::allInstr(l0))
        if (i->opcode == BH_GATHER && red_outs.count(i->operand[1].base)) return {};
    // ... and are read only through the view they are reduced into (the register), since the array
    // is written once, after the row.
    std::map<const bh_base *, const bh_view *> red_view;
    for (const LoopB *C : loops)
        for (const InstrPtr &sw : C->_sweeps) red_view[sw->operand[0].base] = &sw->operand[0];
    for (const InstrPtr &i : jitk::allInstr(l0))
        for (size_t o = 0; o < i->operand.size(); ++o) {
            const bh_view &v = i->operand[o];
            if (v.isConstant()) continue;
            auto r = red_view.find(v.base);
            if (r != red_view.end() && !(v == *r->second)) return {};
        }
    // Element ownership: when what one loop (or the row's own instructions) writes is touched by
    // another loop through another view, an element moves between lanes, and the lanes' memory
    // accesses are ordered by a fence after each lane loop (`cross`).
    // Outputs written in a part, except the wave-folded reductions of a lane loop itself (their
    // registers are stored after the row, and read only through their own view).
    std::set<const bh_instruction *> folded;
    for (const LoopB *C : loops)
        for (const InstrPtr &sw : C->_sweeps) folded.insert(sw.get());
    bool several = false;
    auto writes = [&](const std::vector<InstrPtr> &instrs, std::map<const bh_base *, const bh_view *> &w) {
        for (const InstrPtr &i : instrs) {
            if (i->operand.empty() || i->operand[0].isConstant() || folded.count(i.get())) continue;
            auto it = w.find(i->operand[0].base);
            if (it != w.end() && !(*it->second == i->operand[0])) several = true;
            w[i->operand[0].base] = &i->operand[0];
        }
    };
    std::vector<std::vector<InstrPtr> > parts;
    for (const LoopB *C : loops) parts.push_back(jitk::allInstr(*C));
    parts.push_back(jitk::allLocalInstr(P));
    // Inside one lane loop (its nested loops included) nothing orders the lanes: a base written
    // there is touched there only through the written view.
    for (size_t a = 0; a + 1 < parts.size(); ++a) {
        std::map<const bh_base *, const bh_view *> written;
        writes(parts[a], written);
        if (several) return {};  // one base written through two views
        for (const InstrPtr &i : parts[a])
            for (const bh_view &v : i->operand) {
                if (v.isConstant()) continue;
                auto w = written.find(v.base);
                if (w != written.end() && !(v == *w->second)) return {};
            }
    }
    for (size_t a = 0; a < parts.size(); ++a) {
        std::map<const bh_base *, const bh_view *> written;
        writes(parts[a], written);
        for (size_t b = 0; b < parts.size(); ++b) {
            if (a == b) continue;
            for (const InstrPtr &i : parts[b])
                for (const bh_view &v : i->operand) {
                    if (v.isConstant()) continue;
                    auto w = written.find(v.base);
                    if (w != written.end() && !(v == *w->second) && cross != nullptr) *cross = true;
                }
        }
    }
    return loops;
}

void Writer::emit_row_reduce() {
    const LoopB &l0 = unit._block_list.back().getLoop();
    const uint64_t p = std::max<uint64_t>(1, jitk::parallel_ranks(l0).first);
    const std::vector<const LoopB *> chain = jitk::get_first_loop_blocks(l0);
    bool cross = false;
    const std::vector<const LoopB *> loops = row_lane_loops(l0, &cross);
    if (loops.empty()) throw std::logic_error("row skeleton: block has another form");
    fence_lanes = cross;
    lane_loops.clear();
    lane_loops.insert(loops.begin(), loops.end());
    uint64_t rows = 1;
    for (uint64_t r = 0; r < p; ++r) rows *= static_cast<uint64_t>(chain[r]->size);
    int64_t longest = 0;
    for (const LoopB *C : loops) longest = std::max(longest, C->size);
    kp.work_items = rows * static_cast<uint64_t>(longest);
    Scope ksc;
    declare_scope(unit, ksc, 1);
    body << "  const int64_t rows_ = 1";
    for (uint64_t r = 0; r < p; ++r) body << " * n" << lid.at(chain[r]);
    body << ";\n";
    body << "  const int lane_ = threadIdx.x & 63;\n";
    body << "  for (int64_t f_ = (int64_t)bh_bid * BH_WAVES + (threadIdx.x >> 6); f_ < rows_; f_ += (int64_t)bh_nblk * BH_WAVES) {\n";
    body << "    int64_t r_ = f_;\n";
    for (int64_t r = static_cast<int64_t>(p) - 1; r >= 1; --r)
        body << "    const int64_t i" << r << " = r_ % n" << lid.at(chain[r]) << "; r_ /= n" << lid.at(chain[r]) << ";\n";
    body << "    const int64_t i0 = r_;\n";
    std::vector<Scope> scopes(p);
    const Scope *parent = &ksc;
    for (uint64_t r = 0; r < p; ++r) {
        scopes[r].parent = parent;
        body << std::string(4 + 2 * r, ' ') << "{\n";
        declare_scope(*chain[r], scopes[r], 3 + static_cast<int>(r));
        parent = &scopes[r];
    }
    Scope &ps = scopes[p - 1];
    const int ind = 2 + static_cast<int>(p);
    lane_axis = chain[p - 1]->rank + 1;
    // The row's own instructions run in every lane (same values); each lane loop is strided by the
    // lanes and its reductions are folded across the wave right after it (emit_block).
    emit_blocks(*chain[p - 1], ps, ind);
    indent(body, ind);
    body << "if (lane_ == 0) {\n";
    write_back(*chain[p - 1], ps, ind + 1);
    indent(body, ind);
    body << "}\n";
    for (int64_t r = static_cast<int64_t>(p) - 1; r >= 0; --r) {
        if (r < static_cast<int64_t>(p) - 1) write_back(*chain[r], scopes[r], 3 + static_cast<int>(r));
        body << std::string(4 + 2 * r, ' ') << "}\n";
    }
    body << "  }\n";
    write_back(unit, ksc, 1);
    kp.grid = std::max<uint64_t>(1, std::min<uint64_t>((rows + 3) / 4, cfg.max_grid));
}


/* A segmented reduction: the innermost leading parallel loop P holds constant seeds of the reductions of
 * one innermost loop C, C, and element-wise instructions after it.  C's sweeps reduce its own, last
 * axis; C reads no reduction output, gathers and scatters nothing, and touches a base that it writes
 * only through the written view (elements of one output may be computed by several threads). */
struct SegForm {
    const LoopB *C = nullptr;
    std::vector<const bh_instruction *> seeds;
    std::vector<InstrPtr> post;
    std::set<const bh_base *> loop_temps;  // temporaries of P that only C uses
    bool columns = false;  // the contiguous axis is P's (reduce over rows), else C's
    /* The launch: V neighbours of the contiguous axis per thread and load (16 bytes of the widest view along it),
     * U loads in flight; columns: w threads along the outputs, else `lanes` threads per output; row_blocks
     * workgroups cover the outputs, times `splits` pieces of `chunk` elements of the reduced axis. */
    int V = 1, U = 4;
    uint64_t outs_n = 1, lanes = 1, row_blocks = 1, splits = 1, chunk = 1, w = 1;
    uint64_t reads = 0;  // views that C reads an element of per iteration (broadcasts along either axis left out)
};

// Where one reduction is segmented, from device times of sums of x * x in float32 and float64 (one launch and its gap
// are 6 us of them; a second one, the finalize, adds 2.3 us and 3 us on the host).
// Rows, lanes along the row: from 2^16 elements on the skeletons are level (256^2: 6.1 us) or this one is ahead (8 x
// 8192: row 16.6, seg 6.1 us; 131072 x 16: map 8.0, seg 6.3).
// Columns are split and finalized, so the row skeleton's single launch wins while its waves' walks down the columns
// are short and their lines stay in the L2s: row / seg 2048 x 256 8.6 / 9.4 us, 512 x 2048 6.7 / 9.4, 1024 x 1500 11.1 / 8.8
// (host and device together 11.5 / 14.6); 4096 x 16 11.7 / 8.2, 2048 x 700 16.1 / 9.0, 40 x 60000 15.8 / 9.7.  Its time goes
// with the loads: sums over three arrays 512^2 7.3 / 8.9, 900^2 15.6 / 10.3, 750 x 1500 21.9 / 10.4.
// Fewer than 32 rows: a thread per column reads them coalesced in one launch.  map / seg 16 x 2^20 float32 14.7 / 40.3, 31 x 2^18
// 8.3 / 17.4; 16-byte loads without a split are ahead: 16 x 2^22 64 / 51, 31 x 2^21 56 / 47.
// With a map over the outputs in its finalize (a mean) this skeleton has no launch more: x - x.mean(0) of 256^2 18.5 / 15.3
// us, of 1024^2 22.1 / 15.5.
constexpr uint64_t kSegMinItems = 1u << 16;
constexpr uint64_t kSegMinColumns = 1u << 21;
constexpr uint64_t kSegLongColumn = 4096;

// Several of one code in one flush (`crowd`) run as one batched launch of the row skeleton, which fills the chip with
// columns and rows that a single one leaves idle, against one or two launches each here.  60 uneven matrices, batched rows /
// segmented, device us: by columns 300 x 320 37 / 527, 1000^2 305 / 589, 1400^2 607 / 612, 2000^2 1248 / 756, 32768 x 32 542 / 700,
// 200000 x 8 1860 / 1027; by rows 300 x 320 12 / 375, 2000^2 289 / 514, 4000^2 1058 / 951, 20 x 50000 384 / 593,
// 8 x 200000 1425 / 963.
constexpr uint64_t kCrowdColumns = kSegMinColumns, kCrowdLongColumn = 1u << 15;
constexpr uint64_t kCrowdRows = 1u << 23, kCrowdLongRow = 1u << 16;

bool seg_pays(const SegForm &f, bool tail, bool crowd) {
    const uint64_t R = static_cast<uint64_t>(f.C->size), total = f.outs_n * R, loads = total * std::max<uint64_t>(1, f.reads);
    if (total < kSegMinItems) return false;
    if (crowd && (f.columns ? R <= kCrowdLongColumn && loads < kCrowdColumns : R <= kCrowdLongRow && loads < kCrowdRows)) return false;
    if (!f.columns) return true;
    if (R < 32) return f.V == 4 && f.splits == 1;
    return tail || loads >= kSegMinColumns || R >= kSegLongColumn || (2 * R >= kSegLongColumn && 2 * loads >= kSegMinColumns);
}

// The reduced axis is cut until the launch has about this many workgroups.
constexpr uint64_t kSegBlocks = 2048;

void seg_launch(SegForm &f, int width, int64_t inner, uint64_t W) {
    const uint64_t R = static_cast<uint64_t>(f.C->size);
    f.V = width;
    f.U = f.columns ? (f.V >= 4 ? 4 : 8) : 4;
    f.chunk = R;
    const uint64_t U = static_cast<uint64_t>(f.U);
    if (f.columns) {
        while (inner % f.V != 0) f.V /= 2;  // a thread's outputs are V neighbours of one innermost row
        const uint64_t groups = f.outs_n / static_cast<uint64_t>(f.V);
        f.row_blocks = (groups + W - 1) / W;
        f.w = (groups + f.row_blocks - 1) / f.row_blocks;
        const uint64_t step = W / f.w * U;
        f.splits = std::max<uint64_t>(1, std::min((kSegBlocks + f.row_blocks - 1) / f.row_blocks, R / (2 * step)));
        f.chunk = (R + f.splits - 1) / f.splits;
    } else {
        // A workgroup per row for long rows (and for moderate ones when there are few), else a wave, and
        // fewer lanes for short rows: each lane loads at least twice.
        const uint64_t V = static_cast<uint64_t>(f.V), wide = W * 2 * V;
        f.lanes = R >= wide * U || (f.outs_n < kSegBlocks && R >= wide) ? W : 64;
        while (f.lanes > 4 && f.lanes <= 64 && f.lanes * 2 * V > R) f.lanes /= 2;
        const uint64_t per_block = W / f.lanes;
        f.row_blocks = (f.outs_n + per_block - 1) / per_block;
        if (f.lanes == W)
            f.splits = std::max<uint64_t>(1, std::min((kSegBlocks + f.row_blocks - 1) / f.row_blocks, R / (2 * f.lanes * V * U)));
        f.chunk = (R + f.splits - 1) / f.splits;
        f.chunk = (f.chunk + f.lanes * V - 1) / (f.lanes * V) * (f.lanes * V);
    }
    f.splits = (R + f.chunk - 1) / f.chunk;
}

// (`tail`: the block is to take in a map over its outputs; `crowd`: see seg_pays)
SegForm seg_form(const LoopB &l0, const std::set<const bh_base *> &params, bool crowd, bool tail = false) {
    SegForm none, f;
    const uint64_t p = std::max<uint64_t>(1, jitk::parallel_ranks(l0).first);
    const std::vector<const LoopB *> chain = jitk::get_first_loop_blocks(l0);
    if (chain.size() < p) return none;
    const LoopB &P = *chain[p - 1];
    std::vector<InstrPtr> before;
    for (const Block &b : P._block_list) {
        if (!b.isInstr()) {
            if (f.C != nullptr) return none;
            f.C = &b.getLoop();
            continue;
        }
        const InstrPtr &i = b.getInstr();
        if (bh_opcode_is_system(i->opcode)) continue;
        if (bh_opcode_is_sweep(i->opcode) || i->opcode == BH_GATHER || i->opcode == BH_SCATTER ||
            i->opcode == BH_COND_SCATTER || i->opcode == BH_RANDOM || i->opcode == BH_RANGE)
            return none;
        (f.C == nullptr ? before : f.post).push_back(i);
    }
    if (f.C == nullptr || !f.C->isInnermost() || f.C->_sweeps.empty() || f.C->size < 16) return none;
    uint64_t outs_n = 1;
    for (uint64_t r = 0; r < p; ++r) outs_n *= static_cast<uint64_t>(std::max<int64_t>(0, chain[r]->size));
    if (outs_n >= (1ull << 31)) return none;
    std::map<const bh_base *, const bh_view *> outs;
    for (const InstrPtr &sw : f.C->_sweeps) {
        if (!bh_opcode_is_reduction(sw->opcode) || sw->sweep_axis() != f.C->rank ||
            sw->sweep_axis() != sw->operand[1].ndim - 1 || outs.count(sw->operand[0].base))
            return none;
        outs[sw->operand[0].base] = &sw->operand[0];
    }
    for (const InstrPtr &i : before) {
        if (i->opcode != BH_IDENTITY || !i->operand[1].isConstant()) return none;
        auto o = outs.find(i->operand[0].base);
        if (o == outs.end() || !(i->operand[0] == *o->second)) return none;
        f.seeds.push_back(i.get());
    }
    // Every sweep output is seeded here (the partials start at the identity themselves).
    for (const auto &o : outs) {
        bool seeded = false;
        for (const bh_instruction *i : f.seeds) seeded |= i->operand[0].base == o.first;
        if (!seeded) return none;
    }
    std::map<const bh_base *, const bh_view *> written;
    const std::vector<InstrPtr> body = jitk::allInstr(*f.C);
    for (const InstrPtr &i : body) {
        if (bh_opcode_is_system(i->opcode)) continue;
        if (i->opcode == BH_GATHER || i->opcode == BH_SCATTER || i->opcode == BH_COND_SCATTER) return none;
        if (i->operand[0].isConstant()) return none;
        if (outs.count(i->operand[0].base)) {
            if (!f.C->_sweeps.count(i)) return none;
            continue;
        }
        auto w = written.find(i->operand[0].base);
        if (w != written.end() && !(*w->second == i->operand[0])) return none;
        written[i->operand[0].base] = &i->operand[0];
    }
    for (const InstrPtr &i : body)
        for (size_t o = 0; o < i->operand.size(); ++o) {
            const bh_view &v = i->operand[o];
            if (v.isConstant()) continue;
            if (v.hasSlide()) return none;
            auto w = written.find(v.base);
            if (w != written.end() && !(v == *w->second)) return none;
            if (o > 0 && outs.count(v.base)) return none;
        }
    for (const InstrPtr &i : f.post)
        for (size_t o = 0; o < i->operand.size(); ++o) {
            const bh_view &v = i->operand[o];
            if (v.isConstant()) continue;
            if (v.hasSlide()) return none;
            // (an element that C wrote may still be on its way from another lane)
            if (written.count(v.base)) return none;
            auto r = outs.find(v.base);
            if (r != outs.end() && (o == 0 || !(v == *r->second))) return none;
        }
    // Temporaries of the parallel loops other than the sweep outputs: the reduction loop's own when
    // nothing outside it touches them (a lifted free), else the block has another form.
    const std::set<bh_base *> c_temps = f.C->getLocalTemps();
    for (uint64_t r = 0; r < p; ++r)
        for (bh_base *b : chain[r]->getLocalTemps()) {
            if (outs.count(b) || c_temps.count(b)) continue;
            bool in_body = false, in_post = false;
            for (const InstrPtr &i : body)
                for (const bh_view &v : i->operand) in_body |= !v.isConstant() && v.base == b;
            for (const InstrPtr &i : f.post)
                for (const bh_view &v : i->operand) in_post |= !v.isConstant() && v.base == b;
            if (in_body && in_post) return none;
            if (in_body) f.loop_temps.insert(b);
        }
    // The contiguous axis of the arrays that C reads, weighted by their element size.
    int64_t cols = 0, rows = 0;
    int widest = 1;
    std::set<VKey> seen;
    const int64_t a = static_cast<int64_t>(p) - 1, c = f.C->rank;
    for (const InstrPtr &i : body)
        for (size_t o = 1; o < i->operand.size(); ++o) {
            const bh_view &v = i->operand[o];
            if (v.isConstant() || !params.count(v.base) || v.ndim <= c || !seen.insert(vkey(v)).second) continue;
            if (v.stride[c] == 0 || v.stride[a] == 0) continue;  // (broadcast: a fraction of the elements)
            ++f.reads;
            const int sz = bh_type_size(v.base->dtype());
            if (v.stride[c] == 1 && v.shape[c] > 1 && v.stride[a] != 1) {
                rows += sz;
                widest = std::max(widest, sz);
            } else if (v.stride[a] == 1 && v.shape[a] > 1 && v.stride[c] != 1) {
                cols += sz;
                widest = std::max(widest, sz);
            }
        }
    if (rows == cols) return none;
    f.columns = cols > rows;
    f.outs_n = outs_n;
    const uint64_t W = KernelPlan().block;
    seg_launch(f, std::max(1, std::min(4, 16 / widest)), P.size, W);
    // (a launch holds fewer than 2^32 threads, and this skeleton has a thread group for every output)
    if (f.row_blocks * f.splits * W >= 1ull << 32 || !seg_pays(f, tail || !f.post.empty(), crowd)) return none;
    return f;
}

// ---- SEG_REDUCE
// Bound by HBM when the whole chip loads.  What the row skeleton left idle: a column sum ran one wave
// per column with its lanes a row apart (one 64-byte request per lane and element), and few outputs
// gave few waves.  Here lanes always run along the contiguous axis with 16-byte loads, and the reduced
// axis is cut into `splits` pieces until the launch has about kSegBlocks workgroups.  Measured on float32
// sums: 100000 x 500 by columns 536 -> 40 us (5.0 TB/s), 65536 x 16 137 -> 8.6; by rows (4-byte loads before) 512 x 4096
// 10.6 -> 6.0 us, 64 x 16384 29 -> 8.3.
void Writer::emit_seg_reduce() {
    const LoopB &l0 = unit._block_list.back().getLoop();
    const uint64_t p = std::max<uint64_t>(1, jitk::parallel_ranks(l0).first);
    const std::vector<const LoopB *> chain = jitk::get_first_loop_blocks(l0);
    const SegForm f = seg_form(l0, std::set<const bh_base *>(kp.params.begin(), kp.params.end()), cfg.crowd);
    if (f.C == nullptr) throw std::logic_error("seg skeleton: block has another form");
    for (const bh_instruction *i : f.seeds) skip.insert(i);
    const LoopB &C = *f.C;
    const uint64_t outs_n = f.outs_n, W = kp.block;
    kp.work_items = outs_n * static_cast<uint64_t>(C.size);
    const std::string rk = std::to_string(C.rank), pk = std::to_string(p - 1);
    const std::string nR = "n" + std::to_string(lid.at(&C));
    const int V = f.V, U = f.U;
    const uint64_t lanes = f.lanes, row_blocks = f.row_blocks, splits = f.splits;
    const bool split = splits > 1;
    kp.grid = row_blocks * splits;
    lane_axis = f.columns ? static_cast<int64_t>(p) - 1 : C.rank;
    lane_run = V;
    shape_args = {{"sg_nb", static_cast<int64_t>(row_blocks)}, {"sg_ch", static_cast<int64_t>(f.chunk)}};
    if (f.columns) shape_args.emplace_back("sg_w", static_cast<int64_t>(f.w));

    struct Acc {
        InstrPtr instr;
        bh_type t;
        std::string T, var, ident;
    };
    std::vector<Acc> accs;
    std::vector<InstrPtr> sweeps(C._sweeps.begin(), C._sweeps.end());
    std::sort(sweeps.begin(), sweeps.end(), [](const InstrPtr &x, const InstrPtr &y) { return x->origin_id < y->origin_id; });
    for (const InstrPtr &s : sweeps) {
        Acc a;
        a.instr = s;
        a.t = s->operand[0].base->dtype();
        a.T = hip_type(a.t);
        a.var = "q" + std::to_string(accs.size());
        a.ident = literal(jitk::sweep_identity(s->opcode, a.t));
        accs.push_back(a);
    }
    auto op_lambda = [&](const Acc &a) {
        return "auto op_ = [](" + a.T + " x, " + a.T + " y) -> " + a.T + " { return " +
               combine_expr(a.instr->opcode, "x", "y") + "; };";
    };
    // Partials: per accumulator a slab of splits x outputs.
    uint64_t scratch = 0;
    if (split) {
        for (size_t k = 0; k < accs.size(); ++k) {
            shape_args.emplace_back("sg_o" + std::to_string(k), static_cast<int64_t>(scratch));
            scratch += (splits * outs_n * static_cast<uint64_t>(bh_type_size(accs[k].t)) + 255) / 256 * 256;
        }
        kp.scratch_bytes = static_cast<int64_t>(scratch);
    }
    std::string outs_expr = "1";
    for (uint64_t r = 0; r < p; ++r) outs_expr += " * n" + std::to_string(lid.at(chain[r]));
    Scope ksc;
    // i0 .. i{p-1} of the flat output number `e` (32-bit: there are fewer than 2^31 outputs)
    auto decode = [&](int ind, const std::string &e) {
        const std::string pad(2 * ind, ' ');
        body << pad << "uint32_t d_ = (uint32_t)(" << e << ");\n";
        for (int64_t r = static_cast<int64_t>(p) - 1; r >= 1; --r)
            body << pad << "const int64_t i" << r << " = (int64_t)(d_ % (uint32_t)n" << lid.at(chain[r])
                 << "); d_ /= (uint32_t)n" << lid.at(chain[r]) << ";\n";
        body << pad << "const int64_t i0 = (int64_t)d_;\n";
    };
    // The rest of one output: its reductions are in accumulator registers `var(k)`.
    auto finish = [&](int ind, const std::function<std::string(size_t)> &var) {
        std::vector<Scope> scopes(p);
        const Scope *parent = &ksc;
        for (uint64_t r = 0; r < p; ++r) {
            scopes[r].parent = parent;
            indent(body, ind + static_cast<int>(r));
            body << "{\n";
            declare_scope(*chain[r], scopes[r], ind + 1 + static_cast<int>(r));
            parent = &scopes[r];
        }
        const int in = ind + static_cast<int>(p);
        Scope &ps = scopes[p - 1];
        for (size_t k = 0; k < accs.size(); ++k) {
            const bh_instruction &s = *accs[k].instr;
            indent(body, in);
            body << ref(ps, s.operand[0], static_cast<int>(s.sweep_axis())) << " = " << var(k) << ";\n";
        }
        for (const InstrPtr &i : f.post) emit_instr(*i, ps, in);
        for (int64_t r = static_cast<int64_t>(p) - 1; r >= 0; --r) {
            write_back(*chain[r], scopes[r], ind + 1 + static_cast<int>(r));
            indent(body, ind + static_cast<int>(r));
            body << "}\n";
        }
    };
    // One element of C in a scope whose accumulators are var(k); `pre` names preloaded inputs.
    auto element = [&](int ind, const Scope *pre, const std::function<std::string(size_t)> &var) {
        Scope al;
        al.parent = pre;
        for (size_t k = 0; k < accs.size(); ++k) al.alias[accs[k].instr->operand[0].base] = var(k);
        Scope sc;
        sc.parent = &al;
        for (const bh_base *b : f.loop_temps) {
            sc.tmps.insert(b);
            indent(body, ind);
            body << hip_type(b->dtype()) << " t" << bid.at(b) << ";\n";
        }
        declare_scope(C, sc, ind);
        emit_blocks(C, sc, ind);
        write_back(C, sc, ind);
    };
    const std::vector<const bh_view *> reads = preloadable(C);
    // `U` x `V` elements: load every read-only input, then compute.  head(u, v) declares the indices.
    auto group = [&](int ind, int nu, int nv, const std::function<void(int, int, int)> &head,
                     const std::function<std::string(size_t, int)> &var) {
        const std::string pad(2 * ind, ' ');
        auto ld = [&](size_t k, int u, int v) {
            return "ld" + std::to_string(k) + "_" + std::to_string(u) + "_" + std::to_string(v);
        };
        for (int u = 0; u < nu; ++u)
            for (int v = 0; v < nv; ++v)
                for (size_t k = 0; k < reads.size(); ++k)
                    body << pad << hip_type(reads[k]->base->dtype()) << " " << ld(k, u, v) << ";\n";
        for (int u = 0; u < nu; ++u)
            for (int v = 0; v < nv; ++v) {
                if (reads.empty()) break;
                body << pad << "{\n";
                head(ind + 1, u, v);
                for (size_t k = 0; k < reads.size(); ++k)
                    body << pad << "  " << ld(k, u, v) << " = " << ref(ksc, *reads[k]) << ";\n";
                body << pad << "}\n";
            }
        for (int u = 0; u < nu; ++u)
            for (int v = 0; v < nv; ++v) {
                Scope pre;
                pre.parent = &ksc;
                for (size_t k = 0; k < reads.size(); ++k) pre.preload[vkey(*reads[k])] = ld(k, u, v);
                body << pad << "{\n";
                head(ind + 1, u, v);
                element(ind + 1, &pre, [&](size_t k) { return var(k, v); });
                body << pad << "}\n";
            }
    };
    auto store_partial = [&](size_t k, const std::string &out, const std::string &value) {
        return "((" + accs[k].T + " *)(bh_scratch + sg_o" + std::to_string(k) + "))[sp_ * outs_ + " + out + "] = " + value + ";\n";
    };

    body << "  const int64_t outs_ = " << outs_expr << ";\n";
    body << "  const int64_t sp_ = bh_bid / (unsigned)sg_nb, cb_ = bh_bid % (unsigned)sg_nb;\n";
    body << "  const int64_t r0_ = sp_ * sg_ch, r1_ = r0_ + sg_ch < " << nR << " ? r0_ + sg_ch : " << nR << ";\n";
    const std::string sV = std::to_string(V);
    if (f.columns) {
        // Thread (tx_, ty_): outputs [e_, e_ + V), rows r0_ + ty_, + ty step, ...
        body << "  const unsigned w_ = (unsigned)sg_w, tys_ = BH_WG / w_;\n";
        body << "  const unsigned ty_ = threadIdx.x / w_, tx_ = threadIdx.x - ty_ * w_;\n";
        body << "  const int64_t e_ = (cb_ * w_ + tx_) * " << V << ";\n";
        body << "  const bool on_ = ty_ < tys_ && e_ < outs_;\n";
        for (size_t k = 0; k < accs.size(); ++k)
            for (int v = 0; v < V; ++v)
                body << "  " << accs[k].T << " " << accs[k].var << "_" << v << " = " << accs[k].ident << ";\n";
        auto var = [&](size_t k, int v) { return accs[k].var + "_" + std::to_string(v); };
        body << "  if (on_) {\n";
        // (the first output's indices; the innermost one advances by v)
        {
            const std::string inner = "i" + pk;
            body << "    uint32_t d_ = (uint32_t)e_;\n";
            for (int64_t r = static_cast<int64_t>(p) - 1; r >= 1; --r)
                body << "    const int64_t b" << r << "_ = (int64_t)(d_ % (uint32_t)n" << lid.at(chain[r])
                     << "); d_ /= (uint32_t)n" << lid.at(chain[r]) << ";\n";
            body << "    const int64_t b0_ = (int64_t)d_;\n";
            for (int64_t r = 0; r + 1 < static_cast<int64_t>(p); ++r)
                body << "    const int64_t i" << r << " = b" << r << "_;\n";
            auto head = [&](int ind, int u, int v) {
                indent(body, ind);
                body << "const int64_t " << inner << " = b" << pk << "_ + " << v << ", i" << rk << " = r_ + " << u
                     << " * (int64_t)tys_;\n";
            };
            body << "    int64_t r_ = r0_ + ty_;\n";
            body << "    for (; r_ + " << U - 1 << " * (int64_t)tys_ < r1_; r_ += " << U << " * (int64_t)tys_) {\n";
            group(3, U, V, head, var);
            body << "    }\n";
            body << "    for (; r_ < r1_; r_ += tys_) {\n";
            group(3, 1, V, head, var);
            body << "    }\n";
        }
        body << "  }\n";
        // Fold the rows of the workgroup through LDS, in row order.
        int largest = 1;
        for (const Acc &a : accs) largest = std::max(largest, bh_type_size(a.t));
        body << "  __shared__ __attribute__((aligned(16))) unsigned char bh_lds_[BH_WG * " << V * largest << "];\n";
        for (size_t k = 0; k < accs.size(); ++k) {
            const Acc &a = accs[k];
            body << "  { " << op_lambda(a) << "\n";
            body << "    " << a.T << " *l_ = (" << a.T << " *)bh_lds_;\n";
            if (k > 0) body << "    __syncthreads();\n";
            body << "    if (on_) {\n";
            for (int v = 0; v < V; ++v) body << "      l_[threadIdx.x * " << V << " + " << v << "] = " << var(k, v) << ";\n";
            body << "    }\n    __syncthreads();\n";
            body << "    if (on_ && ty_ == 0) {\n      for (unsigned t_ = 1; t_ < tys_; ++t_) {\n";
            for (int v = 0; v < V; ++v)
                body << "        " << var(k, v) << " = op_(" << var(k, v) << ", l_[(t_ * w_ + tx_) * " << V << " + " << v << "]);\n";
            body << "      }\n    }\n  }\n";
        }
        body << "  if (!on_ || ty_ != 0) return;\n";
        for (int v = 0; v < V; ++v) {
            if (split) {
                for (size_t k = 0; k < accs.size(); ++k)
                    body << "  " << store_partial(k, "e_ + " + std::to_string(v), var(k, v));
            } else {
                body << "  {\n";
                decode(2, "e_ + " + std::to_string(v));
                finish(2, [&](size_t k) { return var(k, v); });
                body << "  }\n";
            }
        }
    } else {
        // `lanes` threads per output, V neighbouring elements each.
        const std::string G = std::to_string(lanes);
        body << "  const unsigned l_ = threadIdx.x % " << G << "u;\n";
        body << "  const int64_t e_ = cb_ * " << W / lanes << " + threadIdx.x / " << G << "u;\n";
        body << "  const bool on_ = e_ < outs_;\n";
        for (const Acc &a : accs) body << "  " << a.T << " " << a.var << " = " << a.ident << ";\n";
        auto var = [&](size_t k, int) { return accs[k].var; };
        body << "  if (on_) {\n";
        decode(2, "e_");
        auto head = [&](int ind, int u, int v) {
            indent(body, ind);
            body << "const int64_t i" << rk << " = r_ + " << u * static_cast<int64_t>(lanes) * V + v << ";\n";
        };
        body << "    int64_t r_ = r0_ + (int64_t)l_ * " << V << ";\n";
        body << "    for (; r_ + " << (U - 1) * static_cast<int64_t>(lanes) * V + V << " <= r1_; r_ += " << U * static_cast<int64_t>(lanes) * V << ") {\n";
        group(3, U, V, head, var);
        body << "    }\n";
        body << "    for (; r_ + " << V << " <= r1_; r_ += " << static_cast<int64_t>(lanes) * V << ") {\n";
        group(3, 1, V, head, var);
        body << "    }\n";
        if (V > 1) {
            // the last (r1_ - r0_) mod V elements, one lane each
            body << "    r_ = r1_ - (r1_ - r0_) % " << V << " + l_;\n    if (r_ < r1_) {\n";
            group(3, 1, 1, head, var);
            body << "    }\n";
        }
        body << "  }\n";
        if (lanes == 256)
            body << "  __shared__ __attribute__((aligned(16))) unsigned char bh_lds_[BH_WAVES * 16];\n";
        for (const Acc &a : accs) {
            body << "  { " << op_lambda(a) << "\n    " << a.var << " = ";
            if (lanes == 256) {
                body << "bh_block_reduce(" << a.var << ", op_, (" << a.T << " *)bh_lds_);\n    __syncthreads(); }\n";
            } else {
                body << "bh_group_reduce<" << G << ">(" << a.var << ", op_); }\n";
            }
        }
        body << "  if (!on_ || l_ != 0) return;\n";
        if (split) {
            for (size_t k = 0; k < accs.size(); ++k) body << "  " << store_partial(k, "e_", accs[k].var);
        } else {
            body << "  {\n";
            decode(2, "e_");
            finish(2, [&](size_t k) { return accs[k].var; });
            body << "  }\n";
        }
    }
    if (!split) return;
    main_body = body.str();
    body.str("");
    body.clear();

    // Finalize: 16 outputs x 16 slices of the partials per workgroup, folded in split order within a
    // slice and then across slices; the first slice's thread finishes the output.
    shape_args.emplace_back("sg_ns", static_cast<int64_t>(splits));
    kp.fin_name = "bh_kernel_fin";
    kp.fin_grid = (outs_n + 15) / 16;
    body << "  const int64_t outs_ = " << outs_expr << ";\n";
    body << "  const unsigned tx_ = threadIdx.x & 15u, ty_ = threadIdx.x >> 4;\n";
    body << "  const int64_t e_ = (int64_t)bh_bid * 16 + tx_;\n";
    body << "  const bool on_ = e_ < outs_;\n";
    int largest = 1;
    for (const Acc &a : accs) largest = std::max(largest, bh_type_size(a.t));
    body << "  __shared__ __attribute__((aligned(16))) unsigned char bh_lds_[16 * 17 * " << largest << "];\n";
    body << "  const int64_t ps_ = (sg_ns + 15) / 16, p0_ = ty_ * ps_, p1_ = p0_ + ps_ < sg_ns ? p0_ + ps_ : sg_ns;\n";
    for (size_t k = 0; k < accs.size(); ++k) {
        const Acc &a = accs[k];
        body << "  " << a.T << " " << a.var << " = " << a.ident << ";\n";
        body << "  { " << op_lambda(a) << "\n";
        body << "    const " << a.T << " *s_ = (const " << a.T << " *)(bh_scratch + sg_o" << k << ");\n";
        body << "    if (on_) {\n      int64_t j_ = p0_;\n";
        body << "      for (; j_ + 8 <= p1_; j_ += 8) {\n        " << a.T << " x_[8];\n#pragma unroll\n"
             << "        for (int u_ = 0; u_ < 8; ++u_) x_[u_] = s_[(j_ + u_) * outs_ + e_];\n#pragma unroll\n"
             << "        for (int u_ = 0; u_ < 8; ++u_) " << a.var << " = op_(" << a.var << ", x_[u_]);\n      }\n";
        body << "      for (; j_ < p1_; ++j_) " << a.var << " = op_(" << a.var << ", s_[j_ * outs_ + e_]);\n    }\n";
        body << "    " << a.T << " *l_ = (" << a.T << " *)bh_lds_;\n";
        if (k > 0) body << "    __syncthreads();\n";
        body << "    l_[ty_ * 17 + tx_] = " << a.var << ";\n    __syncthreads();\n";
        body << "    if (ty_ == 0)\n      for (int t_ = 1; t_ < 16; ++t_) " << a.var << " = op_(" << a.var << ", l_[t_ * 17 + tx_]);\n  }\n";
    }
    body << "  if (!on_ || ty_ != 0) return;\n  {\n";
    decode(2, "e_");
    finish(2, [&](size_t k) { return accs[k].var; });
    body << "  }\n";
}

void Writer::emit_map_tiled(const TiledForm &f, const std::vector<const LoopB *> &chain, uint64_t p, const Scope &ksc) {
    const int64_t a = static_cast<int64_t>(p) - 1;
    const int T = f.side, per = T * T / 256, rows = 256 / T;
    lane_axis = a;
    auto n = [&](int64_t r) { return "n" + std::to_string(lid.at(chain[r])); };
    uint64_t tiles = static_cast<uint64_t>((chain[a]->size + T - 1) / T) * static_cast<uint64_t>((chain[f.q]->size + T - 1) / T);
    for (int64_t r = 0; r < a; ++r)
        if (r != f.q) tiles *= static_cast<uint64_t>(chain[r]->size);
    for (size_t k = 0; k < f.views.size(); ++k) {
        kp.tile_bytes += static_cast<uint64_t>(T * (T + 1) * bh_type_size(f.views[k]->base->dtype()));
        body << "  __shared__ " << hip_type(f.views[k]->base->dtype()) << " tl" << k << "_[" << T * (T + 1) << "];\n";
    }
    const std::string sT = std::to_string(T), qi = "i" + std::to_string(f.q), ai = "i" + std::to_string(a);
    body << "  const int64_t ta_ = (" << n(a) << " + " << T - 1 << ") / " << T << ", tb_ = (" << n(f.q) << " + " << T - 1
         << ") / " << T << ";\n  int64_t tiles_ = ta_ * tb_;\n";
    for (int64_t r = 0; r < a; ++r)
        if (r != f.q) body << "  tiles_ *= " << n(r) << ";\n";
    body << "  const int l_ = threadIdx.x & " << T - 1 << ", w_ = threadIdx.x / " << T << ";\n";
    body << "  for (int64_t g_ = bh_bid; g_ < tiles_; g_ += bh_nblk) {\n";
    body << "    int64_t d_ = g_ / ta_;\n    const int64_t a0_ = (g_ - d_ * ta_) * " << T << ";\n";
    body << "    const int64_t o_ = d_ / tb_;\n    const int64_t b0_ = (d_ - o_ * tb_) * " << T << ";\n    d_ = o_;\n";
    for (int64_t r = a - 1; r >= 0; --r)
        if (r != f.q) body << "    const int64_t i" << r << " = d_ % " << n(r) << "; d_ /= " << n(r) << ";\n";
    std::vector<const bh_view *> others;
    {
        std::set<VKey> tiled;
        for (const bh_view *v : f.views) tiled.insert(vkey(*v));
        for (const bh_view *v : preloadable(*chain[a]))
            if (!tiled.count(vkey(*v))) others.push_back(v);
    }
    for (int full = 1; full >= 0; --full) {
        if (full)
            body << "    if (a0_ + " << T << " <= " << n(a) << " && b0_ + " << T << " <= " << n(f.q) << ") {\n";
        else
            body << "    } else {\n";
        // the tile of every transposed view, lanes along its contiguous axis
        body << "#pragma unroll\n      for (int k_ = 0; k_ < " << per << "; ++k_) {\n";
        body << "        const int64_t " << qi << " = b0_ + l_, " << ai << " = a0_ + w_ + k_ * " << rows << ";\n";
        if (!full) body << "        if (" << qi << " < " << n(f.q) << " && " << ai << " < " << n(a) << ") {\n";
        for (size_t k = 0; k < f.views.size(); ++k)
            body << "        tl" << k << "_[(w_ + k_ * " << rows << ") * " << T + 1 << " + l_] = " << ref(ksc, *f.views[k]) << ";\n";
        if (!full) body << "        }\n";
        body << "      }\n      __syncthreads();\n";
        const int U = full ? 4 : 1;
        body << "      for (int k_ = 0; k_ < " << per << "; k_ += " << U << ") {\n";
        auto ld = [&](size_t k, int u) { return "ld" + std::to_string(k) + "_" + std::to_string(u); };
        auto head = [&](int u) {
            body << "        const int kr_ = w_ + (k_ + " << u << ") * " << rows << ";\n";
            body << "        const int64_t " << qi << " = b0_ + kr_, " << ai << " = a0_ + l_;\n";
        };
        if (full) {
            for (int u = 0; u < U; ++u)
                for (size_t k = 0; k < others.size(); ++k)
                    body << "        " << hip_type(others[k]->base->dtype()) << " " << ld(k, u) << ";\n";
            for (int u = 0; u < U && !others.empty(); ++u) {
                body << "        {\n";
                head(u);
                for (size_t k = 0; k < others.size(); ++k) body << "        " << ld(k, u) << " = " << ref(ksc, *others[k]) << ";\n";
                body << "        }\n";
            }
        }
        for (int u = 0; u < U; ++u) {
            Scope pre;
            pre.parent = &ksc;
            for (size_t k = 0; k < f.views.size(); ++k)
                pre.preload[vkey(*f.views[k])] = "tl" + std::to_string(k) + "_[l_ * " + std::to_string(T + 1) + " + kr_]";
            if (full)
                for (size_t k = 0; k < others.size(); ++k) pre.preload[vkey(*others[k])] = ld(k, u);
            body << "        {\n";
            head(u);
            if (!full) body << "        if (" << qi << " < " << n(f.q) << " && " << ai << " < " << n(a) << ") {\n";
            std::vector<Scope> scopes(p);
            const Scope *parent = &pre;
            for (uint64_t r = 0; r < p; ++r) {
                scopes[r].parent = parent;
                declare_scope(*chain[r], scopes[r], 5);
                if (r == p - 1) emit_blocks(*chain[r], scopes[r], 5);
                parent = &scopes[r];
            }
            for (int64_t r = a; r >= 0; --r) write_back(*chain[r], scopes[r], 5);
            if (!full) body << "        }\n";
            body << "        }\n";
        }
        body << "      }\n";
    }
    body << "    }\n    __syncthreads();\n  }\n";
    kp.grid = std::max<uint64_t>(1, std::min<uint64_t>(tiles, 4 * static_cast<uint64_t>(cfg.max_grid)));
}

// ---- MAP: grid-stride over the flattened leading parallel ranks
void Writer::emit_map() {
    const LoopB &l0 = unit._block_list.back().getLoop();
    const uint64_t p = std::max<uint64_t>(1, jitk::parallel_ranks(l0).first);
    const std::vector<const LoopB *> chain = jitk::get_first_loop_blocks(l0);
    uint64_t total = 1;
    for (uint64_t r = 0; r < p; ++r) total *= static_cast<uint64_t>(chain[r]->size);
    kp.work_items = total;
    const bool idx32 = total < (1ull << 31);
    Scope ksc;
    declare_scope(unit, ksc, 1);
    body << "  const int64_t tot_ = 1";
    for (uint64_t r = 0; r < p; ++r) body << " * n" << lid.at(chain[r]);
    body << ";\n";
    // Only loops without inner sequential work are unrolled (their body is straight-line code).
    lane_axis = static_cast<int64_t>(p) - 1;
    const bool flat = p == 1 ? l0.isInnermost() : chain[p - 1]->isInnermost();
    if (flat && p > 1) {
        const TiledForm f = tiled_form(chain, p, preloadable(*chain[p - 1]));
        if (!f.views.empty()) {
            // (tot_ is not used: the tiles are counted instead)
            emit_map_tiled(f, chain, p, ksc);
            write_back(unit, ksc, 1);
            return;
        }
    }
    Element e;
    e.outer = &ksc;
    e.body_loop = flat ? chain[p - 1] : nullptr;
    if (p == 2) e.inner = "n" + std::to_string(lid.at(chain[1]));
    e.unit = p == 1;
    e.decode = [&](int ind) {
        const std::string pad(2 * ind, ' ');
        if (p == 1) {
            body << pad << "const int64_t i0 = f_;\n";
        } else if (idx32) {
            body << pad << "uint32_t r_ = (uint32_t)f_;\n";
            for (int64_t r = static_cast<int64_t>(p) - 1; r >= 1; --r)
                body << pad << "const int64_t i" << r << " = (int64_t)(r_ % (uint32_t)n" << lid.at(chain[r])
                     << "); r_ /= (uint32_t)n" << lid.at(chain[r]) << ";\n";
            body << pad << "const int64_t i0 = (int64_t)r_;\n";
        } else {
            body << pad << "int64_t r_ = f_;\n";
            for (int64_t r = static_cast<int64_t>(p) - 1; r >= 1; --r)
                body << pad << "const int64_t i" << r << " = r_ % n" << lid.at(chain[r]) << "; r_ /= n"
                     << lid.at(chain[r]) << ";\n";
            body << pad << "const int64_t i0 = r_;\n";
        }
    };
    e.compute = [&](int ind, const Scope *outer) {
        // Open the scopes of the parallel loops; the innermost one carries the body.
        std::vector<Scope> scopes(p);
        const Scope *parent = outer;
        for (uint64_t r = 0; r < p; ++r) {
            scopes[r].parent = parent;
            body << std::string(2 * ind + 2 * r, ' ') << "{\n";
            declare_scope(*chain[r], scopes[r], ind + 1 + static_cast<int>(r));
            if (r == p - 1) emit_blocks(*chain[r], scopes[r], ind + 1 + static_cast<int>(r));
            parent = &scopes[r];
        }
        for (int64_t r = static_cast<int64_t>(p) - 1; r >= 0; --r) {
            write_back(*chain[r], scopes[r], ind + 1 + static_cast<int>(r));
            body << std::string(2 * ind + 2 * r, ' ') << "}\n";
        }
    };
    parts = cfg.xcd_parts && shifted_reads(l0);
    int64_t tasks = 0;
    if (p == 2 && parts &&
        stencil_walk(e, "n" + std::to_string(lid.at(chain[0])), "n" + std::to_string(lid.at(chain[1])), chain[0]->size,
                     chain[1]->size, cfg.map_unroll, &tasks)) {
        parts = false;
        write_back(unit, ksc, 1);
        kp.grid = std::max<uint64_t>(1, std::min<uint64_t>((static_cast<uint64_t>(tasks) + kp.block - 1) / kp.block, cfg.max_grid));
        return;
    }
    grid_stride("tot_", flat ? cfg.map_unroll : 1, e);
    parts = false;
    write_back(unit, ksc, 1);
    kp.grid = std::max<uint64_t>(1, std::min<uint64_t>((total + kp.block - 1) / kp.block, cfg.max_grid));
}

// A rank-0 reduction loop whose body is one innermost rank-1 loop that reduces rows into
// temporaries, which rank 0 reduces again with the same operator (max_i(max_j x[i][j])),
// is the full reduction of the 2-D iteration space.  Returns, per temporary, the rank-0
// reduction it feeds, and the instructions the flat skeleton implements itself; empty
// when the loop does not have that form.
std::map<const bh_base *, InstrPtr> collapsible_pairs(const LoopB &l0, const std::set<bh_base *> &temps,
                                                      std::set<const bh_instruction *> &skip) {
    std::map<const bh_base *, InstrPtr> none, pairs, inner;
    const LoopB *l1 = nullptr;
    for (const Block &b : l0._block_list) {
        if (b.isInstr()) continue;
        if (l1 != nullptr) return none;
        l1 = &b.getLoop();
    }
    if (l1 == nullptr || l1->rank != 1 || !l1->isInnermost()) return none;
    for (const InstrPtr &s : l1->_sweeps) {
        if (!bh_opcode_is_reduction(s->opcode) || s->sweep_axis() != 1 || !temps.count(s->operand[0].base)) return none;
        inner[s->operand[0].base] = s;
    }
    if (inner.empty()) return none;
    std::set<const bh_instruction *> sk;
    for (const Block &b : l0._block_list) {
        if (!b.isInstr()) continue;
        const InstrPtr &i = b.getInstr();
        if (bh_opcode_is_system(i->opcode)) continue;
        if (i->opcode == BH_IDENTITY && i->operand[1].isConstant() && inner.count(i->operand[0].base)) {
            sk.insert(i.get());
            continue;
        }
        if (bh_opcode_is_reduction(i->opcode) && i->sweep_axis() == 0 && inner.count(i->operand[1].base) &&
            inner.at(i->operand[1].base)->opcode == i->opcode && !pairs.count(i->operand[1].base)) {
            pairs[i->operand[1].base] = i;
            sk.insert(i.get());
            continue;
        }
        return none;
    }
    if (pairs.size() != inner.size()) return none;
    // The row temporaries may not be read anywhere else.
    for (const InstrPtr &i : jitk::allInstr(l0)) {
        if (sk.count(i.get()) || bh_opcode_is_system(i->opcode)) continue;
        for (size_t o = 1; o < i->operand.size(); ++o)
            if (!i->operand[o].isConstant() && inner.count(i->operand[o].base)) return none;
    }
    skip.insert(sk.begin(), sk.end());
    return pairs;
}

// ---- FULL_REDUCE: rank-0 reductions as two launches on one stream.  The main kernel
// leaves one partial per workgroup and reduction in scratch; the finalize kernel (one
// workgroup) folds the partials in workgroup order, stores the results and then runs
// the small scalar blocks that follow the sweeping loop in the unit (the tail) in
// thread 0.  The kernel boundary orders the two, so there is no fence, atomic ticket
// or counter to reset, the sum order is fixed, and the pair can be graph-captured.
void Writer::emit_full_reduce() {
    // The unit is [identity writers, the sweeping loop, tail blocks]; tail blocks may themselves be
    // small loops with sweeps (a 256-element sum or scan), so the sweeping loop is the first one.
    size_t pos = unit._block_list.size();
    for (size_t k = 0; k < unit._block_list.size() && pos == unit._block_list.size(); ++k)
        if (!unit._block_list[k].isInstr() && !unit._block_list[k].getLoop()._sweeps.empty()) pos = k;
    if (pos == unit._block_list.size()) throw std::logic_error("FULL_REDUCE unit without a sweeping loop");
    const LoopB &l0 = unit._block_list[pos].getLoop();
    std::vector<InstrPtr> sweeps;
    for (const InstrPtr &i : jitk::allLocalInstr(l0))
        if (bh_opcode_is_reduction(i->opcode) && i->sweep_axis() == 0) sweeps.push_back(i);
    std::sort(sweeps.begin(), sweeps.end(), [](const InstrPtr &a, const InstrPtr &b) { return a->origin_id < b->origin_id; });

    std::set<bh_base *> all_temps = temps;
    {
        const std::set<bh_base *> lt = unit.getLocalTemps();
        all_temps.insert(lt.begin(), lt.end());
    }
    const std::map<const bh_base *, InstrPtr> pairs = collapsible_pairs(l0, all_temps, skip);
    const LoopB *l1 = nullptr;
    uint64_t total = static_cast<uint64_t>(l0.size);
    if (!pairs.empty()) {
        for (const Block &b : l0._block_list)
            if (!b.isInstr()) l1 = &b.getLoop();
        total *= static_cast<uint64_t>(l1->size);
    }
    kp.work_items = total;
    // Each thread folds at least reduce_min_items elements before another workgroup (and its
    // partial) is added; at most reduce_max_grid workgroups.
    // A light loop body (a few operations per element, a stencil) streams better from half as many
    // workgroups, each folding twice the elements; a heavy one (Black-Scholes' ~70 operations) from
    // the full number (MI355X: Jacobi 8190^2 stencil+max 5 % faster at 2048 than 4096 workgroups,
    // Black-Scholes 2-4 % slower).
    const uint64_t per_wg = static_cast<uint64_t>(kp.block) * static_cast<uint64_t>(std::max(1, cfg.reduce_min_items));
    const bool light = jitk::allInstr(l0).size() <= kLightReduceInstrs;
    const uint64_t cap = std::max<uint64_t>(1, light ? cfg.reduce_max_grid / 2 : cfg.reduce_max_grid);
    const uint64_t grid = std::max<uint64_t>(1, std::min<uint64_t>((total + per_wg - 1) / per_wg, cap));
    kp.grid = grid;

    // Kernel scope: every rank-0 reduction output is a per-thread accumulator that starts at the identity.
    Scope ksc;
    struct Acc {
        InstrPtr instr;
        std::string var;
        bh_type t;
        bool is_tmp;
    };
    std::vector<Acc> accs;
    const std::set<bh_base *> ktmps = unit.getLocalTemps();
    for (const InstrPtr &s : sweeps) {
        const bh_view &v = s->operand[0];
        const bh_type t = v.base->dtype();
        Acc a;
        a.instr = s;
        a.t = t;
        a.is_tmp = ktmps.count(v.base) > 0 || temps.count(v.base) > 0;
        const std::string ident = literal(jitk::sweep_identity(s->opcode, t));
        if (a.is_tmp) {
            a.var = "t" + std::to_string(bid.at(v.base));
            if (!ksc.tmps.count(v.base)) {
                ksc.tmps.insert(v.base);
                body << "  " << hip_type(t) << " " << a.var << " = " << ident << ";\n";
            }
        } else {
            a.var = "s" + std::to_string(bid.at(v.base)) + "_" + std::to_string(view_id(v));
            if (!ksc.srep.count(vkey(v))) {
                ksc.srep.insert(vkey(v));
                body << "  " << hip_type(t) << " " << a.var << " = " << ident << ";\n";
            }
        }
        accs.push_back(a);
    }
    // Partials: one 16-byte slot per workgroup and distinct accumulator, workgroup-major, so the
    // layout (and the kernel source) does not depend on the grid size.
    std::map<std::string, int> slot;
    for (const Acc &a : accs)
        if (!slot.count(a.var)) slot.emplace(a.var, static_cast<int>(slot.size()));
    const int nslots = static_cast<int>(slot.size());
    kp.scratch_bytes = static_cast<int64_t>(grid) * nslots * 16;
    auto slot_addr = [&](const Acc &a, const std::string &wg) {
        return "(bh_scratch + ((size_t)" + wg + " * " + std::to_string(nslots) + " + " +
               std::to_string(slot.at(a.var)) + ") * 16)";
    };
    declare_scope(unit, ksc, 1);
    lane_axis = pairs.empty() ? 0 : 1;
    if (!pairs.empty()) {
        // One flat grid-stride loop over (i0, i1); each row temporary is the accumulator
        // of the rank-0 reduction it feeds.
        for (const auto &p : pairs)
            for (const Acc &a : accs)
                if (a.instr == p.second) ksc.alias[p.first] = a.var;
        const std::string n0 = "n" + std::to_string(lid.at(&l0)), n1 = "n" + std::to_string(lid.at(l1));
        body << "  const int64_t tot_ = " << n0 << " * " << n1 << ";\n";
        Element e;
        e.outer = &ksc;
        e.body_loop = l1;
        e.inner = n1;
        e.decode = [&](int ind) {
            const std::string pad(2 * ind, ' ');
            if (total < (1ull << 31)) {
                body << pad << "const int64_t i0 = (int64_t)((uint32_t)f_ / (uint32_t)" << n1 << ");\n";
                body << pad << "const int64_t i1 = (int64_t)((uint32_t)f_ - (uint32_t)i0 * (uint32_t)" << n1 << ");\n";
            } else {
                body << pad << "const int64_t i0 = f_ / " << n1 << ";\n" << pad << "const int64_t i1 = f_ - i0 * " << n1
                     << ";\n";
            }
        };
        e.compute = [&](int ind, const Scope *outer) {
            Scope sc0;
            sc0.parent = outer;
            Scope sc;
            sc.parent = &sc0;
            declare_scope(*l1, sc, ind);
            emit_blocks(*l1, sc, ind);
            write_back(*l1, sc, ind);
        };
        parts = cfg.xcd_parts && shifted_reads(l0);
        int64_t tasks = 0;
        if (!(parts && stencil_walk(e, n0, n1, l0.size, l1->size, cfg.reduce_unroll, &tasks)))
            grid_stride("tot_", cfg.reduce_unroll, e);
        parts = false;
    } else {
        Element e;
        e.outer = &ksc;
        e.body_loop = l0.isInnermost() ? &l0 : nullptr;
        e.unit = true;
        e.decode = [&](int ind) { body << std::string(2 * ind, ' ') << "const int64_t i0 = f_;\n"; };
        e.compute = [&](int ind, const Scope *outer) {
            Scope sc;
            sc.parent = outer;
            declare_scope(l0, sc, ind);
            emit_blocks(l0, sc, ind);
            write_back(l0, sc, ind);
        };
        parts = cfg.xcd_parts && shifted_reads(l0);
        grid_stride("n" + std::to_string(lid.at(&l0)), l0.isInnermost() ? cfg.reduce_unroll : 1, e);
        parts = false;
    }
    body << "  __shared__ __attribute__((aligned(16))) unsigned char bh_lds_[BH_WAVES * 16];\n";
    auto op_lambda = [&](const Acc &a) {
        const std::string T = hip_type(a.t);
        return "auto op_ = [](" + T + " x, " + T + " y) -> " + T + " { return " +
               combine_expr(a.instr->opcode, "x", "y") + "; };";
    };
    lane_axis = -1;
    // Store the results (in registers of thread 0) and run the tail.
    auto results = [&](int ind) {
        Scope fsc;
        for (const Acc &a : accs) {
            const bh_view &v = a.instr->operand[0];
            if (a.is_tmp)
                fsc.tmps.insert(v.base);
            else
                fsc.srep.insert(vkey(v));
        }
        std::set<std::string> stored;
        for (const Acc &a : accs) {
            if (a.is_tmp || !stored.insert(a.var).second) continue;
            const bh_view &v = a.instr->operand[0];
            indent(body, ind);
            body << "a" << bid.at(v.base) << "[" << index(v) << "] = " << a.var << ";\n";
        }
        declare_scope(unit, fsc, ind);
        for (size_t k = pos + 1; k < unit._block_list.size(); ++k) emit_block(unit._block_list[k], fsc, ind);
        write_back(unit, fsc, ind);
    };
    // One workgroup has the whole result: it finishes the unit itself and the finalize launch (4 us of the 10 us
    // that a sum of 1000 numbers takes on the device, and a launch on the host) is left out.  Not in the code of
    // large reductions, whose main loop should not share registers with a tail.
    // Only for a tail that shares no array with the loop: its thread would have to see the others' stores.
    bool one = total <= kOneWorkgroupItems;
    if (one) {
        std::set<const bh_base *> outs, in_loop;
        for (const Acc &a : accs) outs.insert(a.instr->operand[0].base);
        for (const bh_base *b : l0.getAllBases())
            if (!outs.count(b)) in_loop.insert(b);
        for (size_t k = pos + 1; k < unit._block_list.size(); ++k)
            for (const InstrPtr &i : jitk::allInstr(unit._block_list[k]))
                for (const bh_view &v : i->operand)
                    if (!bh_opcode_is_system(i->opcode) && !v.isConstant() && in_loop.count(v.base)) one = false;
    }
    std::set<std::string> done;
    for (const Acc &a : accs) {
        if (!done.insert(a.var).second) continue;
        const std::string T = hip_type(a.t);
        body << "  { " << op_lambda(a) << "\n";
        body << "    " << a.var << " = bh_block_reduce(" << a.var << ", op_, (" << T << " *)bh_lds_);\n";
        body << "    if (threadIdx.x == 0" << (one ? " && bh_nblk != 1" : "") << ") *(" << T << " *)" << slot_addr(a, "bh_bid")
             << " = " << a.var << ";\n";
        body << "    __syncthreads(); }\n";
    }
    if (one) {
        body << "  if (bh_nblk == 1 && threadIdx.x == 0) {\n";
        results(2);
        body << "  }\n";
        kp.one_workgroup = true;
    }
    main_body = body.str();
    body.str("");
    body.clear();

    // Finalize kernel: fold the partials, store, run the tail in thread 0.
    done.clear();
    if (one) body << "  if (bh_nparts == 1) return;\n";
    body << "  __shared__ __attribute__((aligned(16))) unsigned char bh_lds_[BH_WAVES * 16];\n";
    for (const Acc &a : accs) {
        if (!done.insert(a.var).second) continue;
        const std::string T = hip_type(a.t);
        body << "  " << T << " " << a.var << ";\n";
        body << "  { " << op_lambda(a) << "\n";
        body << "    " << T << " v_ = " << literal(jitk::sweep_identity(a.instr->opcode, a.t)) << ";\n";
        // Sixteen partials per thread are loaded before any is folded, so their memory latencies overlap
        // (one load in flight at a time made this one-workgroup kernel latency-bound: up to 4096
        // partials take one round trip); each thread still folds j_ = tid, tid + BH_WG, ... in order.
        body << "    for (unsigned j_ = threadIdx.x; j_ < bh_nparts; j_ += 16u * BH_WG) {\n";
        body << "      " << T << " x_[16];\n";
        body << "#pragma unroll\n";
        body << "      for (unsigned u_ = 0; u_ < 16u; ++u_)\n";
        body << "        if (j_ + u_ * BH_WG < bh_nparts) x_[u_] = *(const " << T << " *)"
             << slot_addr(a, "(j_ + u_ * BH_WG)") << ";\n";
        body << "#pragma unroll\n";
        body << "      for (unsigned u_ = 0; u_ < 16u; ++u_)\n";
        body << "        if (j_ + u_ * BH_WG < bh_nparts) v_ = op_(v_, x_[u_]);\n";
        body << "    }\n";
        body << "    " << a.var << " = bh_block_reduce(v_, op_, (" << T << " *)bh_lds_);\n";
        body << "    __syncthreads(); }\n";
    }
    body << "  if (threadIdx.x != 0) return;\n";
    results(1);
    kp.fin_name = "bh_kernel_fin";
}

// ---- SCAN: decoupled look-back over tiles of BH_WG * items elements
void Writer::emit_scan() {
    const LoopB &l0 = unit._block_list.back().getLoop();
    kp.work_items = static_cast<uint64_t>(l0.size);
    InstrPtr acc;
    for (const InstrPtr &i : jitk::allLocalInstr(l0))
        if (bh_opcode_is_accumulate(i->opcode)) acc = i;
    const bh_type t = acc->operand[0].base->dtype();
    const std::string T = hip_type(t);
    const int items = cfg.scan_items;
    const int64_t tile_elems = static_cast<int64_t>(kp.block) * items;
    // V neighbours per thread when every array is walked contiguously (16 bytes of the widest array, so that a
    // wave's stores are contiguous as well)
    int V = 1;
    {
        bool unit = true;
        int widest = bh_type_size(t);
        for (const InstrPtr &i : jitk::allInstr(l0)) {
            if (bh_opcode_is_system(i->opcode)) continue;
            for (size_t o = 0; o < i->operand.size(); ++o) {
                const bh_view &v = i->operand[o];
                if (v.isConstant() || (i->opcode == BH_GATHER && o == 1) || v.ndim < 1) continue;
                unit &= v.ndim == 1 && (v.stride[0] == 1 || v.stride[0] == 0 || v.shape[0] == 1);
                if (o > 0 && std::find(kp.params.begin(), kp.params.end(), v.base) != kp.params.end())
                    widest = std::max(widest, bh_type_size(v.base->dtype()));
            }
        }
        if (unit) V = std::max(1, std::min(4, 16 / widest));
        while (items % V != 0) V /= 2;
    }
    const int groups = items / V;
    lane_axis = 0;
    lane_run = V;
    const int64_t ntiles = (l0.size + tile_elems - 1) / tile_elems;
    kp.grid = static_cast<uint64_t>(std::max<int64_t>(1, ntiles));
    // Scratch layout: [tile counter u64 = epoch << 32 | tiles taken, pad to 256], then one record
    // of 8 bytes per 32-bit chunk of T per tile; no offset depends on the size.
    const int64_t nchunks = std::max<int64_t>(1, bh_type_size(t) / 4);
    kp.scratch_bytes = 256 + ntiles * 8 * nchunks;
    const std::string ident = literal(jitk::sweep_identity(acc->opcode, t));
    scan_instr = acc.get();
    scan_sink = "x_";
    kp.uses_error_flag = true;

    body << "  auto op_ = [](" << T << " x, " << T << " y) -> " << T << " { return "
         << combine_expr(acc->opcode, "x", "y") << "; };\n";
    body << "  unsigned char *bh_rec = bh_scratch + 256;\n";
    body << "  __shared__ unsigned int bh_tile_s, bh_ep_s;\n";
    body << "  __shared__ " << T << " bh_wtot_[BH_WAVES];\n";
    body << "  __shared__ " << T << " bh_excl_s;\n";
    // Tiles are numbered in the order workgroups start, so a tile only waits for tiles whose
    // workgroups already run.  The workgroup taking the last tile starts the next epoch.
    body << "  if (threadIdx.x == 0) {\n";
    body << "    const unsigned long long t_ = atomicAdd((unsigned long long *)bh_scratch, 1ull);\n";
    body << "    bh_tile_s = (unsigned int)t_;\n    bh_ep_s = (unsigned int)(t_ >> 32);\n";
    body << "    if ((unsigned int)t_ == bh_nblk - 1u)\n";
    body << "      __hip_atomic_store((unsigned long long *)bh_scratch, (unsigned long long)(bh_ep_s + 1u) << 32, "
            "__ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);\n";
    body << "  }\n";
    body << "  __syncthreads();\n";
    body << "  const int64_t tile_ = (int64_t)__builtin_amdgcn_readfirstlane(bh_tile_s);\n"
            "  const unsigned int fb_ = bh_ep_s << 2;\n";
    body << "  const int lane_ = threadIdx.x & 63, wave_ = threadIdx.x >> 6;\n";
    body << "  const int64_t tb_ = tile_ * " << tile_elems << ";\n";
    body << "  " << T << " v_[" << items << "];\n";
    Scope ksc;
    declare_scope(unit, ksc, 1);
    // A thread owns `groups` runs of V neighbouring elements: 16-byte loads where the views are
    // contiguous, and one wave scan per run instead of one per element.  The elements first (every load of
    // the tile issued before the first wave scan waits for one): a full tile without bounds checks, the
    // last tile with them; both unrolled, so that v_ stays in registers.  Measured: the int64 running count of
    // 6e7 float32 279 -> 180 us of device time (one element per thread and wave scan, 16 per tile and thread, before; 64
    // now).  At no tile size and length is it behind the form before: 8 per thread 391 -> 385 us, 1e6 elements 17.8 -> 17.2.
    for (int full = 1; full >= 0; --full) {
        if (full)
            body << "  if (tb_ + " << tile_elems << " <= n" << lid.at(&l0) << ") {\n";
        else
            body << "  } else {\n";
        body << "#pragma unroll\n  for (int j_ = 0; j_ < " << groups << "; ++j_) {\n";
        body << "#pragma unroll\n  for (int e_ = 0; e_ < " << V << "; ++e_) {\n";
        body << "    const int64_t i0 = tb_ + (((int64_t)wave_ * " << groups << " + j_) * 64 + lane_) * " << V << " + e_;\n";
        body << "    " << T << " x_ = " << ident << ";\n";
        body << (full ? "    {\n" : "    if (i0 < n" + std::to_string(lid.at(&l0)) + ") {\n");
        {
            Scope sc;
            sc.parent = &ksc;
            declare_scope(l0, sc, 3);
            emit_blocks(l0, sc, 3);
            write_back(l0, sc, 3);
        }
        body << "    }\n    v_[j_ * " << V << " + e_] = x_;\n  }\n  }\n";
    }
    body << "  }\n";
    // Prefixes inside a run by the thread, of the runs across the wave, and carried from row to row.
    body << "  " << T << " carry_ = " << ident << ", g_[" << groups << "];\n";
    body << "#pragma unroll\n  for (int j_ = 0; j_ < " << groups << "; ++j_) {\n";
    body << "#pragma unroll\n    for (int e_ = 1; e_ < " << V << "; ++e_) v_[j_ * " << V << " + e_] = op_(v_[j_ * " << V
         << " + e_ - 1], v_[j_ * " << V << " + e_]);\n";
    body << "    " << T << " tot_;\n";
    body << "    const " << T << " ex_ = bh_wave_exclusive_scan(v_[j_ * " << V << " + " << V - 1 << "], op_, " << T << "(" << ident
         << "), &tot_);\n";
    body << "    g_[j_] = op_(carry_, ex_);\n    carry_ = op_(carry_, tot_);\n  }\n";
    body << "  if (lane_ == 63) bh_wtot_[wave_] = carry_;\n  __syncthreads();\n";
    body << "  " << T << " wpre_ = " << ident << ", ttot_ = " << ident << ";\n";
    body << "  for (int w_ = 0; w_ < BH_WAVES; ++w_) { if (w_ < wave_) wpre_ = op_(wpre_, bh_wtot_[w_]); ttot_ = op_(ttot_, bh_wtot_[w_]); }\n";
    // Look-back by wave 0: lane l reads the record of tile (hi - l); the window ends at the
    // nearest inclusive prefix, and the aggregates after it are folded in.
    const std::string LB = "bh_lookback<" + T + ">";
    body << "  if (wave_ == 0) {\n";
    body << "    " << T << " ex_ = " << ident << ";\n";
    body << "    if (tile_ == 0) {\n";
    body << "      if (lane_ == 0) " << LB << "::put(bh_rec, 0, ttot_, fb_ | 2u);\n";
    body << "    } else {\n";
    body << "      if (lane_ == 0) " << LB << "::put(bh_rec, tile_, ttot_, fb_ | 1u);\n";
    body << "      for (int64_t hi_ = tile_ - 1;; hi_ -= 64) {\n";
    body << "        const int64_t j_ = hi_ - lane_;\n";
    body << "        " << T << " w_ = " << ident << ";\n";
    body << "        unsigned int st_ = 2u;\n";
    // A record that never arrives (lost or of another epoch) must not hang the device: after
    // BH_SCAN_SPIN polls the wait gives up, raises BH_ERR_SCAN and the host reports it.
    body << "        if (j_ >= 0) {\n";
    body << "          unsigned int sp_ = 0u;\n";
    body << "          while ((st_ = " << LB << "::get(bh_rec, j_, fb_, &w_)) == 0u) {\n";
    body << "            if (++sp_ >= BH_SCAN_SPIN) { atomicOr(bh_err, BH_ERR_SCAN); st_ = 2u; break; }\n";
    body << "          }\n";
    body << "        }\n";
    body << "        const unsigned long long pm_ = __ballot(st_ == 2u);\n";
    body << "        const int first_ = pm_ ? __ffsll((long long)pm_) - 1 : 64;\n";
    body << "        ex_ = op_(bh_wave_reduce(lane_ <= first_ ? w_ : " << ident << ", op_), ex_);\n";
    body << "        if (pm_) break;\n";
    body << "      }\n";
    body << "      if (lane_ == 0) " << LB << "::put(bh_rec, tile_, op_(ex_, ttot_), fb_ | 2u);\n";
    body << "    }\n";
    body << "    if (lane_ == 0) bh_excl_s = ex_;\n";
    body << "  }\n";
    body << "  __syncthreads();\n";
    body << "  const " << T << " pre_ = op_(bh_excl_s, wpre_);\n";
    const bh_view &out = acc->operand[0];
    for (int full = 1; full >= 0; --full) {
        body << (full ? "  if (tb_ + " + std::to_string(tile_elems) + " <= n" + std::to_string(lid.at(&l0)) + ") {\n" : "  } else {\n");
        body << "#pragma unroll\n  for (int j_ = 0; j_ < " << groups << "; ++j_) {\n    const " << T << " p_ = op_(pre_, g_[j_]);\n";
        body << "#pragma unroll\n  for (int e_ = 0; e_ < " << V << "; ++e_) {\n";
        body << "    const int64_t i0 = tb_ + (((int64_t)wave_ * " << groups << " + j_) * 64 + lane_) * " << V << " + e_;\n";
        const std::string at = "a" + std::to_string(bid.at(out.base)) + "[" + index(out) + "]";
        const std::string value = "op_(p_, v_[j_ * " + std::to_string(V) + " + e_])";
        body << (full ? "    " : "    if (i0 < n" + std::to_string(lid.at(&l0)) + ") ")
             << (streamed(out) ? "__builtin_nontemporal_store(" + value + ", &" + at + ")" : at + " = " + value)
             << ";\n  }\n  }\n";
    }
    body << "  }\n";
    write_back(unit, ksc, 1);
}

// ---- SERIAL: one thread runs the whole loop nest
void Writer::emit_serial() {
    kp.block = 64;
    kp.grid = 1;
    body << "  if (bh_bid != 0 || threadIdx.x != 0) return;\n";
    emit_body(unit, nullptr, 1);
    kp.work_items = 1;
}

KernelPlan Writer::plan(Strategy s) {
    kp.strategy = s;
    kp.name = "bh_kernel";
    if (s == Strategy::SERIAL) kp.block = 64;
    switch (s) {
        case Strategy::MAP: emit_map(); break;
        case Strategy::ROW_REDUCE: emit_row_reduce(); break;
        case Strategy::SEG_REDUCE: emit_seg_reduce(); break;
        case Strategy::FULL_REDUCE: emit_full_reduce(); break;
        case Strategy::SCAN: emit_scan(); break;
        case Strategy::SERIAL: emit_serial(); break;
    }
    std::vector<KernelParam> params = parameters();
    const bool two_kernels = !kp.fin_name.empty();
    if (s == Strategy::FULL_REDUCE || s == Strategy::SCAN || (s == Strategy::SEG_REDUCE && two_kernels)) {
        params.push_back({"unsigned char *", "bh_scratch", true});
        ArgSpec a;
        a.kind = ArgSpec::SCRATCH_PTR;
        kp.args.push_back(a);
    }
    if (s == Strategy::FULL_REDUCE) {
        // The finalize kernel folds this many partials (the main kernel's grid).
        params.push_back({"uint32_t", "bh_nparts", false});
        ArgSpec a;
        a.kind = ArgSpec::GRID_U32;
        a.size = 4;
        a.align = 4;
        kp.args.push_back(a);
    }
    kp.param_decls.clear();
    kp.param_types.clear();
    kp.param_names.clear();
    for (const KernelParam &p : params) {
        kp.param_decls.push_back(p.is_ptr ? p.type + "__restrict__ " + p.name : "const " + p.type + " " + p.name);
        kp.param_types.push_back(p.type);
        kp.param_names.push_back(p.name);
    }
    // The body is a device function of the parameters and of the workgroup's place in its
    // grid; the kernels below (and the batched kernels of batch_source) only call it.
    std::string plist, nlist;
    for (size_t i = 0; i < params.size(); ++i) {
        plist += (i ? ",\n    " : "") + kp.param_decls[i];
        nlist += (i ? ", " : "") + params[i].name;
    }
    std::ostringstream dev;
    const std::string main_src = two_kernels ? main_body : body.str();
    // Gathers mark an index outside its base in bh_bad_; the flag is raised once per thread at the end
    // (every early return in a body comes before its first gather).
    const std::string bad0 = kp.uses_gather_flag ? "  bool bh_bad_ = false;\n" : "";
    const std::string bad1 = kp.uses_gather_flag ? "  if (bh_bad_) atomicOr(bh_err, BH_ERR_INDEX);\n" : "";
    dev << "__device__ __forceinline__ void bh_main_(" << plist << (plist.empty() ? "" : ",\n    ")
        << "const unsigned bh_bid, const unsigned bh_nblk) {\n" << bad0 << main_src << bad1 << "}\n";
    const bool seg = s == Strategy::SEG_REDUCE;
    if (two_kernels)
        dev << "\n__device__ __forceinline__ void bh_fin_(" << plist << (seg ? ",\n    const unsigned bh_bid" : "")
            << ") {\n" << bad0 << body.str() << bad1 << "}\n";
    kp.device_code = dev.str();
    std::ostringstream src;
    // Occupancy hint for the main kernel (waves per SIMD the register allocator must allow).
    kp.attributes = cfg.waves_per_eu > 0 && s != Strategy::SERIAL
                        ? " __attribute__((amdgpu_waves_per_eu(" + std::to_string(cfg.waves_per_eu) + ")))"
                        : "";
    // With xcd_remap the grid-stride skeletons number their workgroups per XCD (bh_xcd_block); the
    // scan skeleton takes its tiles from a ticket counter and the serial one has one workgroup.
    const bool remap = cfg.xcd_remap && (s == Strategy::MAP || s == Strategy::FULL_REDUCE || s == Strategy::ROW_REDUCE);
    src << kp.device_code << "\nextern \"C\" __global__ void __launch_bounds__(" << kp.block << ")" << kp.attributes
        << " " << kp.name << "("
        << plist << ") {\n  bh_main_(" << nlist << (nlist.empty() ? "" : ", ")
        << (remap ? "bh_xcd_block(blockIdx.x, gridDim.x)" : "blockIdx.x") << ", gridDim.x);\n}\n";
    if (two_kernels)
        src << "\nextern \"C\" __global__ void __launch_bounds__(" << kp.block << ") " << kp.fin_name << "(" << plist
            << ") {\n  bh_fin_(" << nlist << (seg ? ", blockIdx.x" : "") << ");\n}\n";
    kp.source = src.str();
    return kp;
}

bool scan_compatible(const LoopB &l0, const InstrPtr &acc) {
    if (!(acc->opcode == BH_ADD_ACCUMULATE || acc->opcode == BH_MULTIPLY_ACCUMULATE)) return false;
    if (!l0.isInnermost()) return false;
    const bh_base *out = acc->operand[0].base;
    for (const InstrPtr &i : jitk::allInstr(l0)) {
        if (i == acc) continue;
        for (const bh_view &v : i->operand)
            if (!v.isConstant() && v.base == out) return false;
    }
    for (const bh_view &v : acc->operand)
        if (&v != &acc->operand[0] && !v.isConstant() && v.base == out) return false;
    return true;
}

} // namespace

Strategy classify_root_block(const LoopB &l0) {
    if (l0._sweeps.empty()) return Strategy::MAP;
    const auto local = jitk::allLocalInstr(l0);
    auto is_local = [&](const InstrPtr &s) { return std::find(local.begin(), local.end(), s) != local.end(); };
    bool all_red_local = true;
    for (const InstrPtr &s : l0._sweeps)
        if (!bh_opcode_is_reduction(s->opcode) || !is_local(s)) all_red_local = false;
    if (all_red_local) return Strategy::FULL_REDUCE;
    if (l0._sweeps.size() == 1) {
        const InstrPtr &s = *l0._sweeps.begin();
        if (bh_opcode_is_accumulate(s->opcode) && is_local(s) && scan_compatible(l0, s)) return Strategy::SCAN;
    }
    return Strategy::SERIAL;
}

namespace {
// Sweep axis per input rank of every sweep in `l` (nested loops included).
void sweep_axes(const LoopB &l, std::map<int64_t, std::set<int> > &out) {
    for (const InstrPtr &i : jitk::allInstr(l))
        if (bh_opcode_is_sweep(i->opcode) && i->operand.size() > 1 && !i->operand[1].isConstant())
            out[i->operand[1].ndim].insert(i->sweep_axis());
}
} // namespace

bool root_merge_allowed(const LoopB &l1, const LoopB &l2) {
    // Sweeps along two axes of inputs of one rank (a column sum and a row sum of one shape) cannot
    // both be inner reductions of one loop nest, at any depth of the nest; the merged block would
    // run on one thread.  (A full reduction through a row temporary reduces inputs of two ranks.)
    std::map<int64_t, std::set<int> > axes;
    sweep_axes(l1, axes);
    sweep_axes(l2, axes);
    for (const auto &kv : axes)
        if (kv.first > 1 && kv.second.size() > 1) return false;
    if (l1.rank != 0 || l2.rank != 0) return true;
    size_t nsweeps = l1._sweeps.size() + l2._sweeps.size();
    bool acc = false;
    for (const InstrPtr &s : l1._sweeps) acc |= bh_opcode_is_accumulate(s->opcode) != 0;
    for (const InstrPtr &s : l2._sweeps) acc |= bh_opcode_is_accumulate(s->opcode) != 0;
    if (acc && nsweeps > 1) return false;
    if (acc && (!l1.isInnermost() || !l2.isInnermost())) return false;
    if (acc) {
        // Work that shares no array with the scan gains nothing from its loop and would wait on its
        // tiles' look-back: it keeps a map of its own (measured on 4096 uneven arrays: a gather beside
        // an independent cumsum took 2.12 ms fused, 0.82 + 1.18 ms apart).
        const std::set<const bh_base *> b1 = l1.getAllBases();
        bool shared = false;
        for (const bh_base *b : l2.getAllBases()) shared |= b1.count(b) != 0;
        if (!shared) return false;
    }
    return true;
}

namespace {
// A block that only writes sweep identities (BH_IDENTITY of a constant).
bool identity_only(const LoopB &l) {
    const auto all = jitk::allInstr(l);
    if (all.empty()) return false;
    for (const InstrPtr &i : all)
        if (i->opcode != BH_IDENTITY || !i->operand[1].isConstant()) return false;
    return true;
}

// True when every identity in `ids` initialises the output of a sweep of `l0`.
bool identities_of(const std::vector<Block> &ids, const LoopB &l0) {
    std::set<const bh_base *> outs;
    for (const InstrPtr &s : l0._sweeps) outs.insert(s->operand[0].base);
    for (const Block &b : ids)
        for (const InstrPtr &i : jitk::allInstr(b))
            if (!outs.count(i->operand[0].base)) return false;
    return true;
}
} // namespace

namespace {
// Iterations one thread runs for a block: the product of its nested loop sizes.
uint64_t serial_cost(const Block &b) {
    if (b.isInstr()) return 1;
    const LoopB &l = b.getLoop();
    uint64_t inner = 1;
    for (const Block &c : l._block_list) inner = std::max(inner, serial_cost(c));
    return static_cast<uint64_t>(std::max<int64_t>(l.size, 0)) * inner;
}

// Blocks this small run in thread 0 of a FULL_REDUCE finalize kernel instead of a launch of their own.
constexpr uint64_t kTailLimit = 256;
bool tail_block(const Block &b) { return serial_cost(b) <= kTailLimit; }

bool is_full_reduce_loop(const Block &b) {
    return !b.isInstr() && !b.getLoop()._sweeps.empty() && classify_root_block(b.getLoop()) == Strategy::FULL_REDUCE;
}

// True when the kernel's last sizeable block is a FULL_REDUCE loop (only tail blocks after it).
bool open_tail(const LoopB &kernel) {
    for (auto it = kernel._block_list.rbegin(); it != kernel._block_list.rend(); ++it) {
        if (is_full_reduce_loop(*it)) return true;
        if (!(it->isSystemOnly() || tail_block(*it))) return false;
    }
    return false;
}
} // namespace

namespace {
// Bases a kernel reads and writes (a BH_FREE counts as a write).
struct Access {
    std::set<const bh_base *> reads, writes;
    explicit Access(const LoopB &k) {
        for (const InstrPtr &i : jitk::allInstr(k)) {
            for (size_t o = 0; o < i->operand.size(); ++o) {
                const bh_view &v = i->operand[o];
                if (v.isConstant()) continue;
                if (o == 0 || i->opcode == BH_FREE) {
                    writes.insert(v.base);
                } else {
                    reads.insert(v.base);
                }
            }
        }
    }
    // True when running `this` before `m` instead of after it could change a result.
    bool conflicts(const Access &m) const {
        for (const bh_base *b : m.writes)
            if (reads.count(b) || writes.count(b)) return true;
        for (const bh_base *b : writes)
            if (m.reads.count(b)) return true;
        return false;
    }
};
} // namespace

std::vector<LoopB> fold_serial_tails(std::vector<LoopB> kernels) {
    std::vector<LoopB> out;
    for (LoopB &k : kernels) {
        bool small = !k._block_list.empty();
        for (const Block &b : k._block_list) small &= b.isSystemOnly() || tail_block(b);
        size_t target = out.size();
        if (small) {
            // The nearest earlier kernel with an open tail, if `k` can move before the kernels after it.
            const Access ak(k);
            for (size_t m = out.size(); m-- > 0;) {
                if (open_tail(out[m])) {
                    target = m;
                    break;
                }
                if (ak.conflicts(Access(out[m]))) break;
            }
        }
        if (target < out.size()) {
            for (Block &b : k._block_list) out[target]._block_list.push_back(std::move(b));
            out[target].metadataUpdate();
        } else {
            out.push_back(std::move(k));
        }
    }
    return out;
}

namespace {
// The bases a unit addresses as arrays (its writer's parameters).
std::set<const bh_base *> param_bases(const LoopB &unit) {
    std::set<const bh_base *> out;
    for (const bh_base *b : unit.getAllNonTemps()) out.insert(b);
    return out;
}

// The position of a kernel's only computing block when that is a loop, else -1.
int only_loop(const LoopB &kernel) {
    int at = -1;
    for (size_t k = 0; k < kernel._block_list.size(); ++k) {
        const Block &b = kernel._block_list[k];
        if (b.isSystemOnly()) continue;
        if (b.isInstr() || at >= 0) return -1;
        at = static_cast<int>(k);
    }
    return at;
}
} // namespace

std::vector<bool> crowded_reductions(const std::vector<LoopB> &kernels, int batch_min) {
    std::vector<bool> out(kernels.size(), false);
    if (batch_min <= 0 || kernels.size() < static_cast<size_t>(batch_min)) return out;
    // Segmented blocks that a crowd leaves to the rows, by what their code is made of: operations, types, axis.
    std::map<std::string, std::vector<size_t> > like;
    for (size_t k = 0; k < kernels.size(); ++k) {
        const std::set<const bh_base *> params = param_bases(kernels[k]);
        std::string key;
        for (const Block &b : kernels[k]._block_list) {
            if (b.isInstr() || b.getLoop().rank != 0) continue;
            const SegForm f = seg_form(b.getLoop(), params, false, true);
            if (f.C == nullptr || seg_form(b.getLoop(), params, true, true).C != nullptr) continue;
            key += f.columns ? "c" : "r";
            for (const InstrPtr &i : jitk::allInstr(*f.C)) {
                if (bh_opcode_is_system(i->opcode)) continue;
                key += std::to_string(i->opcode) + ":";
                for (const bh_view &v : i->operand) key += v.isConstant() ? "-" : std::to_string(static_cast<int>(v.base->dtype())) + "/" + std::to_string(v.ndim) + ",";
            }
        }
        if (!key.empty()) like[key].push_back(k);
    }
    for (const auto &l : like)
        if (l.second.size() >= static_cast<size_t>(batch_min))
            for (size_t k : l.second) out[k] = true;
    return out;
}

std::vector<LoopB> fold_row_tails(std::vector<LoopB> kernels, int batch_min) {
    const std::vector<bool> crowd = crowded_reductions(kernels, batch_min);
    std::vector<LoopB> out;
    bool crowd_a = false;  // of out.back()
    for (size_t n = 0; n < kernels.size(); ++n) {
        LoopB &k = kernels[n];
        const int b = only_loop(k);
        const int a = out.empty() || crowd_a ? -1 : only_loop(out.back());
        bool folded = false;
        if (a >= 0 && b >= 0) {
            const LoopB &la = out.back()._block_list[a].getLoop(), &lb = k._block_list[b].getLoop();
            if (la.rank == 0 && lb.rank == 0 && la.size == lb.size && lb.isInnermost() && lb._sweeps.empty() &&
                seg_form(la, param_bases(out.back()), false, true).C != nullptr &&
                jitk::mergeable(out.back()._block_list[a], k._block_list[b], false)) {
                LoopB merged = out.back();
                merged._block_list[a] = Block(jitk::merge(la, lb));
                for (size_t i = 0; i < k._block_list.size(); ++i)
                    if (static_cast<int>(i) != b) merged._block_list.push_back(k._block_list[i]);
                merged.metadataUpdate();
                if (seg_form(merged._block_list[a].getLoop(), param_bases(merged), false).C != nullptr) {
                    out.back() = std::move(merged);
                    folded = true;
                }
            }
        }
        if (folded) continue;
        out.push_back(std::move(k));
        crowd_a = crowd[n];
    }
    return out;
}

namespace {
// Every operand dimension of every instruction must be iterated by the enclosing loop of the
// matching rank, and that loop may not run past the dimension (the generated index is
// start + sum(i_rank * stride), in bounds only then).  `sizes` holds the enclosing loop sizes
// by rank.
void verify_loop_ranks(const LoopB &l, std::vector<int64_t> &sizes, std::string &err) {
    if (l.rank >= 0) {
        if (static_cast<int64_t>(sizes.size()) != l.rank) {
            err += "loop rank " + std::to_string(l.rank) + " nested at depth " + std::to_string(sizes.size()) + "; ";
            return;
        }
        sizes.push_back(l.size);
    }
    for (const Block &b : l._block_list) {
        if (!b.isInstr()) {
            verify_loop_ranks(b.getLoop(), sizes, err);
            continue;
        }
        const InstrPtr &i = b.getInstr();
        if (bh_opcode_is_system(i->opcode)) continue;
        for (size_t o = 0; o < i->operand.size(); ++o) {
            const bh_view &v = i->operand[o];
            if (v.isConstant()) continue;
            if (i->opcode == BH_GATHER && o == 1) continue;            // indexed by value, checked at run time
            if ((i->opcode == BH_SCATTER || i->opcode == BH_COND_SCATTER) && o == 0) continue;
            int hidden = BH_MAXDIM;
            if (o == 0 && bh_opcode_is_reduction(i->opcode) && i->operand[1].ndim > 1) hidden = i->sweep_axis();
            if (o == 0 && bh_opcode_is_reduction(i->opcode) && i->operand[1].ndim <= 1) continue;  // scalar output
            for (int64_t d = 0; d < v.ndim; ++d) {
                const int64_t t = d >= hidden ? d + 1 : d;
                // an extent-1 axis only ever takes index 0 unless a loop of several iterations walks it
                if (v.shape[d] <= 1 && (v.stride[d] == 0 || t >= static_cast<int64_t>(sizes.size()) || sizes[t] <= 1))
                    continue;
                if (t >= static_cast<int64_t>(sizes.size()) || sizes[t] > v.shape[d]) {
                    err += std::string(bh_opcode_text(i->opcode)) + " operand " + std::to_string(o) + " dim " +
                           std::to_string(d) + " (extent " + std::to_string(v.shape[d]) + ") iterated by rank " +
                           std::to_string(t) + (t < static_cast<int64_t>(sizes.size()) ? " of size " + std::to_string(sizes[t]) : " (none)") + "; ";
                }
            }
        }
    }
    if (l.rank >= 0) sizes.pop_back();
}
} // namespace

std::string verify_kernel(const LoopB &kernel) {
    std::vector<int64_t> sizes;
    std::string err;
    verify_loop_ranks(kernel, sizes, err);
    return err;
}

std::vector<KernelPlan> plan_kernel(const LoopB &kernel, const WriterConfig &cfg) {
    std::vector<KernelPlan> ret;
    auto emit = [&](LoopB unit, Strategy s) {
        unit.metadataUpdate();
        Writer w(unit, cfg);
        ret.push_back(w.plan(s));
    };
    // Each top-level loop is one launch.  Identity writers that precede a sweeping
    // loop are folded into it when its skeleton seeds the sweep with the identity
    // itself (FULL_REDUCE, SCAN); otherwise they run first.
    std::vector<Block> pending;
    const std::vector<Block> &blocks = kernel._block_list;
    for (size_t bi = 0; bi < blocks.size(); ++bi) {
        const Block &b = blocks[bi];
        if (b.isInstr()) {
            pending.push_back(b);
            continue;
        }
        if (b.isSystemOnly()) continue;
        if (identity_only(b.getLoop())) {
            pending.push_back(b);
            continue;
        }
        const LoopB &l0 = b.getLoop();
        Strategy s = classify_root_block(l0);
        const bool seeds_itself = s == Strategy::FULL_REDUCE || s == Strategy::SCAN;
        std::vector<Block> scalar_ids;
        if (!(seeds_itself && identities_of(pending, l0))) {
            for (const Block &p : pending) {
                if (p.isInstr()) {
                    scalar_ids.push_back(p);
                } else {
                    emit(LoopB(-1, 1, {p}), Strategy::MAP);
                }
            }
        }
        pending.clear();
        if (s == Strategy::MAP && l0.size == 0) continue;
        // Scalar writers in front of a map run first as their own one-thread launch, so the
        // map keeps its grid instead of running serially behind them.
        if (s == Strategy::MAP && !scalar_ids.empty()) {
            emit(LoopB(-1, 1, scalar_ids), Strategy::SERIAL);
            scalar_ids.clear();
        }
        LoopB unit(-1, 1, scalar_ids);
        unit._block_list.push_back(b);
        if (s == Strategy::MAP && cfg.row_reduce) {
            unit.metadataUpdate();
            if (seg_form(l0, param_bases(unit), cfg.crowd).C != nullptr) {
                s = Strategy::SEG_REDUCE;
            } else if (!row_lane_loops(l0).empty()) {
                s = Strategy::ROW_REDUCE;
            }
        }
        if (s == Strategy::FULL_REDUCE) {
            while (bi + 1 < blocks.size() && (blocks[bi + 1].isSystemOnly() || tail_block(blocks[bi + 1])))
                unit._block_list.push_back(blocks[++bi]);
        }
        emit(unit, s);
    }
    for (const Block &p : pending) {
        if (p.isInstr()) {
            emit(LoopB(-1, 1, {p}), Strategy::SERIAL);
        } else {
            emit(LoopB(-1, 1, {p}), Strategy::MAP);
        }
    }
    return ret;
}

std::vector<size_t> arg_offsets(const std::vector<ArgSpec> &args, size_t *total) {
    std::vector<size_t> off;
    size_t n = 0;
    for (const ArgSpec &a : args) {
        while (n % static_cast<size_t>(a.align)) ++n;
        off.push_back(n);
        n += static_cast<size_t>(a.size);
    }
    while (n % 8) ++n;
    if (total != nullptr) *total = n;
    return off;
}

std::string persist_source(const std::vector<const KernelPlan *> &codes) {
    std::ostringstream s;
    std::ostringstream cases;
    for (size_t c = 0; c < codes.size(); ++c) {
        const KernelPlan &p = *codes[c];
        const std::string tag = "_c" + std::to_string(c) + "_";
        std::string code = p.device_code;
        for (const char *fn : {"bh_main_", "bh_fin_"}) {
            const std::string from = std::string("void ") + fn + "(";
            const std::string to = std::string("void ") + fn + tag.substr(1) + "(";
            for (size_t pos = code.find(from); pos != std::string::npos; pos = code.find(from, pos + to.size()))
                code.replace(pos, from.size(), to);
        }
        s << code << "\n";
        const std::vector<size_t> off = arg_offsets(p.args, nullptr);
        std::string unpack;
        for (size_t i = 0; i < p.param_types.size(); ++i) {
            const std::string &t = p.param_types[i];
            const bool ptr = !t.empty() && t.back() == '*';
            unpack += std::string(i ? ", " : "") + "*(" + t + (ptr ? "const *" : " const *") + ")(A_ + " +
                      std::to_string(off[i]) + ")";
        }
        const std::string sep = unpack.empty() ? "" : ", ";
        cases << "        case " << 2 * c << "u: bh_main" << tag << "(" << unpack << sep << "b_, nb_); break;\n";
        if (!p.fin_name.empty()) cases << "        case " << 2 * c + 1 << "u: bh_fin" << tag << "(" << unpack << "); break;\n";
    }
    // Workgroup w of the cooperative grid runs tasks w, w + grid, ... of each level, the levels in
    // order with a grid barrier between them.  A task is (case, workgroup number within its launch,
    // that launch's workgroup count, arguments offset / 16); case 2c runs code c's main body, 2c + 1
    // its finalize; any other case (padding) nothing.  All control flow is wave-uniform.
    s << "\nextern \"C\" __global__ void __launch_bounds__(256) bh_kernel_persist("
      << "const unsigned char *__restrict__ bh_args, const uint4 *__restrict__ bh_tasks, "
         "const unsigned *__restrict__ bh_levels, const unsigned bh_nlevels, unsigned *__restrict__ bh_bar, "
         "unsigned *__restrict__ bh_gerr, const unsigned bh_spin) {\n"
      << "  for (unsigned L_ = 0; L_ < bh_nlevels; ++L_) {\n"
      << "    const unsigned t1_ = __builtin_amdgcn_readfirstlane(bh_levels[L_ + 1u]);\n"
      << "    for (unsigned t_ = __builtin_amdgcn_readfirstlane(bh_levels[L_]) + blockIdx.x; t_ < t1_; t_ += gridDim.x) {\n"
      << "      const uint4 k_ = bh_tasks[t_];\n"
      << "      const unsigned c_ = __builtin_amdgcn_readfirstlane(k_.x);\n"
      << "      const unsigned b_ = __builtin_amdgcn_readfirstlane(k_.y);\n"
      << "      const unsigned nb_ = __builtin_amdgcn_readfirstlane(k_.z);\n"
      << "      const unsigned char *A_ = bh_args + (size_t)__builtin_amdgcn_readfirstlane(k_.w) * 16u;\n"
      << "      switch (c_) {\n" << cases.str() << "        default: break;\n      }\n"
      << "      __syncthreads();\n"
      << "    }\n"
      << "    if (L_ + 1u < bh_nlevels) bh_grid_sync(bh_bar, (L_ + 1u) * gridDim.x, bh_gerr, bh_spin);\n"
      << "  }\n"
      << "  bh_grid_exit(bh_bar);\n"
      << "}\n";
    return s.str();
}

std::string batch_source(const KernelPlan &p) {
    const std::vector<size_t> off = arg_offsets(p.args, nullptr);
    std::string unpack;
    for (size_t i = 0; i < p.param_types.size(); ++i) {
        const std::string &t = p.param_types[i];
        const bool ptr = !t.empty() && t.back() == '*';
        unpack += std::string(i ? ",\n      " : "") + "*(" + t + (ptr ? "const *" : " const *") + ")(A_ + " +
                  std::to_string(off[i]) + ")";
    }
    const std::string sep = unpack.empty() ? "" : ", ";
    std::ostringstream s;
    s << p.device_code;
    if (p.strategy == Strategy::SCAN) {
        // A scan tile takes its tile number from its item's ticket counter, so any workgroup may run
        // any item: bh_first holds the item of each workgroup (the order is the host's; all ones: no
        // item, the workgroup ends at once), then from position bh_items (the workgroup count) the tile
        // count of each item.
        s << "\nextern \"C\" __global__ void __launch_bounds__(" << p.block << ")" << p.attributes
          << " bh_kernel_batch("
          << "const unsigned char *__restrict__ bh_args, const unsigned *__restrict__ bh_first, const unsigned bh_items, "
             "const unsigned bh_stride) {\n"
          << "  const unsigned it_ = bh_first[blockIdx.x];\n"
          << "  if (it_ == 0xffffffffu) return;\n"
          << "  const unsigned char *A_ = bh_args + (size_t)it_ * bh_stride;\n"
          << "  bh_main_(" << unpack << sep << "blockIdx.x, bh_first[bh_items + it_]);\n}\n";
        return s.str();
    }
    // Workgroup b of the batched grid runs workgroup b - first[i] of item i, where
    // first[i] <= b < first[i + 1]; each item's packed arguments sit at args + i * stride.
    s << "\nextern \"C\" __global__ void __launch_bounds__(" << p.block << ")" << p.attributes << " bh_kernel_batch("
      << "const unsigned char *__restrict__ bh_args, const unsigned *__restrict__ bh_first, const unsigned bh_items, "
         "const unsigned bh_stride) {\n"
      << "  const unsigned b_ = blockIdx.x;\n"
      << "  unsigned lo_ = 0, hi_ = bh_items;\n"
      << "  while (hi_ - lo_ > 1u) { const unsigned mid_ = (lo_ + hi_) >> 1; if (bh_first[mid_] <= b_) lo_ = mid_; "
         "else hi_ = mid_; }\n"
      << "  const unsigned char *A_ = bh_args + (size_t)lo_ * bh_stride;\n"
      << "  bh_main_(" << unpack << sep << "b_ - bh_first[lo_], bh_first[lo_ + 1] - bh_first[lo_]);\n}\n";
    if (!p.fin_name.empty()) {
        s << "\nextern \"C\" __global__ void __launch_bounds__(" << p.block << ") bh_kernel_fin_batch("
          << "const unsigned char *__restrict__ bh_args, const unsigned bh_stride) {\n"
          << "  const unsigned char *A_ = bh_args + (size_t)blockIdx.x * bh_stride;\n"
          << "  bh_fin_(" << unpack << ");\n}\n";
    }
    return s.str();
}

} // namespace vehip
} // namespace bohrium

// Fused element-wise chains (the FusionGroup kernels).
//
// The reference lowers a FusionGroup on the GPU by generating CUDA source at compile
// time (compiler/nvrtc_builder.cc:91-206), compiling it with NVRTC on first use and
// launching one thread per element over inputs that were first broadcast and copied
// (runtime/ops/nvrtc.cc:90-161).  Here the FusionGroup travels as a small SSA program
// text; the HIP source is generated at run time, when the operand layouts are known,
// so that
//   - broadcast operands are read through their strides (a [1024] vector against a
//     [64,1024,1024] tensor costs 4 KiB of traffic, not 256 MiB),
//   - every full-size operand moves in 128-bit accesses,
//   - the arithmetic is the CPU path's: one IEEE operation per node in topological
//     order, no contraction, tanh/exp as the host C library computes them
//     (faithful_math.h), sigmoid as 1/(1+exp(-x)).
// Compiled code objects are cached by generated source text; loaded kernels by the
// same key (the reference's two-level cache, runtime/ops/nvrtc.cc:41-84, here under a
// mutex).
//
// Program text (one statement per line, '#' starts a comment):
//   chxhip-fusion 1
//   in  <name>:<dtype> ...            dtype: float32 | float16 | float64 | uint8 | int8
//   <name> = <Op> <operand> ...       operands are earlier names or, where noted, literals
//   out <name>:<dtype> ...
// Ops: Identity a | Neg a | Abs a | Floor a | Round a | Add a b | Sub a b | Mul a b | Div a b | Max a b | Min a b
//      Tanh a | Sigmoid a | Exp a | Relu a | Clip a <lo> <hi> | Const <value>
//      QuantizeLinear a <scale> <zero_point> <uint8|int8> [rne]   (float -> 8-bit code)
//      DequantizeLinear q <scale> <zero_point>                    (8-bit code -> float)
// Float literals are decimal or 0x######## (the bit pattern of the float32).
// The arithmetic type of a program is that of its floating-point ports (one type per program, as the reference's
// `typedef ... T`, compiler/nvrtc_builder.cc:118-127): float32; float16, where every node computes in float32 and
// rounds to float16 (what a half-precision operation is); or float64.  The 8-bit ops go with float32 only.
//
// The CUDA C text that the reference's compiler emits for a group (BuildNvrtcProgram, nvrtc_builder.cc:91-206) is
// accepted as well and turned into the same internal program: `typedef half|float|double T;`, the kernel's
// parameters `T* i_<name>` / `T* o_<name>`, one `const T <name> = <expression>;` per node (a + b, a - b, a * b,
// a / b, tanh(a), exp(a), sigmoid(a), a, or a number) and `o_<name>[tid] = <name>;` per output.  Its sigmoid is the
// helper that text defines, tanh(x * 0.5) * 0.5 + 0.5, one rounding per operation.
#include <hip/hiprtc.h>

#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <sstream>
#include <string>
#include <unordered_map>
#include <vector>

#include "chx_internal.h"
#include "conv_mfma.h"

namespace chx {
namespace {

const char* kFaithfulMathText =
#include "faithful_math_text.inc"
        ;

struct Stmt {
    std::string out, op;
    std::vector<std::string> args;
};

struct Port {
    std::string name;
    int32_t dtype;
};

struct Program {
    std::vector<Port> inputs, outputs;
    std::vector<Stmt> stmts;
    int32_t arith = CHX_HIP_FLOAT32;  // type of the floating-point values: float32, float16 or float64
};

bool is_float_dtype(int32_t dt) {
    return dt == CHX_HIP_FLOAT32 || dt == CHX_HIP_FLOAT16 || dt == CHX_HIP_FLOAT64;
}

bool parse_dtype(const std::string& s, int32_t* dt) {
    if (s == "float32") *dt = CHX_HIP_FLOAT32;
    else if (s == "float16") *dt = CHX_HIP_FLOAT16;
    else if (s == "float64") *dt = CHX_HIP_FLOAT64;
    else if (s == "uint8") *dt = CHX_HIP_UINT8;
    else if (s == "int8") *dt = CHX_HIP_INT8;
    else return false;
    return true;
}

std::vector<std::string> split_ws(const std::string& line) {
    std::vector<std::string> out;
    std::istringstream iss(line);
    std::string tok;
    while (iss >> tok) out.push_back(tok);
    return out;
}

int parse_port(const std::string& tok, Port* p) {
    const size_t c = tok.find(':');
    CHX_REQUIRE(c != std::string::npos, "fusion program: expected name:dtype, got '%s'", tok.c_str());
    p->name = tok.substr(0, c);
    CHX_REQUIRE(parse_dtype(tok.substr(c + 1), &p->dtype), "fusion program: unsupported dtype in '%s'", tok.c_str());
    return CHX_HIP_OK;
}

int parse_nvrtc_source(const char* code, Program* prog);

// One floating-point type per program; 8-bit ports only beside float32.
int settle_arithmetic_type(Program* prog) {
    int32_t arith = 0;
    bool any8 = false;
    auto see = [&](const Port& p) -> int {
        if (!is_float_dtype(p.dtype)) {
            any8 = true;
            return CHX_HIP_OK;
        }
        CHX_REQUIRE(arith == 0 || arith == p.dtype, "fusion program: ports of two floating-point types (%s and %s)", dtype_name(arith),
                    dtype_name(p.dtype));
        arith = p.dtype;
        return CHX_HIP_OK;
    };
    for (const Port& p : prog->inputs) CHX_PROPAGATE(see(p));
    for (const Port& p : prog->outputs) CHX_PROPAGATE(see(p));
    prog->arith = arith ? arith : CHX_HIP_FLOAT32;
    CHX_REQUIRE(!any8 || prog->arith == CHX_HIP_FLOAT32, "fusion program: 8-bit ports go with float32 arithmetic, not %s", dtype_name(prog->arith));
    return CHX_HIP_OK;
}

int parse_program(const char* code, Program* prog) {
    CHX_REQUIRE(code != nullptr, "fusion program: null code");
    if (strstr(code, "__global__") != nullptr && strstr(code, "typedef") != nullptr) return parse_nvrtc_source(code, prog);
    std::istringstream iss(code);
    std::string line;
    bool header = false;
    while (std::getline(iss, line)) {
        const size_t hash = line.find('#');
        if (hash != std::string::npos) line.resize(hash);
        std::vector<std::string> t = split_ws(line);
        if (t.empty()) continue;
        if (!header) {
            CHX_REQUIRE(t.size() == 2 && t[0] == "chxhip-fusion" && t[1] == "1",
                        "fusion program: missing 'chxhip-fusion 1' header (is this NVRTC source?)");
            header = true;
            continue;
        }
        if (t[0] == "in" || t[0] == "out") {
            for (size_t i = 1; i < t.size(); ++i) {
                Port p;
                CHX_PROPAGATE(parse_port(t[i], &p));
                (t[0] == "in" ? prog->inputs : prog->outputs).push_back(p);
            }
            continue;
        }
        CHX_REQUIRE(t.size() >= 3 && t[1] == "=", "fusion program: cannot parse statement '%s'", line.c_str());
        Stmt s;
        s.out = t[0];
        s.op = t[2];
        s.args.assign(t.begin() + 3, t.end());
        prog->stmts.push_back(s);
    }
    CHX_REQUIRE(header, "fusion program: empty");
    CHX_REQUIRE(!prog->inputs.empty(), "fusion program: no inputs");
    CHX_REQUIRE(!prog->outputs.empty(), "fusion program: no outputs");
    return settle_arithmetic_type(prog);
}

std::string trimmed(const std::string& s) {
    size_t a = 0, b = s.size();
    while (a < b && isspace((unsigned char)s[a])) ++a;
    while (b > a && isspace((unsigned char)s[b - 1])) --b;
    return s.substr(a, b - a);
}

bool is_identifier(const std::string& s) {
    if (s.empty() || !(isalpha((unsigned char)s[0]) || s[0] == '_')) return false;
    for (char c : s)
        if (!(isalnum((unsigned char)c) || c == '_')) return false;
    return true;
}

// The CUDA C text of BuildNvrtcProgram (compiler/nvrtc_builder.cc:91-206).  Port names are the variables the kernel
// loads its inputs into / stores its outputs from; inputs and outputs keep the order of the kernel's parameters,
// which is the order the op hands its arrays over in (runtime/ops/nvrtc.cc:134-150).
int parse_nvrtc_source(const char* code, Program* prog) {
    std::vector<std::string> lines;
    {
        std::istringstream iss(code);
        std::string line;
        while (std::getline(iss, line)) {
            const size_t c = line.find("//");
            if (c != std::string::npos) line.resize(c);
            line = trimmed(line);
            if (!line.empty()) lines.push_back(line);
        }
    }
    int32_t arith = 0;
    size_t i = 0;
    for (; i < lines.size(); ++i) {
        if (lines[i].compare(0, 8, "typedef ") != 0) continue;
        const std::vector<std::string> t = split_ws(lines[i]);
        CHX_REQUIRE(t.size() == 3 && t[2] == "T;", "fusion source: expected 'typedef <type> T;', got '%s'", lines[i].c_str());
        if (t[1] == "half") arith = CHX_HIP_FLOAT16;
        else if (t[1] == "float") arith = CHX_HIP_FLOAT32;
        else if (t[1] == "double") arith = CHX_HIP_FLOAT64;
        else CHX_FAIL(CHX_HIP_EUNSUPPORTED, "fusion source: element type '%s' (half, float or double expected)", t[1].c_str());
        ++i;
        break;
    }
    CHX_REQUIRE(arith != 0, "fusion source: no 'typedef ... T;'");
    // the sigmoid helper, when the group has one
    if (i < lines.size() && lines[i].compare(0, 10, "__device__") == 0) {
        CHX_REQUIRE(lines[i].find("T sigmoid(T x)") != std::string::npos, "fusion source: unknown helper '%s'", lines[i].c_str());
        bool body = false;
        for (++i; i < lines.size() && lines[i] != "}"; ++i)
            if (lines[i].find("tanh(x * half) * half + half") != std::string::npos) body = true;
        CHX_REQUIRE(body && i < lines.size(), "fusion source: the sigmoid helper is not tanh(x * half) * half + half");
        ++i;
    }
    // extern "C" __global__ / void fusionN(size_t n, T* i_a, ..., T* o_y) {
    std::string sig;
    for (; i < lines.size(); ++i) {
        if (lines[i].compare(0, 5, "void ") == 0) {
            sig = lines[i++];
            break;
        }
        CHX_REQUIRE(lines[i].find("__global__") != std::string::npos, "fusion source: unexpected line '%s' in front of the kernel", lines[i].c_str());
    }
    const size_t lp = sig.find('('), rp = sig.rfind(')');
    CHX_REQUIRE(!sig.empty() && lp != std::string::npos && rp != std::string::npos && rp > lp, "fusion source: no kernel signature");
    std::vector<std::string> in_params, out_params;
    {
        std::istringstream ps(sig.substr(lp + 1, rp - lp - 1));
        std::string param;
        bool first = true;
        while (std::getline(ps, param, ',')) {
            param = trimmed(param);
            if (first) {
                CHX_REQUIRE(param == "size_t n", "fusion source: the first kernel parameter is '%s', not 'size_t n'", param.c_str());
                first = false;
                continue;
            }
            CHX_REQUIRE(param.compare(0, 3, "T* ") == 0, "fusion source: kernel parameter '%s' is not a T*", param.c_str());
            const std::string name = trimmed(param.substr(3));
            if (name.compare(0, 2, "i_") == 0) in_params.push_back(name);
            else if (name.compare(0, 2, "o_") == 0) out_params.push_back(name);
            else CHX_FAIL(CHX_HIP_EINVAL, "fusion source: kernel parameter '%s' is neither an input (i_) nor an output (o_)", name.c_str());
        }
    }
    CHX_REQUIRE(!in_params.empty() && !out_params.empty(), "fusion source: the kernel needs inputs and outputs");
    std::vector<std::string> in_var(in_params.size()), out_var(out_params.size());
    for (; i < lines.size(); ++i) {
        std::string line = lines[i];
        if (line == "}") break;
        if (line.compare(0, 11, "size_t tid ") == 0 || line.compare(0, 13, "if (tid >= n)") == 0) continue;
        CHX_REQUIRE(line.back() == ';', "fusion source: statement without ';': '%s'", line.c_str());
        line.resize(line.size() - 1);
        const size_t eq = line.find(" = ");
        CHX_REQUIRE(eq != std::string::npos, "fusion source: cannot parse '%s'", lines[i].c_str());
        const std::string lhs = trimmed(line.substr(0, eq)), rhs = trimmed(line.substr(eq + 3));
        if (lhs.compare(0, 8, "const T ") != 0) {
            // o_<name>[tid] = <name>
            const size_t br = lhs.find("[tid]");
            CHX_REQUIRE(br != std::string::npos && br + 5 == lhs.size(), "fusion source: cannot parse '%s'", lines[i].c_str());
            const std::string param = lhs.substr(0, br);
            size_t k = 0;
            while (k < out_params.size() && out_params[k] != param) ++k;
            CHX_REQUIRE(k < out_params.size() && is_identifier(rhs), "fusion source: '%s' stores to something that is not an output", lines[i].c_str());
            out_var[k] = rhs;
            continue;
        }
        const std::string out = trimmed(lhs.substr(8));
        CHX_REQUIRE(is_identifier(out), "fusion source: '%s' does not define a variable", lines[i].c_str());
        const size_t br = rhs.find("[tid]");
        if (br != std::string::npos) {
            // <name> = i_<name>[tid]
            const std::string param = rhs.substr(0, br);
            size_t k = 0;
            while (k < in_params.size() && in_params[k] != param) ++k;
            CHX_REQUIRE(k < in_params.size() && br + 5 == rhs.size(), "fusion source: '%s' loads from something that is not an input", lines[i].c_str());
            CHX_REQUIRE(in_var[k].empty(), "fusion source: input '%s' is loaded twice", param.c_str());
            in_var[k] = out;
            continue;
        }
        Stmt st;
        st.out = out;
        const std::vector<std::string> t = split_ws(rhs);
        const size_t call = rhs.find('(');
        if (t.size() == 3 && t[1].size() == 1 && strchr("+-*/", t[1][0]) && is_identifier(t[0]) && is_identifier(t[2])) {
            st.op = t[1] == "+" ? "Add" : t[1] == "-" ? "Sub" : t[1] == "*" ? "Mul" : "Div";
            st.args = {t[0], t[2]};
            prog->stmts.push_back(st);
        } else if (call != std::string::npos && rhs.back() == ')') {
            const std::string fn = rhs.substr(0, call), arg = trimmed(rhs.substr(call + 1, rhs.size() - call - 2));
            CHX_REQUIRE(is_identifier(arg), "fusion source: cannot parse the argument of '%s'", lines[i].c_str());
            if (fn == "tanh" || fn == "exp") {
                st.op = fn == "tanh" ? "Tanh" : "Exp";
                st.args = {arg};
                prog->stmts.push_back(st);
            } else if (fn == "sigmoid") {
                // the helper of this text, operation by operation: tanh(x * half) * half + half with half = 0.5
                const std::string h = out + "__half", a = out + "__arg", th = out + "__tanh", m = out + "__scaled";
                prog->stmts.push_back(Stmt{h, "Const", {"0.5"}});
                prog->stmts.push_back(Stmt{a, "Mul", {arg, h}});
                prog->stmts.push_back(Stmt{th, "Tanh", {a}});
                prog->stmts.push_back(Stmt{m, "Mul", {th, h}});
                prog->stmts.push_back(Stmt{out, "Add", {m, h}});
            } else {
                CHX_FAIL(CHX_HIP_EUNSUPPORTED, "fusion source: function '%s' is not one the reference's builder emits", fn.c_str());
            }
        } else if (t.size() == 1 && is_identifier(t[0])) {
            st.op = "Identity";
            st.args = {t[0]};
            prog->stmts.push_back(st);
        } else {
            char* end = nullptr;
            (void)strtod(rhs.c_str(), &end);
            CHX_REQUIRE(end && *end == 0 && end != rhs.c_str(), "fusion source: cannot parse the expression of '%s'", lines[i].c_str());
            st.op = "Const";
            st.args = {rhs};
            prog->stmts.push_back(st);
        }
    }
    CHX_REQUIRE(i < lines.size(), "fusion source: the kernel body does not end");
    for (size_t k = 0; k < in_params.size(); ++k) {
        // an input that the kernel never loads keeps its place in the argument list
        prog->inputs.push_back(Port{in_var[k].empty() ? in_params[k] + "__unused" : in_var[k], arith});
    }
    for (size_t k = 0; k < out_params.size(); ++k) {
        CHX_REQUIRE(!out_var[k].empty(), "fusion source: output '%s' is never stored", out_params[k].c_str());
        prog->outputs.push_back(Port{out_var[k], arith});
    }
    return settle_arithmetic_type(prog);
}

std::string ident(const std::string& s) {
    std::string o = "v_";
    for (char c : s) o += (isalnum((unsigned char)c) ? c : '_');
    return o;
}

int float_value(const std::string& tok, float* value);

// A literal of the program's arithmetic type, as source text that reproduces its bits: float32 and float64 by their
// bit patterns; float16 as the float32 that equals the literal rounded to float16.
int float_literal(const std::string& tok, std::string* out, int32_t arith = CHX_HIP_FLOAT32) {
    char buf[80];
    if (arith == CHX_HIP_FLOAT64 || arith == CHX_HIP_FLOAT16) {
        double d;
        if (tok.size() == 10 && tok[0] == '0' && (tok[1] == 'x' || tok[1] == 'X')) {
            float f;
            CHX_PROPAGATE(float_value(tok, &f));
            d = f;
        } else {
            char* end = nullptr;
            d = strtod(tok.c_str(), &end);
            CHX_REQUIRE(end && *end == 0 && end != tok.c_str(), "fusion program: bad float literal '%s'", tok.c_str());
        }
        if (arith == CHX_HIP_FLOAT64) {
            uint64_t bits;
            memcpy(&bits, &d, 8);
            snprintf(buf, sizeof(buf), "__builtin_bit_cast(double, 0x%016llxull)", (unsigned long long)bits);
        } else {
            const float f = (float)(_Float16)d;
            uint32_t bits;
            memcpy(&bits, &f, 4);
            snprintf(buf, sizeof(buf), "__builtin_bit_cast(float, 0x%08xu)", bits);
        }
        *out = buf;
        return CHX_HIP_OK;
    }
    float f;
    CHX_PROPAGATE(float_value(tok, &f));
    uint32_t bits;
    memcpy(&bits, &f, 4);
    snprintf(buf, sizeof(buf), "__builtin_bit_cast(float, 0x%08xu)", bits);
    *out = buf;
    return CHX_HIP_OK;
}

int float_value(const std::string& tok, float* value) {
    float f;
    if (tok.size() == 10 && tok[0] == '0' && (tok[1] == 'x' || tok[1] == 'X')) {
        char* end = nullptr;
        const unsigned long u = strtoul(tok.c_str(), &end, 16);
        CHX_REQUIRE(end && *end == 0, "fusion program: bad float bit pattern '%s'", tok.c_str());
        const uint32_t u32 = (uint32_t)u;
        memcpy(&f, &u32, 4);
    } else {
        char* end = nullptr;
        const double d = strtod(tok.c_str(), &end);
        CHX_REQUIRE(end && *end == 0 && end != tok.c_str(), "fusion program: bad float literal '%s'", tok.c_str());
        f = (float)d;
    }
    *value = f;
    return CHX_HIP_OK;
}

// tanh for a float16 argument whose result is rounded to float16: an odd rational function of degree 7 over 6 (minimax in
// the relative error, 2^-25, up to 4.53, beyond which the result rounds to 1).  It is not the C library's float32 tanh, but
// rounded to float16 it is for every one of the 65536 arguments (a test compares them all).  15 instructions instead of
// about 60, which bound the float16 chains: two operands of [8, 333, 1001] and two of [1001] through Mul, Add, Tanh, Sigmoid,
// Mul, Add and Relu 13.4 us, with this and the sigmoid below 7.5 (profiled).  NaN is left to the second evaluation.
const char* const kTanhOfF16 = R"(
__device__ __forceinline__ float chx_tanh_of_f16(float x, bool& rare) {
  rare = rare || x != x;
  const float v = __builtin_fminf(__builtin_fabsf(x), 0x1.21eb86p+2f), s = v * v;
  float p = __builtin_fmaf(0x1.6ed3dep-18f, s, 0x1.4ea1ecp-9f);
  p = __builtin_fmaf(p, s, 0x1.01e116p-3f);
  p = __builtin_fmaf(p, s, 1.0f);
  float q = __builtin_fmaf(0x1.6df1f6p-13f, s, 0x1.6d6cb6p-6f);
  q = __builtin_fmaf(q, s, 0x1.d645cep-2f);
  q = __builtin_fmaf(q, s, 1.0f);
  return __builtin_copysignf((v * p) * __builtin_amdgcn_rcpf(q), x);
}
)";

// Emits the per-element device function:  elem(in..., &out...).
// Value kinds: 'f' floating-point value, 'q' 8-bit code held in an int.  A floating-point value is held as TY:
// float for float32 and for float16 programs (in the latter every node's result goes through R(), the rounding
// to float16, so that it is a float16 value at all times), double for float64 programs.
int emit_elem(const Program& prog, bool use_fma, std::ostringstream& os, bool* uses_exp_table) {
    std::map<std::string, char> kind;
    const bool f64 = prog.arith == CHX_HIP_FLOAT64, f16 = prog.arith == CHX_HIP_FLOAT16;
    const std::string TY = f64 ? "double" : "float";
    const std::string decl = "  const " + TY + " ";
    const char* R0 = f16 ? "chx_round_f16(" : "(";
    const std::string zero = f64 ? "0.0" : "0.0f";
    // kFast: Exp and Sigmoid without their rare cases (arguments beyond +-88, quotients near the denormal range);
    // `rare` comes back set when an element met one, and the caller evaluates it again with kFast = false
    os << "template <bool kFast>\n__device__ __forceinline__ void elem(";
    bool first = true;
    for (const Port& p : prog.inputs) {
        CHX_REQUIRE(!kind.count(p.name), "fusion program: duplicate input '%s'", p.name.c_str());
        kind[p.name] = is_float_dtype(p.dtype) ? 'f' : 'q';
        os << (first ? "" : ", ") << (is_float_dtype(p.dtype) ? "const " + TY + " " : std::string("const int ")) << ident(p.name);
        first = false;
    }
    for (size_t i = 0; i < prog.outputs.size(); ++i)
        os << ", " << (is_float_dtype(prog.outputs[i].dtype) ? TY + "& " : std::string("int& ")) << "o_" << i;
    os << ", bool& rare) {\n";
    const char* fma = use_fma ? "true" : "false";
    for (const Stmt& s : prog.stmts) {
        CHX_REQUIRE(!kind.count(s.out), "fusion program: '%s' assigned twice", s.out.c_str());
        auto need = [&](size_t n) -> int {
            CHX_REQUIRE(s.args.size() == n, "fusion program: %s takes %zu operands, got %zu", s.op.c_str(), n,
                        s.args.size());
            return CHX_HIP_OK;
        };
        auto val = [&](size_t i, char k, std::string* out) -> int {
            auto it = kind.find(s.args[i]);
            CHX_REQUIRE(it != kind.end(), "fusion program: '%s' used before definition in '%s'", s.args[i].c_str(),
                        s.op.c_str());
            CHX_REQUIRE(it->second == k, "fusion program: operand '%s' of %s has the wrong kind (%s expected)",
                        s.args[i].c_str(), s.op.c_str(), k == 'f' ? "float" : "8-bit code");
            *out = ident(s.args[i]);
            return CHX_HIP_OK;
        };
        const std::string o = ident(s.out);
        std::string a, b, l0, l1;
        char out_kind = 'f';
        static const std::map<std::string, const char*> binops = {{"Add", "+"}, {"Sub", "-"}, {"Mul", "*"}, {"Div", "/"}};
        if (binops.count(s.op)) {
            CHX_PROPAGATE(need(2));
            CHX_PROPAGATE(val(0, 'f', &a));
            CHX_PROPAGATE(val(1, 'f', &b));
            os << decl << o << " = " << R0 << a << " " << binops.at(s.op) << " " << b << ");\n";
        } else if (s.op == "Max" || s.op == "Min") {
            CHX_PROPAGATE(need(2));
            CHX_PROPAGATE(val(0, 'f', &a));
            CHX_PROPAGATE(val(1, 'f', &b));
            if (s.op == "Max")
                os << decl << o << " = " << a << " < " << b << " ? " << b << " : " << a << ";\n";
            else
                os << decl << o << " = " << b << " < " << a << " ? " << b << " : " << a << ";\n";
        } else if (s.op == "Identity") {
            CHX_PROPAGATE(need(1));
            auto it = kind.find(s.args[0]);
            CHX_REQUIRE(it != kind.end(), "fusion program: '%s' used before definition", s.args[0].c_str());
            out_kind = it->second;
            os << "  const " << (out_kind == 'f' ? TY + " " : std::string("int ")) << o << " = " << ident(s.args[0]) << ";\n";
        } else if (s.op == "Neg") {
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(val(0, 'f', &a));
            os << decl << o << " = -" << a << ";\n";
        } else if (s.op == "Abs") {
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(val(0, 'f', &a));
            os << decl << o << " = " << (f64 ? "__builtin_fabs(" : "__builtin_fabsf(") << a << ");\n";
        } else if (s.op == "Floor") {
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(val(0, 'f', &a));
            os << decl << o << " = " << (f64 ? "__builtin_floor(" : "__builtin_floorf(") << a << ");\n";
        } else if (s.op == "Round") {
            // to the nearest integer, ties to even (RoundOp, runtime/ops/quantize.cc:148-151)
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(val(0, 'f', &a));
            os << decl << o << " = " << (f64 ? "__builtin_rint(" : "__builtin_rintf(") << a << ");\n";
        } else if (s.op == "Tanh") {
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(val(0, 'f', &a));
            if (f64) os << decl << o << " = ::tanh(" << a << ");\n";
            else if (f16) os << decl << o << " = chx_round_f16(kFast ? chx_tanh_of_f16(" << a << ", rare) : chx_fm::tanhf_faithful(" << a << "));\n";
            else os << decl << o << " = " << R0 << "chx_fm::tanhf_faithful(" << a << "));\n";
        } else if (s.op == "Exp") {
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(val(0, 'f', &a));
            if (f64) {
                os << decl << o << " = ::exp(" << a << ");\n";
            } else {
                os << decl << o << " = " << R0 << "kFast ? chx_fm::expf_unless_rare<" << fma << ">(" << a << ", rare) : chx_fm::expf_faithful<"
                   << fma << ">(" << a << "));\n";
                *uses_exp_table = true;
            }
        } else if (s.op == "Sigmoid") {
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(val(0, 'f', &a));
            if (f64) {
                // 1 / (1 + exp(-x)), as the CPU path spells it
                os << decl << o << " = 1.0 / (1.0 + ::exp(-" << a << "));\n";
            } else if (f16) {
                // the same, every operation a float16 operation.  Which exponential and which reciprocal give the
                // float16 results of the C library's exp and of the division is a question of 65536 arguments, and a
                // test asks it for all of them: the device's own instructions do.
                os << decl << o << "_e = chx_round_f16(__builtin_amdgcn_exp2f(-0x1.715476p+0f * " << a << "));\n";
                os << decl << o << "_d = chx_round_f16(1.0f + " << o << "_e);\n";
                os << decl << o << " = chx_round_f16(__builtin_amdgcn_rcpf(" << o << "_d));\n";
            } else {
                os << decl << o << " = kFast ? chx_fm::sigmoid_unless_rare<" << fma << ">(" << a
                   << ", rare) : chx_fm::sigmoid_faithful<" << fma << ">(" << a << ");\n";
                *uses_exp_table = true;
            }
        } else if (s.op == "Relu") {
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(val(0, 'f', &a));
            os << decl << o << " = " << a << " < " << zero << " ? " << zero << " : " << a << ";\n";
        } else if (s.op == "Clip") {
            CHX_PROPAGATE(need(3));
            CHX_PROPAGATE(val(0, 'f', &a));
            CHX_PROPAGATE(float_literal(s.args[1], &l0, prog.arith));
            CHX_PROPAGATE(float_literal(s.args[2], &l1, prog.arith));
            os << decl << o << "_lo = " << a << " < " << l0 << " ? " << l0 << " : " << a << ";\n";
            os << decl << o << " = " << o << "_lo < " << l1 << " ? " << o << "_lo : " << l1 << ";\n";
        } else if (s.op == "Const") {
            CHX_PROPAGATE(need(1));
            CHX_PROPAGATE(float_literal(s.args[0], &l0, prog.arith));
            os << decl << o << " = " << l0 << ";\n";
        } else if (s.op == "QuantizeLinear") {
            CHX_REQUIRE(s.args.size() == 4 || (s.args.size() == 5 && s.args[4] == "rne"),
                        "fusion program: QuantizeLinear a scale zero_point dtype [rne]");
            CHX_REQUIRE(prog.arith == CHX_HIP_FLOAT32, "fusion program: QuantizeLinear inside a %s program", dtype_name(prog.arith));
            CHX_PROPAGATE(val(0, 'f', &a));
            CHX_PROPAGATE(float_literal(s.args[1], &l0));
            char* end = nullptr;
            const long zp = strtol(s.args[2].c_str(), &end, 10);
            CHX_REQUIRE(end && *end == 0, "fusion program: bad zero point '%s'", s.args[2].c_str());
            int32_t dt;
            CHX_REQUIRE(parse_dtype(s.args[3], &dt) && is_q8(dt), "fusion program: QuantizeLinear dtype must be uint8 or int8");
            const bool i8 = dt == CHX_HIP_INT8;
            CHX_REQUIRE(zp >= (i8 ? -128 : 0) && zp <= (i8 ? 127 : 255), "fusion program: zero point %ld out of range", zp);
            const char* lo = i8 ? "-128.0f" : "0.0f";
            const char* hi = i8 ? "127.0f" : "255.0f";
            // quantize_array, runtime/ops/quantize.cc:29-34.  The correctly rounded quotient comes from
            // three multiply-adds with the rounded reciprocal (q0 within an ulp, exact residual, one
            // correction) instead of the ten-instruction IEEE division.  The dividend is first limited
            // to +-2^40 * scale: beyond that both the true quotient and the limited one are far outside
            // the 8-bit range and saturate alike, and no intermediate can overflow.
            float scale_value;
            CHX_PROPAGATE(float_value(s.args[1], &scale_value));
            if (scale_value >= 0x1p-60f && scale_value <= 0x1p60f) {
                const float inv = 1.0f / scale_value, big = 0x1p40f * scale_value;
                uint32_t inv_bits, big_bits;
                memcpy(&inv_bits, &inv, 4);
                memcpy(&big_bits, &big, 4);
                char inv_lit[64], big_lit[64];
                snprintf(inv_lit, sizeof(inv_lit), "__builtin_bit_cast(float, 0x%08xu)", inv_bits);
                snprintf(big_lit, sizeof(big_lit), "__builtin_bit_cast(float, 0x%08xu)", big_bits);
                os << "  const float " << o << "_v = __builtin_amdgcn_fmed3f(" << a << ", -" << big_lit << ", " << big_lit << ");\n";
                os << "  const float " << o << "_q0 = " << o << "_v * " << inv_lit << ";\n";
                os << "  const float " << o << "_r = __builtin_fmaf(-" << o << "_q0, " << l0 << ", " << o << "_v);\n";
                os << "  float " << o << "_s = __builtin_fmaf(" << o << "_r, " << inv_lit << ", " << o << "_q0);\n";
            } else {
                os << "  float " << o << "_s = " << a << " / " << l0 << ";\n";
            }
            // the clamp is one median instruction: the same function as Maximum(lo, Minimum(s, hi))
            // for every value that is not a NaN
            if (s.args.size() == 5) {
                os << "  " << o << "_s = __builtin_rintf(" << o << "_s) + " << zp << ".0f;\n";
                os << "  " << o << "_s = __builtin_amdgcn_fmed3f(" << o << "_s, " << lo << ", " << hi << ");\n";
            } else {
                os << "  " << o << "_s = " << o << "_s + " << zp << ".0f;\n";
                os << "  " << o << "_s = __builtin_amdgcn_fmed3f(" << o << "_s, " << lo << ", " << hi << ");\n";
                os << "  " << o << "_s = " << o << "_s + 0.5f;\n";
            }
            os << "  const int " << o << " = (int)" << o << "_s;\n";
            out_kind = 'q';
        } else if (s.op == "DequantizeLinear") {
            CHX_PROPAGATE(need(3));
            CHX_REQUIRE(prog.arith == CHX_HIP_FLOAT32, "fusion program: DequantizeLinear inside a %s program", dtype_name(prog.arith));
            CHX_PROPAGATE(val(0, 'q', &a));
            CHX_PROPAGATE(float_literal(s.args[1], &l0));
            char* end = nullptr;
            const long zp = strtol(s.args[2].c_str(), &end, 10);
            CHX_REQUIRE(end && *end == 0, "fusion program: bad zero point '%s'", s.args[2].c_str());
            // dequantize_array, runtime/ops/quantize.cc:37-44
            os << "  const float " << o << "_f = (float)" << a << " - " << zp << ".0f;\n";
            os << "  const float " << o << " = " << o << "_f * " << l0 << ";\n";
        } else {
            CHX_FAIL(CHX_HIP_EUNSUPPORTED, "fusion program: op '%s' is not in the fusable set", s.op.c_str());
        }
        kind[s.out] = out_kind;
    }
    for (size_t i = 0; i < prog.outputs.size(); ++i) {
        auto it = kind.find(prog.outputs[i].name);
        CHX_REQUIRE(it != kind.end(), "fusion program: output '%s' is never defined", prog.outputs[i].name.c_str());
        const char want = is_float_dtype(prog.outputs[i].dtype) ? 'f' : 'q';
        CHX_REQUIRE(it->second == want, "fusion program: output '%s' is declared %s but computed as %s",
                    prog.outputs[i].name.c_str(), dtype_name(prog.outputs[i].dtype), it->second == 'f' ? "float" : "code");
        os << "  o_" << i << " = " << ident(prog.outputs[i].name) << ";\n";
    }
    os << "}\n";
    return CHX_HIP_OK;
}

enum Mode : char { kFull = 'F', kScalar = 'S', kPeriodic = 'P' };

const char* ctype_of(int32_t dt) {
    return dt == CHX_HIP_FLOAT32 ? "float" : dt == CHX_HIP_FLOAT16 ? "_Float16" : dt == CHX_HIP_FLOAT64 ? "double"
           : dt == CHX_HIP_INT8 ? "signed char" : "unsigned char";
}

// How the general kernel addresses an operand:
//   kFlat    dense in the order of the result: the flat index      kOne       one element
//   kRow     innermost stride 1      kRepeat  innermost stride 0   kStrided   any strides
enum Addressing : char { kFlat = 'F', kOne = 'S', kRow = 'C', kRepeat = 'Z', kStrided = 'X' };

// What the general kernel is compiled for, beside the program.
struct GeneralForm {
    std::string modes;  // Addressing, per input
    int vec = 1;        // elements per thread: 16 bytes of the widest operand (the program's); 1: rows shorter than that
    int axes = 3;       // collapsed axes: up to three (nearly all calls), or kAxes
    bool wide = false;  // 2^31 elements or more in the result or in the reach of an operand, or negative strides: 64-bit indices
};
constexpr int kAxes = CHX_HIP_MAX_NDIM;

// The general kernel: any strides, types and alignments.  A thread computes `vec` neighbouring elements of the result.
// Where they lie in one row of the innermost axis (nearly always) each operand is one access of 16 bytes at whatever
// alignment (kFlat, kRow), one element (kOne, kRepeat), or `vec` strided ones; a run that crosses the end of a row is
// read element by element from two positions.  (Of rows shorter than that a thread computes one element: every run would
// cross.)  Divisions by the extents are multiplications with their reciprocals.
// Axes are collapsed ones, the innermost first; those past the last have extent 1, so that the rank of a call is no part of
// its kernel (a compilation takes 0.3 s of the first call).  The kernel before, one for each rank and with
// each operand converted beside its load, took 16.1 us for the chain below in float32 on [16, 333, 1001], this one 16.5; which
// of the two differences costs it was not measured apart.  The operands' addressing is: as an argument it made the chain
// below 17 % slower in float32 rows of 1001 (scalar loads behind each branch), which one kernel for all calls would cost.
// Chain of two operands of [8, 333, 1001] and two of [1001] through Mul, Add, Tanh, Sigmoid, Mul, Add and Relu in float16:
// 15.2 us with one element per thread and 64-bit divisions, 8.6 with each operand converted beside its load, 6.9 with all
// loads in flight first.
void emit_general(const Program& prog, const std::string& name, const GeneralForm& g, const std::string& VT, std::ostringstream& os) {
    const size_t nin = prog.inputs.size(), nout = prog.outputs.size();
    const int V = g.vec;
    auto placed = [&](size_t i) { return g.modes[i] != kFlat && g.modes[i] != kOne; };  // by the position in the result
    bool any_placed = false;
    for (size_t i = 0; i < nin; ++i) any_placed = any_placed || placed(i);
    const char* idx = g.wide ? "unsigned long long" : "unsigned int";
    auto value_type = [&](const Port& p) { return is_float_dtype(p.dtype) ? VT : std::string("int"); };
    auto vec_type = [&](int32_t dt) {
        return std::string("V") + (dt == CHX_HIP_FLOAT32 ? "f" : dt == CHX_HIP_FLOAT16 ? "h" : dt == CHX_HIP_FLOAT64 ? "d" : "b");
    };
    os << "typedef " << idx << " gidx;\ntypedef " << (g.wide ? "long long" : "unsigned int") << " sidx;  // (wide: positions before the operand's first element)\n";
    os << "struct GenDesc { unsigned int mul[" << kAxes << "], shift[" << kAxes << "]; long long shape[" << kAxes << "]; long long istr[" << nin << "][" << kAxes
       << "]; };\n";
    os << "typedef float Vf __attribute__((ext_vector_type(" << V << "), aligned(4)));\n";
    os << "typedef _Float16 Vh __attribute__((ext_vector_type(" << V << "), aligned(2)));\n";
    os << "typedef double Vd __attribute__((ext_vector_type(" << V << "), aligned(8)));\n";
    os << "typedef unsigned int Vb __attribute__((ext_vector_type(" << (V < 4 ? 1 : V / 4) << "), aligned(1)));\n";
    os << "__device__ __forceinline__ gidx gdiv(gidx r, const GenDesc& d, int a) {\n";
    if (g.wide) os << "  return r / (gidx)d.shape[a];\n}\n";
    else os << "  return (__umulhi(r, d.mul[a]) + r) >> d.shift[a];\n}\n";
    // the position along each axis of flat position r, and an operand's element there
    os << "__device__ __forceinline__ void place(gidx r, const GenDesc& d, gidx (&at)[" << g.axes << "]) {\n";
    os << "#pragma unroll\n  for (int a = 0; a < " << g.axes - 1 << "; ++a) {\n    const gidx q = gdiv(r, d, a);\n    at[a] = r - q * (gidx)d.shape[a];\n    r = q;\n  }\n";
    os << "  at[" << g.axes - 1 << "] = r;\n}\n";
    os << "__device__ __forceinline__ gidx offset(const long long (&stride)[" << kAxes << "], const gidx (&at)[" << g.axes << "]) {\n  gidx off = 0;\n";
    os << "#pragma unroll\n  for (int a = 0; a < " << g.axes << "; ++a) off += at[a] * (gidx)stride[a];\n  return off;\n}\n";

    os << "extern \"C\" __global__ __launch_bounds__(256) void " << name << "_gen(unsigned long long total, unsigned long long first";
    for (size_t i = 0; i < nin; ++i) os << ", const " << ctype_of(prog.inputs[i].dtype) << "* __restrict__ i" << i;
    for (size_t i = 0; i < nout; ++i) os << ", " << ctype_of(prog.outputs[i].dtype) << "* __restrict__ o" << i;
    os << ", GenDesc d) {\n";
    os << "  const gidx n = (gidx)total, base = (gidx)first + ((gidx)blockIdx.x * 256u + threadIdx.x) * " << V << "u;\n";
    os << "  if (base >= n) return;\n";
    os << "  const int cnt = n - base < " << V << "u ? (int)(n - base) : " << V << ";\n";
    // What an operand's elements are as loaded: a vector, and converted behind the last of the loads only (a conversion
    // beside its load waits for it, one operand after the other).  8-bit codes arrive as words.
    auto element = [&](size_t i, const std::string& e, const std::string& at) {  // statement: element e of operand i
        const std::string k = std::to_string(i);
        if (is_float_dtype(prog.inputs[i].dtype)) return "r" + k + "[" + e + "] = i" + k + "[(sidx)(" + at + ")]; ";
        return "r" + k + "[" + e + " / 4] |= (unsigned int)(unsigned char)i" + k + "[(sidx)(" + at + ")] << (8 * (" + e + " % 4)); ";
    };
    for (size_t i = 0; i < nin; ++i) os << "  " << vec_type(prog.inputs[i].dtype) << " r" << i << " = 0;\n";
    os << "  const bool whole = cnt == " << V << ";\n";
    auto whole_access = [&](const Port& p) { return is_float_dtype(p.dtype) || V >= 4; };  // (codes come in words)
    auto elements = [&](size_t i, const std::string& condition, const std::string& at) {
        os << "  {\n#pragma unroll\n    for (int e = 0; e < " << V << "; ++e) " << condition << "{ " << element(i, "e", at) << "}\n  }\n";
    };
    // (dense operands before the others' addresses are known)
    for (size_t i = 0; i < nin; ++i) {
        const std::string k = std::to_string(i), vt = vec_type(prog.inputs[i].dtype);
        if (g.modes[i] == kOne) elements(i, "", "0");
        if (g.modes[i] != kFlat) continue;
        if (whole_access(prog.inputs[i])) os << "  if (whole) r" << k << " = __builtin_nontemporal_load((const " << vt << "*)(i" << k << " + base));\n  else\n";
        elements(i, "if (e < cnt) ", "base + e");
    }
    if (any_placed) {
        os << "  gidx at[" << g.axes << "];\n  place(base, d, at);\n";
        if (V > 1) os << "  const gidx left = (gidx)d.shape[0] - at[0];\n  if (whole && left >= " << V << "u) {\n";
        for (size_t i = 0; i < nin; ++i) {
            if (!placed(i)) continue;
            const std::string k = std::to_string(i), vt = vec_type(prog.inputs[i].dtype);
            os << "  { const gidx off = offset(d.istr[" << k << "], at);\n";
            if (g.modes[i] == kRow && whole_access(prog.inputs[i])) os << "    r" << k << " = *(const " << vt << "*)(i" << k << " + (sidx)off);\n";
            else elements(i, "", g.modes[i] == kRepeat || V == 1 ? "off" : "off + e * (gidx)d.istr[" + k + "][0]");
            os << "  }\n";
        }
        if (V > 1) {
            // (`there` is where the elements behind the end of the row would begin if they had all been on the next one)
            os << "  } else {\n    gidx next[" << g.axes << "];\n    place(base + left < n ? base + left : base, d, next);\n";
            for (size_t i = 0; i < nin; ++i) {
                if (!placed(i)) continue;
                const std::string k = std::to_string(i), step = g.modes[i] == kRow ? "1u" : g.modes[i] == kRepeat ? "0u" : "(gidx)d.istr[" + k + "][0]";
                os << "  { const gidx here = offset(d.istr[" << k << "], at), there = offset(d.istr[" << k << "], next) - left * " << step << ";\n";
                elements(i, "if (e < cnt) ", "((gidx)e < left ? here : there) + e * " + step);
                os << "  }\n";
            }
            os << "  }\n";
        }
    }
    for (size_t i = 0; i < nin; ++i) {
        const std::string k = std::to_string(i);
        const int32_t dt = prog.inputs[i].dtype;
        os << "  " << value_type(prog.inputs[i]) << " x" << k << "[" << V << "];\n";
        if (is_float_dtype(dt)) {
            os << "  for (int e = 0; e < " << V << "; ++e) x" << k << "[e] = (" << VT << ")r" << k << "[e];\n";
        } else {
            for (int e = 0; e < V; ++e)
                os << "  x" << k << "[" << e << "] = (int)" << (dt == CHX_HIP_INT8 ? "(signed char)" : "") << "((r" << k << "[" << e / 4 << "] >> " << 8 * (e % 4) << ") & 0xffu);\n";
        }
    }
    for (size_t i = 0; i < nout; ++i) os << "  " << value_type(prog.outputs[i]) << " y" << i << "[" << V << "];\n";
    os << "  bool rare = false;\n";
    for (int fast = 1; fast >= 0; --fast) {
        if (!fast) os << "  if (__builtin_expect(FM_ANY_LANE(rare), 0)) {\n";
        os << "#pragma unroll\n  for (int e = 0; e < " << V << "; ++e) elem<" << (fast ? "true" : "false") << ">(";
        for (size_t i = 0; i < nin; ++i) os << (i ? ", " : "") << "x" << i << "[e]";
        for (size_t i = 0; i < nout; ++i) os << ", y" << i << "[e]";
        os << ", rare);\n";
        if (!fast) os << "  }\n";
    }
    os << "  if (cnt == " << V << ") {\n";
    for (size_t i = 0; i < nout; ++i) {
        const int32_t dt = prog.outputs[i].dtype;
        if (!whole_access(prog.outputs[i])) {
            os << "    for (int e = 0; e < " << V << "; ++e) o" << i << "[base + e] = (" << ctype_of(dt) << ")y" << i << "[e];\n";
            continue;
        }
        if (is_float_dtype(dt)) {
            os << "    { " << vec_type(dt) << " t; for (int e = 0; e < " << V << "; ++e) t[e] = (" << ctype_of(dt) << ")y" << i << "[e];\n";
        } else {
            os << "    { Vb t;\n";
            for (int w = 0; w < V / 4; ++w) {
                os << "      t[" << w << "] = ";
                for (int k = 0; k < 4; ++k) os << (k ? " | " : "") << "(((unsigned int)y" << i << "[" << 4 * w + k << "] & 0xffu) << " << 8 * k << ")";
                os << ";\n";
            }
        }
        os << "      __builtin_nontemporal_store(t, (" << vec_type(dt) << "*)(o" << i << " + base)); }\n";
    }
    os << "  } else {\n#pragma unroll\n    for (int e = 0; e < " << V << "; ++e) if (e < cnt) {\n";
    for (size_t i = 0; i < nout; ++i) os << "      o" << i << "[base + e] = (" << ctype_of(prog.outputs[i].dtype) << ")y" << i << "[e];\n";
    os << "    }\n  }\n}\n";
}

// What both kernels of a program begin with: the per-element function and what it needs.  The kernels are sources of their
// own, compiled when a call first takes one of them:
//   <name>_vec : V elements per thread through 128-bit accesses; operands are full
//                (same flat index as the output), scalar, or periodic (index modulo a
//                period that is a multiple of V).  float32 programs.
//   <name>_gen : emit_general.
int emit_common(const Program& prog, bool use_fma, std::ostringstream& os) {
    os << "#pragma clang fp contract(off)\n";
    os << "#define FM_FN __device__ __forceinline__\n";
    os << "#define FM_TABLE_QUALIFIER static __device__ const\n";
    os << "#define FM_DEVICE_DIV 1\n";
    os << "#define FM_ANY_LANE(c) (__builtin_amdgcn_ballot_w64(c) != 0ull)\n";
    std::ostringstream body;
    bool uses_table = false;
    CHX_PROPAGATE(emit_elem(prog, use_fma, body, &uses_table));
    os << kFaithfulMathText << "\n";
    os << "__device__ __forceinline__ float chx_round_f16(float x) { return (float)(_Float16)x; }\n";
    if (prog.arith == CHX_HIP_FLOAT16) os << kTanhOfF16;
    os << "typedef float v4f __attribute__((ext_vector_type(4)));\n";
    os << "typedef unsigned int v4u __attribute__((ext_vector_type(4)));\n";
    os << "namespace {\n" << body.str() << "}\n";
    return CHX_HIP_OK;
}

const char* value_type_of(const Program& prog) {  // what elem() takes and gives
    return prog.arith == CHX_HIP_FLOAT64 ? "double" : "float";
}

int general_source(const Program& prog, const std::string& name, const GeneralForm& form, bool use_fma, std::string* out) {
    std::ostringstream os;
    CHX_PROPAGATE(emit_common(prog, use_fma, os));
    emit_general(prog, name, form, value_type_of(prog), os);
    *out = os.str();
    return CHX_HIP_OK;
}

int vector_source(
        const Program& prog, const std::string& name, const std::string& modes, const std::vector<uint32_t>& periods, int vec, bool use_fma, std::string* out) {
    std::ostringstream os;
    CHX_PROPAGATE(emit_common(prog, use_fma, os));
    const size_t nin = prog.inputs.size(), nout = prog.outputs.size();
    // `vec` elements per lane and step: 4 when any full-size operand is float32 (float32
    // moves as one 128-bit access per lane, 8-bit codes as one 32-bit access), 16 when all
    // of them are 8-bit (one 128-bit access each).  kSteps steps per thread at a stride of
    // one block keep every access instruction of a wavefront on one contiguous span.
    const int steps = 2;
    os << "extern \"C\" __global__ __launch_bounds__(256) void " << name << "_vec(unsigned int n_vec";
    for (size_t i = 0; i < nin; ++i) os << ", const " << ctype_of(prog.inputs[i].dtype) << "* __restrict__ i" << i;
    for (size_t i = 0; i < nout; ++i) os << ", " << ctype_of(prog.outputs[i].dtype) << "* __restrict__ o" << i;
    os << ") {\n";
    os << "  const unsigned int vid0 = blockIdx.x * " << 256 * steps << "u + threadIdx.x;\n";
    os << "#pragma unroll\n  for (int st = 0; st < " << steps << "; ++st) {\n";
    os << "  const unsigned int vid = vid0 + st * 256u;\n";
    os << "  if (vid < n_vec) {\n";
    os << "  const unsigned int base = vid * " << vec << "u;  // fewer than 2^31 elements\n";
    for (size_t i = 0; i < nin; ++i) {
        const bool f32 = prog.inputs[i].dtype == CHX_HIP_FLOAT32;
        const bool sgn = prog.inputs[i].dtype == CHX_HIP_INT8;
        os << "  " << (f32 ? "float" : "int") << " x" << i << "[" << vec << "];\n";
        if (modes[i] == kScalar) {
            os << "  for (int e = 0; e < " << vec << "; ++e) x" << i << "[e] = i" << i << "[0];\n";
            continue;
        }
        std::string idx = "base";
        if (modes[i] == kPeriodic) idx = "(base % " + std::to_string(periods[i]) + "u)";
        const bool nt = modes[i] == kFull;
        const char* ld0 = nt ? "__builtin_nontemporal_load(" : "*(";
        if (f32) {
            os << "  { const v4f* src = (const v4f*)(i" << i << " + " << idx << ");\n";
            for (int j = 0; j < vec / 4; ++j) {
                os << "    const v4f t" << j << " = " << ld0 << "src + " << j << ");\n";
                for (int k = 0; k < 4; ++k) os << "    x" << i << "[" << (j * 4 + k) << "] = t" << j << "[" << k << "];\n";
            }
            os << "  }\n";
        } else {
            const int words = vec / 4;
            os << "  { unsigned int t[" << words << "];\n";
            if (words == 4) {
                os << "    const v4u tv = " << ld0 << "(const v4u*)(i" << i << " + " << idx << "));\n";
                os << "    t[0] = tv[0]; t[1] = tv[1]; t[2] = tv[2]; t[3] = tv[3];\n";
            } else {
                os << "    t[0] = " << ld0 << "(const unsigned int*)(i" << i << " + " << idx << "));\n";
            }
            for (int e = 0; e < vec; ++e) {
                os << "    x" << i << "[" << e << "] = ";
                if (sgn)
                    os << "(int)(signed char)((t[" << (e / 4) << "] >> " << (8 * (e % 4)) << ") & 0xffu);\n";
                else
                    os << "(int)((t[" << (e / 4) << "] >> " << (8 * (e % 4)) << ") & 0xffu);\n";
            }
            os << "  }\n";
        }
    }
    for (size_t i = 0; i < nout; ++i)
        os << "  " << (prog.outputs[i].dtype == CHX_HIP_FLOAT32 ? "float" : "int") << " y" << i << "[" << vec << "];\n";
    // all elements of the step without the rare cases first, one wavefront-wide test, and again in full if any lane
    // met one: a branch per element costs more than the rare cases' few instructions
    os << "  bool rare = false;\n";
    for (int fast = 1; fast >= 0; --fast) {
        if (!fast) os << "  if (__builtin_expect(FM_ANY_LANE(rare), 0)) {\n";
        os << "#pragma unroll\n  for (int e = 0; e < " << vec << "; ++e) elem<" << (fast ? "true" : "false") << ">(";
        for (size_t i = 0; i < nin; ++i) os << (i ? ", " : "") << "x" << i << "[e]";
        for (size_t i = 0; i < nout; ++i) os << ", y" << i << "[e]";
        os << ", rare);\n";
        if (!fast) os << "  }\n";
    }
    for (size_t i = 0; i < nout; ++i) {
        if (prog.outputs[i].dtype == CHX_HIP_FLOAT32) {
            os << "  { v4f* dst = (v4f*)(o" << i << " + base);\n";
            for (int j = 0; j < vec / 4; ++j) {
                os << "    v4f t" << j << ";\n";
                for (int k = 0; k < 4; ++k) os << "    t" << j << "[" << k << "] = y" << i << "[" << (j * 4 + k) << "];\n";
                os << "    __builtin_nontemporal_store(t" << j << ", dst + " << j << ");\n";
            }
            os << "  }\n";
        } else {
            const int words = vec / 4;
            os << "  { unsigned int t[" << words << "];\n";
            for (int w = 0; w < words; ++w) {
                os << "    t[" << w << "] = ";
                for (int k = 0; k < 4; ++k)
                    os << (k ? " | " : "") << "(((unsigned int)y" << i << "[" << (w * 4 + k) << "] & 0xffu) << " << (8 * k) << ")";
                os << ";\n";
            }
            if (words == 4) {
                os << "    v4u tv; tv[0] = t[0]; tv[1] = t[1]; tv[2] = t[2]; tv[3] = t[3];\n";
                os << "    __builtin_nontemporal_store(tv, (v4u*)(o" << i << " + base));\n  }\n";
            } else {
                os << "    __builtin_nontemporal_store(t[0], (unsigned int*)(o" << i << " + base));\n  }\n";
            }
        }
    }
    os << "  }\n  }\n}\n";
    *out = os.str();
    return CHX_HIP_OK;
}

struct CompiledKernel {
    std::vector<char> code;
    hipModule_t module = nullptr;  // loaded lazily, per process (one GPU)
    hipFunction_t function = nullptr;
};

std::mutex g_cache_mutex;
std::map<std::string, std::shared_ptr<CompiledKernel>> g_cache;  // key: generated source

int compile_source(const std::string& src, const std::string& name, std::vector<char>* code) {
    hiprtcProgram p;
    if (hiprtcCreateProgram(&p, src.c_str(), (name + ".hip").c_str(), 0, nullptr, nullptr) != HIPRTC_SUCCESS)
        CHX_FAIL(CHX_HIP_ERUNTIME, "hiprtcCreateProgram failed for %s", name.c_str());
    const char* opts[] = {"--offload-arch=gfx950", "-O3", "-ffp-contract=off", "-Xclang", "-target-feature",
                          "-Xclang", "-packed-fp32-ops"};
    const hiprtcResult r = hiprtcCompileProgram(p, (int)(sizeof(opts) / sizeof(opts[0])), opts);
    if (r != HIPRTC_SUCCESS) {
        size_t ls = 0;
        hiprtcGetProgramLogSize(p, &ls);
        std::string log(ls, '\0');
        if (ls) hiprtcGetProgramLog(p, &log[0]);
        hiprtcDestroyProgram(&p);
        CHX_FAIL(CHX_HIP_ECOMPILE, "hiprtc could not compile %s: %s\n%s", name.c_str(), hiprtcGetErrorString(r),
                 log.c_str());
    }
    size_t cs = 0;
    hiprtcGetCodeSize(p, &cs);
    code->resize(cs);
    hiprtcGetCode(p, code->data());
    hiprtcDestroyProgram(&p);
    return CHX_HIP_OK;
}

struct Plan {
    std::string modes;             // per input
    bool vector_ok = false;
    int vec = 4;
    int64_t n = 0;
    int ndim = 0;
    int64_t shape[CHX_HIP_MAX_NDIM];
    std::vector<std::vector<int64_t>> istr;  // element strides per input, per collapsed axis
    std::vector<uint32_t> periods;
    GeneralForm gen;
};

int make_plan(
        const Program& prog, const chx_hip_tensor* const* inputs, int32_t n_inputs, chx_hip_tensor* const* outputs,
        int32_t n_outputs, Plan* plan) {
    CHX_REQUIRE((size_t)n_inputs == prog.inputs.size(), "fusion: program declares %zu inputs, %d given",
                prog.inputs.size(), n_inputs);
    CHX_REQUIRE((size_t)n_outputs == prog.outputs.size(), "fusion: program declares %zu outputs, %d given",
                prog.outputs.size(), n_outputs);
    int nd = 0;
    for (int i = 0; i < n_inputs; ++i) {
        CHX_PROPAGATE(check_tensor(inputs[i], "fusion input"));
        CHX_REQUIRE(inputs[i]->dtype == prog.inputs[i].dtype, "fusion: input %d is %s, program says %s", i,
                    dtype_name(inputs[i]->dtype), dtype_name(prog.inputs[i].dtype));
        nd = inputs[i]->ndim > nd ? inputs[i]->ndim : nd;
    }
    // BroadcastShapes over all inputs, runtime/ops/nvrtc.cc:100-104
    int64_t shape[CHX_HIP_MAX_NDIM];
    for (int a = 0; a < nd; ++a) shape[a] = 1;
    for (int i = 0; i < n_inputs; ++i) {
        const chx_hip_tensor& t = *inputs[i];
        for (int a = 0; a < t.ndim; ++a) {
            const int oa = nd - t.ndim + a;
            if (t.shape[a] == 1) continue;
            CHX_REQUIRE(shape[oa] == 1 || shape[oa] == t.shape[a], "fusion: input %d does not broadcast (axis %d: %lld vs %lld)",
                        i, a, (long long)t.shape[a], (long long)shape[oa]);
            shape[oa] = t.shape[a];
        }
    }
    int64_t n = 1;
    for (int a = 0; a < nd; ++a) n *= shape[a];
    plan->n = n;
    for (int i = 0; i < n_outputs; ++i) {
        CHX_PROPAGATE(check_tensor(outputs[i], "fusion output"));
        const chx_hip_tensor& t = *outputs[i];
        CHX_REQUIRE(t.dtype == prog.outputs[i].dtype, "fusion: output %d is %s, program says %s", i, dtype_name(t.dtype),
                    dtype_name(prog.outputs[i].dtype));
        CHX_REQUIRE(t.ndim == nd, "fusion: output %d has ndim %d, the broadcast result has %d", i, t.ndim, nd);
        for (int a = 0; a < nd; ++a)
            CHX_REQUIRE(t.shape[a] == shape[a], "fusion: output %d has extent %lld on axis %d, expected %lld", i,
                        (long long)t.shape[a], a, (long long)shape[a]);
    }
    // Iteration order: axes of output 0 by decreasing stride; every output must be dense in
    // that order with the same element strides.
    int order[CHX_HIP_MAX_NDIM];
    int na = 0;
    const chx_hip_tensor& o0 = *outputs[0];
    const int64_t es0 = dtype_size(o0.dtype);
    for (int a = 0; a < nd; ++a)
        if (shape[a] != 1) order[na++] = a;
    for (int i = 0; i < na; ++i)
        for (int j = i + 1; j < na; ++j)
            if (o0.strides[order[j]] > o0.strides[order[i]]) {
                const int t = order[i];
                order[i] = order[j];
                order[j] = t;
            }
    {
        int64_t expect = 1;
        for (int i = na - 1; i >= 0; --i) {
            for (int k = 0; k < n_outputs; ++k) {
                const int64_t es = dtype_size(outputs[k]->dtype);
                CHX_REQUIRE(outputs[k]->strides[order[i]] == expect * es,
                            "fusion: output %d is not dense, or outputs differ in layout", k);
            }
            expect *= shape[order[i]];
        }
        (void)es0;
    }
    // Element strides of every input along the ordered axes (0 where it broadcasts).
    std::vector<std::vector<int64_t>> istr(n_inputs, std::vector<int64_t>(na, 0));
    for (int i = 0; i < n_inputs; ++i) {
        const chx_hip_tensor& t = *inputs[i];
        const int64_t es = dtype_size(t.dtype);
        for (int k = 0; k < na; ++k) {
            const int ia = order[k] - (nd - t.ndim);
            if (ia < 0 || t.shape[ia] == 1) continue;
            CHX_REQUIRE(t.strides[ia] % es == 0, "fusion: input %d has a stride that is not a multiple of its element size", i);
            istr[i][k] = t.strides[ia] / es;
        }
    }
    // Collapse neighbouring axes that every operand walks contiguously.
    std::vector<int64_t> cshape;
    std::vector<std::vector<int64_t>> cstr(n_inputs);
    for (int k = 0; k < na; ++k) {
        const int64_t ext = shape[order[k]];
        bool merge = !cshape.empty();
        if (merge)
            for (int i = 0; i < n_inputs; ++i)
                if (cstr[i].back() != istr[i][k] * ext) merge = false;
        if (merge) {
            cshape.back() *= ext;
            for (int i = 0; i < n_inputs; ++i) cstr[i].back() = istr[i][k];
        } else {
            cshape.push_back(ext);
            for (int i = 0; i < n_inputs; ++i) cstr[i].push_back(istr[i][k]);
        }
    }
    plan->ndim = (int)cshape.size();
    for (int a = 0; a < plan->ndim; ++a) plan->shape[a] = cshape[a];
    plan->istr = cstr;

    bool any32 = false;  // (an 8-bit operand beside a float32 one moves 4 bytes per access)
    for (const Port& p : prog.inputs) any32 = any32 || p.dtype == CHX_HIP_FLOAT32;
    for (const Port& p : prog.outputs) any32 = any32 || p.dtype == CHX_HIP_FLOAT32;
    plan->vec = any32 ? 4 : 16;
    plan->modes.assign(n_inputs, kFull);
    plan->periods.assign(n_inputs, 0);
    bool ok = n < (int64_t(1) << 31);  // CHECK_GT(1 << 31, size), runtime/ops/nvrtc.cc:127
    // dense inner strides of the output in collapsed axes
    std::vector<int64_t> dense(plan->ndim, 1);
    for (int a = plan->ndim - 2; a >= 0; --a) dense[a] = dense[a + 1] * cshape[a + 1];
    for (int i = 0; i < n_inputs; ++i) {
        bool all_zero = true, full = true;
        for (int a = 0; a < plan->ndim; ++a) {
            if (cstr[i][a] != 0) all_zero = false;
            if (cstr[i][a] != dense[a]) full = false;
        }
        const int64_t es = dtype_size(inputs[i]->dtype);
        if (plan->ndim == 0 || all_zero) {
            plan->modes[i] = kScalar;
        } else if (full) {
            plan->modes[i] = kFull;
            if (!aligned(inputs[i]->data, 16)) ok = false;
        } else {
            // periodic: zero strides on the outer axes, dense strides on the inner ones
            int a = 0;
            while (a < plan->ndim && cstr[i][a] == 0) ++a;
            bool inner_dense = a > 0;
            for (int b = a; b < plan->ndim; ++b)
                if (cstr[i][b] != dense[b]) inner_dense = false;
            const int64_t period = a > 0 ? dense[a - 1] : 0;
            if (inner_dense && period % plan->vec == 0 && period < (int64_t(1) << 31) && aligned(inputs[i]->data, 16)) {
                plan->modes[i] = kPeriodic;
                plan->periods[i] = (uint32_t)period;
            } else {
                ok = false;
            }
        }
        (void)es;
    }
    for (int k = 0; k < n_outputs; ++k)
        if (!aligned(outputs[k]->data, 16)) ok = false;
    plan->vector_ok = ok && n >= plan->vec && prog.arith == CHX_HIP_FLOAT32;
    GeneralForm& g = plan->gen;
    g.vec = any32 ? 4 : prog.arith == CHX_HIP_FLOAT64 ? 2 : prog.arith == CHX_HIP_FLOAT16 ? 8 : 16;
    g.wide = n >= (int64_t(1) << 31) - 4096;  // (indices run past the last element by less than a work-group's share)
    g.axes = plan->ndim > 3 ? kAxes : 3;
    g.modes.assign(n_inputs, kStrided);
    bool placed = false;
    for (int i = 0; i < n_inputs; ++i) {
        bool flat = true, one = true;
        int64_t reach = 0;
        for (int a = 0; a < plan->ndim; ++a) {
            flat = flat && cstr[i][a] == dense[a];
            one = one && cstr[i][a] == 0;
            reach += (cshape[a] - 1) * cstr[i][a];
            if (cstr[i][a] < 0) g.wide = true;
        }
        if (reach >= (int64_t(1) << 31) - 4096) g.wide = true;
        if (plan->ndim == 0 || one) g.modes[i] = kOne;
        else if (flat) g.modes[i] = kFlat;
        else if (cstr[i][plan->ndim - 1] == 1) g.modes[i] = kRow;
        else if (cstr[i][plan->ndim - 1] == 0) g.modes[i] = kRepeat;
        placed = placed || (g.modes[i] != kOne && g.modes[i] != kFlat);
    }
    if (placed && cshape[plan->ndim - 1] < g.vec) {
        g.vec = 1;
        for (char& m : g.modes)
            if (m == kRow || m == kRepeat) m = kStrided;  // (the same for one element)
    }
    if (!placed) g.axes = 3;  // (none is looked at)
    return CHX_HIP_OK;
}

struct ArgPacker {
    std::vector<char> buf;
    template <typename T>
    void push(const T& v) {
        const size_t a = alignof(T);
        const size_t off = (buf.size() + a - 1) / a * a;
        buf.resize(off + sizeof(T));
        memcpy(buf.data() + off, &v, sizeof(T));
    }
    void push_bytes(const void* p, size_t n, size_t a) {
        const size_t off = (buf.size() + a - 1) / a * a;
        buf.resize(off + n);
        memcpy(buf.data() + off, p, n);
    }
};

// Whether a call takes the vector kernel.  (Elements beyond whole vectors would be a launch of their own.)
bool takes_vector(const Plan& plan) {
    return plan.vector_ok && plan.n % plan.vec == 0;
}

int prepare(
        const char* code, int32_t fusion_id, const chx_hip_tensor* const* inputs, int32_t n_inputs,
        chx_hip_tensor* const* outputs, int32_t n_outputs, Program* prog, Plan* plan, std::string* name) {
    CHX_REQUIRE(inputs != nullptr && n_inputs > 0, "fusion: no inputs");  // CHECK(!inputs.empty()), nvrtc.cc:93
    CHX_REQUIRE(outputs != nullptr && n_outputs > 0, "fusion: no outputs");
    CHX_PROPAGATE(parse_program(code, prog));
    CHX_PROPAGATE(make_plan(*prog, inputs, n_inputs, outputs, n_outputs, plan));
    *name = "fusion" + std::to_string(fusion_id < 0 ? 0 : fusion_id);
    return CHX_HIP_OK;
}

int source_of(const Program& prog, const Plan& plan, const std::string& name, bool vector, std::string* src) {
    if (vector) return vector_source(prog, name, plan.modes, plan.periods, plan.vec, host_libm_uses_fma(), src);
    return general_source(prog, name, plan.gen, host_libm_uses_fma(), src);
}

int get_compiled(const std::string& src, const std::string& name, std::shared_ptr<CompiledKernel>* out) {
    std::lock_guard<std::mutex> lock(g_cache_mutex);
    auto it = g_cache.find(src);
    if (it != g_cache.end()) {
        *out = it->second;
        return CHX_HIP_OK;
    }
    auto ck = std::make_shared<CompiledKernel>();
    CHX_PROPAGATE(compile_source(src, name, &ck->code));
    g_cache.emplace(src, ck);
    *out = ck;
    return CHX_HIP_OK;
}

int load_kernel(CompiledKernel* ck, const std::string& function) {
    std::lock_guard<std::mutex> lock(g_cache_mutex);
    if (ck->module) return CHX_HIP_OK;
    hipModule_t m;
    CHX_HIP_CALL(hipModuleLoadData(&m, ck->code.data()));
    CHX_HIP_CALL(hipModuleGetFunction(&ck->function, m, function.c_str()));
    ck->module = m;
    return CHX_HIP_OK;
}

int launch(hipFunction_t f, unsigned grid, ArgPacker& args, hipStream_t s) {
    size_t size = args.buf.size();
    void* extra[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, args.buf.data(), HIP_LAUNCH_PARAM_BUFFER_SIZE, &size,
                     HIP_LAUNCH_PARAM_END};
    CHX_HIP_CALL(hipModuleLaunchKernel(f, grid, 1, 1, 256, 1, 1, 0, s, nullptr, extra));
    return CHX_HIP_OK;
}

}  // namespace
}  // namespace chx

using namespace chx;

extern "C" int chx_hip_elementwise_output_dtypes(const char* code, int32_t* dtypes, int32_t capacity, int32_t* count) {
    CHX_REQUIRE(count != nullptr && (dtypes != nullptr || capacity == 0), "elementwise_output_dtypes: null output");
    CHX_REQUIRE(code != nullptr, "fusion program: null code");
    static std::mutex mutex;
    static std::unordered_map<std::string, std::vector<int32_t>> known;  // asked on every call of a group
    std::vector<int32_t> found;
    {
        std::lock_guard<std::mutex> lock(mutex);
        auto it = known.find(code);
        if (it != known.end()) found = it->second;
    }
    if (found.empty()) {
        Program prog;
        CHX_PROPAGATE(parse_program(code, &prog));
        for (const Port& p : prog.outputs) found.push_back(p.dtype);
        std::lock_guard<std::mutex> lock(mutex);
        if (known.size() >= 4096) known.clear();
        known.emplace(code, found);
    }
    *count = (int32_t)found.size();
    for (int32_t i = 0; i < *count && i < capacity; ++i) dtypes[i] = found[(size_t)i];
    return CHX_HIP_OK;
}

extern "C" int chx_hip_elementwise_source(
        const char* code, int32_t fusion_id, const chx_hip_tensor* const* inputs, int32_t n_inputs,
        chx_hip_tensor* const* outputs, int32_t n_outputs, int32_t compile, char* buffer, size_t buffer_size,
        size_t* needed) {
    Program prog;
    Plan plan;
    std::string name, text;
    CHX_PROPAGATE(prepare(code, fusion_id, inputs, n_inputs, outputs, n_outputs, &prog, &plan, &name));
    // both kernels where the operands are the vector kernel's (a count that is not whole vectors takes the other)
    for (const bool vector : {true, false}) {
        if (vector && !plan.vector_ok) continue;
        std::string src;
        CHX_PROPAGATE(source_of(prog, plan, name, vector, &src));
        if (compile && vector == takes_vector(plan)) {
            std::shared_ptr<CompiledKernel> ck;
            CHX_PROPAGATE(get_compiled(src, name, &ck));
        }
        text += "// modes=" + (plan.vector_ok ? plan.modes + " vector" : std::string((size_t)n_inputs, kFull) + " general") + "\n" + src;
    }
    if (needed) *needed = text.size() + 1;
    if (buffer && buffer_size) {
        const size_t n = text.size() < buffer_size - 1 ? text.size() : buffer_size - 1;
        memcpy(buffer, text.data(), n);
        buffer[n] = 0;
    }
    return CHX_HIP_OK;
}

namespace chx {
namespace {

// What a call needs beyond its pointers, kept per (program text, operand layouts): parsing the text, planning and writing
// out the kernel's source to look the compiled kernel up took 35 us of host time per call.
struct PreparedCall {
    std::shared_ptr<CompiledKernel> kernel;
    bool vector = false;
    int vec = 0;
    int64_t n = 0;
    int64_t blocks = 0;
    std::vector<char> desc;  // GenDesc of the general kernel
};
constexpr size_t kMostPrepared = 4096;  // (a few hundred bytes each; all are dropped when there are more)
std::mutex g_prepared_mutex;
std::unordered_map<std::string, std::shared_ptr<const PreparedCall>> g_prepared;

void append_layout(const chx_hip_tensor* t, std::string* key) {
    if (!t || t->ndim < 0 || t->ndim > CHX_HIP_MAX_NDIM) return;  // refused when the call is prepared
    const int32_t head[3] = {t->dtype, t->ndim, aligned(t->data, 16) ? 1 : 0};
    key->append(reinterpret_cast<const char*>(head), sizeof(head));
    key->append(reinterpret_cast<const char*>(t->shape), sizeof(int64_t) * (size_t)t->ndim);
    key->append(reinterpret_cast<const char*>(t->strides), sizeof(int64_t) * (size_t)t->ndim);
}

int prepare_call(
        const char* code, int32_t fusion_id, const chx_hip_tensor* const* inputs, int32_t n_inputs, chx_hip_tensor* const* outputs,
        int32_t n_outputs, PreparedCall* call) {
    Program prog;
    Plan plan;
    std::string name, src;
    CHX_PROPAGATE(prepare(code, fusion_id, inputs, n_inputs, outputs, n_outputs, &prog, &plan, &name));
    call->n = plan.n;
    if (plan.n == 0) return CHX_HIP_OK;
    CHX_REQUIRE(plan.n < (int64_t(1) << 39), "fusion: %lld elements is beyond what the general kernel covers", (long long)plan.n);
    call->vector = takes_vector(plan);
    call->vec = plan.vec;
    CHX_PROPAGATE(source_of(prog, plan, name, call->vector, &src));
    CHX_PROPAGATE(get_compiled(src, name, &call->kernel));
    CHX_PROPAGATE(load_kernel(call->kernel.get(), name + (call->vector ? "_vec" : "_gen")));
    if (call->vector) {
        call->blocks = (plan.n / plan.vec + 511) / 512;
        return CHX_HIP_OK;
    }
    call->vec = plan.gen.vec;
    call->blocks = (plan.n + 256 * plan.gen.vec - 1) / (256 * plan.gen.vec);
    // GenDesc { unsigned mul[kAxes], shift[kAxes]; long long shape[kAxes], istr[nin][kAxes]; }
    const size_t M = kAxes;
    call->desc.assign(2 * M * 4 + M * 8 + (size_t)n_inputs * M * 8, 0);
    uint32_t* mul = reinterpret_cast<uint32_t*>(call->desc.data());
    int64_t* shape = reinterpret_cast<int64_t*>(call->desc.data() + 2 * M * 4);
    for (size_t k = 0; k < M; ++k) {
        const bool there = k < (size_t)plan.ndim;
        const size_t a = (size_t)plan.ndim - 1 - k;  // (the kernel's first axis is the innermost)
        shape[k] = there ? plan.shape[a] : 1;
        if (!plan.gen.wide) magic_divisor((uint32_t)shape[k], &mul[k], &mul[M + k]);
        for (size_t i = 0; there && i < (size_t)n_inputs; ++i) shape[M * (1 + i) + k] = plan.istr[i][a];
    }
    return CHX_HIP_OK;
}

}  // namespace
}  // namespace chx

extern "C" int chx_hip_elementwise(
        const char* code, int32_t fusion_id, const chx_hip_tensor* const* inputs, int32_t n_inputs,
        chx_hip_tensor* const* outputs, int32_t n_outputs, void* stream) {
    CHX_REQUIRE(code != nullptr, "fusion program: null code");
    CHX_REQUIRE(inputs != nullptr && n_inputs > 0, "fusion: no inputs");  // CHECK(!inputs.empty()), nvrtc.cc:93
    CHX_REQUIRE(outputs != nullptr && n_outputs > 0, "fusion: no outputs");
    for (int i = 0; i < n_inputs; ++i) CHX_PROPAGATE(check_tensor(inputs[i], "fusion input"));
    for (int i = 0; i < n_outputs; ++i) CHX_PROPAGATE(check_tensor(outputs[i], "fusion output"));
    std::string key(code);
    const int32_t ids[3] = {fusion_id, n_inputs, n_outputs};
    key.append(1, '\0').append(reinterpret_cast<const char*>(ids), sizeof(ids));
    for (int i = 0; i < n_inputs; ++i) append_layout(inputs[i], &key);
    for (int i = 0; i < n_outputs; ++i) append_layout(outputs[i], &key);
    std::shared_ptr<const PreparedCall> call;
    {
        std::lock_guard<std::mutex> lock(g_prepared_mutex);
        auto it = g_prepared.find(key);
        if (it != g_prepared.end()) call = it->second;
    }
    if (!call) {
        auto made = std::make_shared<PreparedCall>();
        CHX_PROPAGATE(prepare_call(code, fusion_id, inputs, n_inputs, outputs, n_outputs, made.get()));
        call = made;
        std::lock_guard<std::mutex> lock(g_prepared_mutex);
        if (g_prepared.size() >= kMostPrepared) g_prepared.clear();
        g_prepared.emplace(std::move(key), call);
    }
    if (call->n == 0) return CHX_HIP_OK;
    // a launch has fewer than 2^32 threads (fewer than 2^31 elements, and one launch, for the vector kernel)
    constexpr int64_t kMostBlocks = int64_t(1) << 23;
    for (int64_t block = 0; block < call->blocks; block += kMostBlocks) {
        ArgPacker a;
        if (call->vector) {
            a.push((uint32_t)(call->n / call->vec));
        } else {
            a.push((unsigned long long)call->n);
            a.push((unsigned long long)(block * 256 * call->vec));
        }
        for (int i = 0; i < n_inputs; ++i) a.push(inputs[i]->data);
        for (int i = 0; i < n_outputs; ++i) a.push(outputs[i]->data);
        if (!call->vector) a.push_bytes(call->desc.data(), call->desc.size(), 8);
        const int64_t left = call->blocks - block;
        CHX_PROPAGATE(launch(call->kernel->function, (unsigned)(left < kMostBlocks ? left : kMostBlocks), a, as_stream(stream)));
    }
    return CHX_HIP_OK;
}

extern "C" int chx_hip_elementwise_match_residual_add(const char* code, int32_t* matches, chx_hip_residual_group* group) {
    using namespace chx;
    CHX_REQUIRE(matches != nullptr && group != nullptr, "match_residual_add: null output");
    *matches = 0;
    memset(group, 0, sizeof(*group));
    Program prog;
    CHX_PROPAGATE(parse_program(code, &prog));
    if (prog.inputs.size() != 2 || prog.outputs.size() != 1) return CHX_HIP_OK;
    if (!is_q8(prog.inputs[0].dtype) || !is_q8(prog.inputs[1].dtype) || !is_q8(prog.outputs[0].dtype)) return CHX_HIP_OK;
    if (prog.stmts.size() != 4 && prog.stmts.size() != 5) return CHX_HIP_OK;
    const bool relu = prog.stmts.size() == 5;
    std::string dq_name[2];
    for (int i = 0; i < 2; ++i) {
        // one DequantizeLinear per input, among the first two statements
        const Stmt* found = nullptr;
        for (int j = 0; j < 2; ++j)
            if (prog.stmts[j].op == "DequantizeLinear" && prog.stmts[j].args.size() == 3 && prog.stmts[j].args[0] == prog.inputs[i].name)
                found = found ? nullptr : &prog.stmts[j];
        if (!found || prog.inputs[0].name == prog.inputs[1].name) return CHX_HIP_OK;
        CHX_PROPAGATE(float_value(found->args[1], &group->in_scale[i]));
        char* end = nullptr;
        const long zp = strtol(found->args[2].c_str(), &end, 10);
        if (!end || *end != 0) return CHX_HIP_OK;
        group->in_zero_point[i] = (int32_t)zp;
        group->in_dtype[i] = prog.inputs[i].dtype;
        dq_name[i] = found->out;
    }
    const Stmt& add = prog.stmts[2];
    if (add.op != "Add" || add.args.size() != 2) return CHX_HIP_OK;
    if (!((add.args[0] == dq_name[0] && add.args[1] == dq_name[1]) || (add.args[0] == dq_name[1] && add.args[1] == dq_name[0])))
        return CHX_HIP_OK;
    std::string last = add.out;
    if (relu) {
        const Stmt& r = prog.stmts[3];
        if (r.op != "Relu" || r.args.size() != 1 || r.args[0] != last) return CHX_HIP_OK;
        last = r.out;
    }
    const Stmt& q = prog.stmts.back();
    if (q.op != "QuantizeLinear" || q.args.size() != 4 || q.args[0] != last || q.out != prog.outputs[0].name) return CHX_HIP_OK;
    CHX_PROPAGATE(float_value(q.args[1], &group->out_scale));
    char* end = nullptr;
    const long zp = strtol(q.args[2].c_str(), &end, 10);
    int32_t qdt = 0;
    if (!end || *end != 0 || !parse_dtype(q.args[3], &qdt) || qdt != prog.outputs[0].dtype) return CHX_HIP_OK;
    group->out_zero_point = (int32_t)zp;
    group->out_dtype = qdt;
    group->relu = relu ? 1 : 0;
    *matches = 1;
    return CHX_HIP_OK;
}

#include "chxvm.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <fstream>
#include <iomanip>
#include <map>
#include <sstream>

#include <set>

#include <iostream>

#include "chainerx_util.h"
#include "chrome_tracing.h"

namespace chainer_compiler {
namespace runtime {

namespace {

// DequantizeLinear(a), DequantizeLinear(b), MatMul, QuantizeLinear as one instruction: the
// quantized matrix product with the reference's float semantics (chx_hip_qlinear_matmul).
class FusedQLinearMatMulOp : public ChxVMOp {
public:
    FusedQLinearMatMulOp(const ChxVMInstructionProto& quantize, const ChxVMInstructionProto& dq_a,
                         const ChxVMInstructionProto& dq_b)
        : ChxVMOp(quantize),
          a_(dq_a.inputs[0].array), a_scale_(dq_a.inputs[1].scalar), a_zp_(dq_a.inputs[2].scalar),
          b_(dq_b.inputs[0].array), b_scale_(dq_b.inputs[1].scalar), b_zp_(dq_b.inputs[2].scalar),
          y_scale_(quantize.inputs[1].scalar), y_zp_(quantize.inputs[2].scalar), y_(quantize.outputs[0]) {
    }

    void Run(ChxVMState* st) override {
        if (st->trace_level()) std::cerr << "QLinearMatMul(fused) $" << a_ << " $" << b_ << " -> $" << y_ << std::endl;
        const chainerx::Array a = st->GetArray(a_), b = st->GetArray(b_);
        auto zp_of = [&](int slot) -> StrictScalar {
            absl::optional<StrictScalar> z = st->GetOptionalScalar(slot);
            return z.has_value() ? *z : StrictScalar(chainerx::Dtype::kUInt8, chainerx::Scalar(0u), false);
        };
        const StrictScalar az = zp_of(a_zp_), bz = zp_of(b_zp_), yz = zp_of(y_zp_);
        CHECK_LE(2, a.ndim());
        CHECK_EQ(a.ndim(), b.ndim());
        chainerx::Shape shape(a.shape().begin(), a.shape().end() - 1);
        shape.push_back(b.shape()[b.ndim() - 1]);
        chainerx::Array y = chainerx::Empty(shape, yz.dtype());
        chx_hip_tensor at = a.hip(), bt = b.hip(), yt = y.hip();
        CHXVM_HIP_CALL(chx_hip_qlinear_matmul(
                &at, static_cast<float>(st->GetScalar(a_scale_)), static_cast<int32_t>(static_cast<int64_t>(az)), &bt,
                static_cast<float>(st->GetScalar(b_scale_)), static_cast<int32_t>(static_cast<int64_t>(bz)),
                static_cast<float>(st->GetScalar(y_scale_)), static_cast<int32_t>(static_cast<int64_t>(yz)),
                nullptr, CHX_HIP_ROUND_REFERENCE, &yt, chainerx::CurrentStream()));
        st->SetArray(y_, y);
    }

private:
    int a_, a_scale_, a_zp_, b_, b_scale_, b_zp_, y_scale_, y_zp_, y_;
};

// Instructions of a program, with their places in it.
typedef std::vector<std::pair<int, ChxVMOp*>> ChxVMSteps;

// Several instructions as one launch.  It stands where the last of them stood; what its kernel does not take runs as the program
// wrote it.  Operands that are constants of the program are laid out when it is loaded.
class GroupOp : public ChxVMOp {
public:
    // steps: the instructions that this one replaces and the Free's of their operands between them, in the program's order
    GroupOp(const ChxVMInstructionProto& last, ChxVMSteps steps, std::vector<int> freed) : ChxVMOp(last), steps_(std::move(steps)), freed_(std::move(freed)) {
    }

    void Run(ChxVMState* st) override {
        if (RunAsOne(st)) {
            for (int slot : freed_) st->FreeVar(slot);
            return;
        }
        RunSteps(st);
    }

protected:
    // false: nothing has been written
    virtual bool RunAsOne(ChxVMState* st) = 0;

    virtual void RunSteps(ChxVMState* st) {
        for (const auto& step : steps_) {
            st->set_pc(step.first);  // (what an error is reported with)
            step.second->Run(st);
        }
    }

    static int32_t Integer(const StrictScalar& z) {
        return static_cast<int32_t>(static_cast<int64_t>(z));
    }

private:
    ChxVMSteps steps_;
    std::vector<int> freed_;
};

std::atomic<int64_t> g_matmul_chains{0};

// A chain of such products, with the QuantizeLinear in front of it and the DequantizeLinear behind it where nobody else
// reads what lies between, as one launch (chx_hip_qlinear_chain).
class QLinearMatMulChainOp : public GroupOp {
public:
    struct Layer {
        int a_scale, a_zp, b_scale, b_zp, y_scale, y_zp;
        std::shared_ptr<chx_hip_chain_weights> b;
    };
    QLinearMatMulChainOp(const ChxVMInstructionProto& last, const ChxVMInstructionProto* quantize, std::vector<Layer> layers, int64_t columns, int a,
                         const ChxVMInstructionProto* dequantize, ChxVMSteps steps, std::vector<int> freed)
        : GroupOp(last, std::move(steps), std::move(freed)), quantize_(quantize != nullptr), dequantize_(dequantize != nullptr), x_(quantize ? quantize->inputs[0].array : a),
          x_scale_(quantize ? quantize->inputs[1].scalar : -1), x_zp_(quantize ? quantize->inputs[2].scalar : -1),
          y_scale_(dequantize ? dequantize->inputs[1].scalar : -1), y_zp_(dequantize ? dequantize->inputs[2].scalar : -1),
          y_(last.outputs[0]), columns_(columns), layers_(std::move(layers)) {
    }

private:
    bool RunAsOne(ChxVMState* st) override {
        auto is_null = [&](int slot) { return slot >= 0 && st->GetVar(slot)->IsNull(); };
        if (is_null(x_) || is_null(x_scale_) || is_null(x_zp_) || is_null(y_scale_) || is_null(y_zp_)) return false;
        for (const Layer& l : layers_)
            if (is_null(l.a_scale) || is_null(l.a_zp) || is_null(l.b_scale) || is_null(l.b_zp) || is_null(l.y_scale) || is_null(l.y_zp)) return false;
        auto zp_of = [&](int slot) -> StrictScalar {
            absl::optional<StrictScalar> z = st->GetOptionalScalar(slot);
            return z.has_value() ? *z : StrictScalar(chainerx::Dtype::kUInt8, chainerx::Scalar(0u), false);
        };
        const chainerx::Array& x = st->GetArray(x_);
        if (x.ndim() != 2) return false;
        const StrictScalar x_zp = zp_of(x_zp_);
        std::vector<chx_hip_chain_layer> layers(layers_.size());
        chainerx::Dtype dtype = chainerx::Dtype::kFloat32;
        for (size_t i = 0; i < layers.size(); ++i) {
            const Layer& in = layers_[i];
            chx_hip_chain_layer& l = layers[i];
            const StrictScalar y_zp = zp_of(in.y_zp);
            l.b = in.b.get();
            l.a_scale = static_cast<float>(st->GetScalar(in.a_scale));
            l.b_scale = static_cast<float>(st->GetScalar(in.b_scale));
            l.y_scale = static_cast<float>(st->GetScalar(in.y_scale));
            l.a_zero_point = Integer(zp_of(in.a_zp));
            l.b_zero_point = Integer(zp_of(in.b_zp));
            l.y_zero_point = Integer(y_zp);
            l.y_dtype = static_cast<int32_t>(y_zp.dtype());
            dtype = y_zp.dtype();
        }
        if (dtype != chainerx::Dtype::kUInt8 && dtype != chainerx::Dtype::kInt8) return false;
        chainerx::Array y = chainerx::Empty(chainerx::Shape{x.shape()[0], columns_}, dequantize_ ? chainerx::Dtype::kFloat32 : dtype);
        const chx_hip_tensor xt = x.hip();
        chx_hip_tensor yt = y.hip();
        const int rc = chx_hip_qlinear_chain(
                &xt, quantize_ ? static_cast<float>(st->GetScalar(x_scale_)) : 1.f, quantize_ ? Integer(x_zp) : 0,
                static_cast<int32_t>(quantize_ ? x_zp.dtype() : x.dtype()), layers.data(), static_cast<int32_t>(layers.size()), &yt,
                dequantize_ ? static_cast<float>(st->GetScalar(y_scale_)) : 1.f, dequantize_ ? Integer(zp_of(y_zp_)) : 0, chainerx::CurrentStream());
        // (what it refuses, and operands that are in error, are for the instructions)
        if (rc == CHX_HIP_EUNSUPPORTED || rc == CHX_HIP_EINVAL) return false;
        CHECK_EQ(CHX_HIP_OK, rc) << chx_hip_last_error();
        if (st->options().recorded_memory)  // a recording may outlive the program
            for (const Layer& l : layers_) st->options().recorded_memory->push_back(l.b);
        st->SetArray(y_, y);
        ++g_matmul_chains;
        return true;
    }

    bool quantize_, dequantize_;
    int x_, x_scale_, x_zp_, y_scale_, y_zp_, y_;
    int64_t columns_;
    std::vector<Layer> layers_;
};

// DequantizeLinear, MaxPool | AveragePool, QuantizeLinear as one instruction on the 8-bit codes
// (chx_hip_max_pool_q8 / chx_hip_average_pool_q8).  MaxPool operands: x, kernel_shape, strides,
// pads, cover_all, auto_pad; AveragePool: x, kernel_shape, strides, pads, count_include_pad
// (runtime/chxvm_defs.py:314-321 of the chainer-compiler tree).
class FusedQuantizedPoolOp : public ChxVMOp {
public:
    FusedQuantizedPoolOp(const ChxVMInstructionProto& quantize, const ChxVMInstructionProto& pool,
                         const ChxVMInstructionProto& dq, bool is_max)
        : ChxVMOp(quantize), is_max_(is_max),
          x_(dq.inputs[0].array), x_scale_(dq.inputs[1].scalar), x_zp_(dq.inputs[2].scalar),
          y_scale_(quantize.inputs[1].scalar), y_zp_(quantize.inputs[2].scalar), y_(quantize.outputs[0]),
          kernel_(pool.inputs[1].ints), strides_(pool.inputs[2].ints), pads_(pool.inputs[3].ints),
          flag_(static_cast<int>(pool.inputs[4].i)) {
        CHECK_EQ(2u, kernel_.size()) << "only 2-D pooling on the hip backend";
        if (is_max) CHECK(pool.inputs[5].s.empty() || pool.inputs[5].s == "NOTSET") << "auto_pad is not supported for a quantized MaxPool";
    }

    void Run(ChxVMState* st) override {
        if (st->trace_level()) std::cerr << (is_max_ ? "MaxPool" : "AveragePool") << "(quantized, fused) $" << x_ << " -> $" << y_ << std::endl;
        const chainerx::Array x = st->GetArray(x_);
        CHECK_EQ(4, x.ndim());
        auto scalar_or_zero = [&](int slot) -> StrictScalar {
            absl::optional<StrictScalar> z = st->GetOptionalScalar(slot);
            return z.has_value() ? *z : StrictScalar(chainerx::Dtype::kUInt8, chainerx::Scalar(0u), false);
        };
        const float xs = static_cast<float>(st->GetScalar(x_scale_)), ys = static_cast<float>(st->GetScalar(y_scale_));
        const StrictScalar xz = scalar_or_zero(x_zp_), yz = scalar_or_zero(y_zp_);
        const int kh = static_cast<int>(kernel_[0]), kw = static_cast<int>(kernel_[1]);
        const int sh = strides_.empty() ? 1 : static_cast<int>(strides_[0]), sw = strides_.empty() ? 1 : static_cast<int>(strides_[1]);
        int pb[2] = {0, 0}, pe[2] = {0, 0};
        if (pads_.size() == 2) { pb[0] = pe[0] = static_cast<int>(pads_[0]); pb[1] = pe[1] = static_cast<int>(pads_[1]); }
        if (pads_.size() == 4) { pb[0] = static_cast<int>(pads_[0]); pb[1] = static_cast<int>(pads_[1]); pe[0] = static_cast<int>(pads_[2]); pe[1] = static_cast<int>(pads_[3]); }
        auto out_dim = [&](int64_t in, int k, int s, int p0, int p1, bool cover_all) {
            return cover_all ? (in + p0 + p1 - k + s - 1) / s + 1 : (in + p0 + p1 - k) / s + 1;
        };
        const bool cover_all = is_max_ && flag_ != 0;
        const chainerx::Shape shape{x.shape()[0], x.shape()[1], out_dim(x.shape()[2], kh, sh, pb[0], pe[0], cover_all),
                                    out_dim(x.shape()[3], kw, sw, pb[1], pe[1], cover_all)};
        const bool channels_last = !x.IsContiguous() && x.strides()[1] == x.GetItemSize();
        chainerx::Array y = channels_last ? chainerx::EmptyChannelsLastPadded(shape, yz.dtype()) : chainerx::Empty(shape, yz.dtype());
        chx_hip_tensor xt = x.hip(), yt = y.hip();
        if (is_max_) {
            // the maximum of the codes is the quantized maximum only when both sides share the quantization
            CHECK(xs == ys && static_cast<int64_t>(xz) == static_cast<int64_t>(yz) && xz.dtype() == yz.dtype())
                    << "a quantized MaxPool needs the same scale and zero point before and after";
            // (for int8 the kernel returns max + (max < 0): the reference's QuantizeLinear truncates after adding
            // 0.5, so a negative code comes back one higher)
            CHXVM_HIP_CALL(chx_hip_max_pool_q8(&xt, kh, kw, sh, sw, pb[0], pb[1], pe[0], pe[1], cover_all ? 1 : 0, &yt, chainerx::CurrentStream()));
        } else {
            CHECK(pb[0] == pe[0] && pb[1] == pe[1]) << "AveragePool pads must be symmetric";
            CHXVM_HIP_CALL(chx_hip_average_pool_q8(&xt, xs, static_cast<int32_t>(static_cast<int64_t>(xz)), kh, kw, sh, sw, pb[0], pb[1],
                                                   flag_, ys, static_cast<int32_t>(static_cast<int64_t>(yz)), CHX_HIP_ROUND_REFERENCE,
                                                   &yt, chainerx::CurrentStream()));
        }
        st->SetArray(y_, y);
    }

private:
    bool is_max_;
    int x_, x_scale_, x_zp_, y_scale_, y_zp_, y_;
    std::vector<int64_t> kernel_, strides_, pads_;
    int flag_;
};

// MaxPoolOp / AveragePoolOp::RunImpl on a float32 array (runtime/ops/pooling.cc:47-75) that is not between a
// DequantizeLinear and a QuantizeLinear: operands as above.  The second output of the reference's ops, the opaque
// context of a backward pass, is not produced; a program that reads it is refused when it is loaded.
class FloatPoolOp : public ChxVMOp {
public:
    FloatPoolOp(const ChxVMInstructionProto& pool, bool is_max)
        : ChxVMOp(pool), is_max_(is_max), x_(pool.inputs[0].array), y_(pool.outputs[0]), kernel_(pool.inputs[1].ints),
          strides_(pool.inputs[2].ints), pads_(pool.inputs[3].ints), flag_(static_cast<int>(pool.inputs[4].i)) {
        CHECK_EQ(2u, kernel_.size()) << "only 2-D pooling on the hip backend";
        CHECK(pool.outputs.size() < 2 || pool.outputs[1] < 0) << "the backward context of a pool is not produced on the hip backend";
        if (is_max) CHECK(pool.inputs[5].s.empty() || pool.inputs[5].s == "NOTSET") << "auto_pad is not supported for MaxPool on the hip backend";
    }

    void Run(ChxVMState* st) override {
        if (st->trace_level()) std::cerr << (is_max_ ? "MaxPool" : "AveragePool") << "($" << x_ << ") -> $" << y_ << std::endl;
        const chainerx::Array x = st->GetArray(x_);
        CHECK_EQ(4, x.ndim());
        CHECK(x.dtype() == chainerx::Dtype::kFloat32) << "a pool outside a DequantizeLinear / QuantizeLinear pair takes float32, not " << x.dtype();
        const int kh = static_cast<int>(kernel_[0]), kw = static_cast<int>(kernel_[1]);
        const int sh = strides_.empty() ? 1 : static_cast<int>(strides_[0]), sw = strides_.empty() ? 1 : static_cast<int>(strides_[1]);
        int ph = 0, pw = 0;
        if (pads_.size() >= 2) { ph = static_cast<int>(pads_[0]); pw = static_cast<int>(pads_[1]); }
        if (pads_.size() == 4) CHECK(pads_[0] == pads_[2] && pads_[1] == pads_[3]) << "paddings for beginning and end must be the same";
        const bool cover_all = is_max_ && flag_ != 0;
        auto out_dim = [&](int64_t in, int k, int s, int p) { return cover_all ? (in + 2 * p - k + s - 1) / s + 1 : (in + 2 * p - k) / s + 1; };
        const chainerx::Shape shape{x.shape()[0], x.shape()[1], out_dim(x.shape()[2], kh, sh, ph), out_dim(x.shape()[3], kw, sw, pw)};
        chainerx::Array y = chainerx::Empty(shape, chainerx::Dtype::kFloat32);
        chx_hip_tensor xt = x.hip(), yt = y.hip();
        if (is_max_) {
            CHXVM_HIP_CALL(chx_hip_max_pool_f32(&xt, kh, kw, sh, sw, ph, pw, ph, pw, cover_all ? 1 : 0, &yt, chainerx::CurrentStream()));
        } else {
            CHXVM_HIP_CALL(chx_hip_average_pool_f32(&xt, kh, kw, sh, sw, ph, pw, flag_, &yt, chainerx::CurrentStream()));
        }
        st->SetArray(y_, y);
    }

private:
    bool is_max_;
    int x_, y_;
    std::vector<int64_t> kernel_, strides_, pads_;
    int flag_;
};

// A QLinearConv whose result is read only by a residual-sum FusionGroup (and that group): the
// convolution gets the chance to compute the group inside its kernel.  When it does, the group's
// result is stored in the group's output slot now and the group instruction later does nothing;
// when it does not (other quantization constants at run time, operands the kernel does not take),
// both instructions run as they are.
bool g_fuse_residual = true;
bool g_pair_convolutions = true;
bool g_store_minus_128 = true;

struct ResidualFusionState {
    bool fused = false;  // of the current run
};

class QLinearConvWithResidualOp : public ChxVMOp {
public:
    QLinearConvWithResidualOp(const ChxVMInstructionProto& conv, const ChxVMInstructionProto& group, const chx_hip_residual_group& g,
                              int conv_operand, std::shared_ptr<ResidualFusionState> state)
        : ChxVMOp(conv), conv_(MakeChxVMOp(conv)), g_(g), k_(conv_operand), conv_out_(conv.outputs[0]),
          other_(group.inputs[0].array_list[1 - conv_operand]), group_out_(group.outputs[0]), state_(std::move(state)) {
    }
    void InitImpl() override {
        conv_->InitImpl();
    }
    void Run(ChxVMState* st) override {
        QLinearConvResidualRequest req;
        ChxVMVar* other = st->GetVar(other_);
        if (!other->IsNull()) req.r = other->GetArray();
        auto dt = [](int32_t d) { return static_cast<chainerx::Dtype>(d); };
        req.y_scale = g_.in_scale[k_]; req.y_zero_point = g_.in_zero_point[k_]; req.y_dtype = dt(g_.in_dtype[k_]);
        req.r_scale = g_.in_scale[1 - k_]; req.r_zero_point = g_.in_zero_point[1 - k_];
        req.out_scale = g_.out_scale; req.out_zero_point = g_.out_zero_point; req.out_dtype = dt(g_.out_dtype);
        req.relu = g_.relu != 0;
        req.out_slot = group_out_;
        bool r_fits = !req.r.IsNullHandle() && req.r.dtype() == dt(g_.in_dtype[1 - k_]);
        // the other operand kept as code - 128: an int8 tensor with the zero point 128 lower
        const bool r_minus_128 = !req.r.IsNullHandle() && st->store_minus_128(other_) && req.r.dtype() == chainerx::Dtype::kInt8 &&
                                 dt(g_.in_dtype[1 - k_]) == chainerx::Dtype::kUInt8;
        if (r_minus_128) {
            req.r_zero_point -= 128;
            r_fits = true;
        }
        st->set_residual_request(r_fits ? &req : nullptr);
        try {
            conv_->Run(st);
        } catch (...) {
            st->set_residual_request(nullptr);
            throw;
        }
        st->set_residual_request(nullptr);
        state_->fused = req.done;
        if (req.done) {
            if (st->trace_level()) std::cerr << "  (residual sum $" << group_out_ << " computed by the convolution)" << std::endl;
            st->FreeVar(conv_out_);  // holds a null array: the convolution's own result was never written
            st->SetArray(group_out_, req.out);
        } else if (r_minus_128) {
            // the group instruction will run as the program wrote it: it reads plain codes
            const chainerx::Array plain = PlainCodes(req.r);
            st->FreeVar(other_);
            st->SetArray(other_, plain);
        }
    }

private:
    std::unique_ptr<ChxVMOp> conv_;
    chx_hip_residual_group g_;
    int k_, conv_out_, other_, group_out_;
    std::shared_ptr<ResidualFusionState> state_;
};

class ResidualGroupOp : public ChxVMOp {
public:
    ResidualGroupOp(const ChxVMInstructionProto& group, std::shared_ptr<ResidualFusionState> state)
        : ChxVMOp(group), group_(MakeChxVMOp(group)), state_(std::move(state)) {
    }
    void InitImpl() override {
        group_->InitImpl();
    }
    void Run(ChxVMState* st) override {
        if (state_->fused) return;
        group_->Run(st);
    }

private:
    std::unique_ptr<ChxVMOp> group_;
    std::shared_ptr<ResidualFusionState> state_;
};

std::atomic<int64_t> g_inverted_residuals{0};

// The three convolutions of an inverted residual block (1x1 expansion, depthwise 3x3, 1x1 projection whose results in between
// nobody else reads), and the residual sum behind them where the projection may compute it, as one launch
// (chx_hip_inverted_residual_run).
class InvertedResidualOp : public GroupOp {
public:
    struct Quantization {  // the variable slots of a convolution
        int x_scale, x_zp, y_scale, y_zp;
    };
    struct Sum {
        chx_hip_residual_group group;
        int conv_operand = 0, other = -1, out = -1;
        std::shared_ptr<ResidualFusionState> state;  // null: no sum
    };
    InvertedResidualOp(const ChxVMInstructionProto& projection, std::shared_ptr<chx_hip_inverted_residual> block, int x, int between, const std::vector<Quantization>& convs,
                       int64_t out_channels, int stride, bool has_bias, Sum sum, ChxVMSteps steps, std::vector<int> freed)
        : GroupOp(projection, std::move(steps), std::move(freed)), block_(std::move(block)), x_(x), between_(between), y_(projection.outputs[0]), convs_(convs), out_channels_(out_channels), stride_(stride),
          has_bias_(has_bias), sum_(std::move(sum)) {
    }

private:
    bool RunAsOne(ChxVMState* st) override {
        if (st->GetVar(x_)->IsNull() || (has_bias_ && !st->options().qlinearconv_onnx_int32_bias)) return false;
        float scales[3];
        int32_t zero_points[3];
        for (int i = 0; i < 3; ++i) {
            for (int slot : {convs_[i].x_scale, convs_[i].x_zp, convs_[i].y_scale, convs_[i].y_zp})
                if (st->GetVar(slot)->IsNull()) return false;
            const StrictScalar& zp = st->GetScalar(convs_[i].y_zp);
            if (zp.dtype() != chainerx::Dtype::kUInt8) return false;
            scales[i] = static_cast<float>(st->GetScalar(convs_[i].y_scale));
            zero_points[i] = Integer(zp);
            // each reads its input the way the one before wrote it
            if (i > 0 && (static_cast<float>(st->GetScalar(convs_[i].x_scale)) != scales[i - 1] || Integer(st->GetScalar(convs_[i].x_zp)) != zero_points[i - 1] ||
                          st->GetScalar(convs_[i].x_zp).dtype() != chainerx::Dtype::kUInt8))
                return false;
        }
        const chainerx::Array x = st->GetArray(x_);
        if (x.ndim() != 4) return false;
        const StrictScalar& x_zp = st->GetScalar(convs_[0].x_zp);
        // a value kept as code - 128 is an int8 tensor with the zero point 128 lower
        auto minus_128 = [&](int slot, const chainerx::Array& a, chainerx::Dtype type_in_program) {
            return st->store_minus_128(slot) && a.dtype() == chainerx::Dtype::kInt8 && type_in_program == chainerx::Dtype::kUInt8;
        };
        const int out_slot = sum_.state ? sum_.out : y_;
        const bool signed_storage = st->store_minus_128(out_slot);
        const chainerx::Shape shape{x.shape()[0], out_channels_, (x.shape()[2] - 1) / stride_ + 1, (x.shape()[3] - 1) / stride_ + 1};
        chainerx::Array r;
        int32_t r_zp = 0;
        if (sum_.state) {
            const chx_hip_residual_group& g = sum_.group;
            const int k = sum_.conv_operand;
            if (st->GetVar(sum_.other)->IsNull() || g.in_scale[k] != scales[2] || g.in_zero_point[k] != zero_points[2] ||
                static_cast<chainerx::Dtype>(g.in_dtype[k]) != chainerx::Dtype::kUInt8 || static_cast<chainerx::Dtype>(g.out_dtype) != chainerx::Dtype::kUInt8)
                return false;
            r = st->GetArray(sum_.other);
            const chainerx::Dtype r_type = static_cast<chainerx::Dtype>(g.in_dtype[1 - k]);
            const bool lowered = minus_128(sum_.other, r, r_type);
            if ((r.dtype() != r_type && !lowered) || r.shape() != shape) return false;
            r_zp = g.in_zero_point[1 - k] - (lowered ? 128 : 0);
        }
        chainerx::Array out = chainerx::EmptyChannelsLastPadded(shape, signed_storage ? chainerx::Dtype::kInt8 : chainerx::Dtype::kUInt8);
        const chx_hip_tensor xt = x.hip();
        chx_hip_tensor ot = out.hip(), rt;
        if (sum_.state) rt = r.hip();
        const uint32_t flags = CHX_HIP_ROUND_REFERENCE | (st->options().qlinearconv_onnx_int32_bias ? CHX_HIP_BIAS_ONNX_INT32 : CHX_HIP_BIAS_REFERENCE_FLOAT) |
                               (signed_storage ? CHX_HIP_STORE_MINUS_128 : 0u);
        const int rc = chx_hip_inverted_residual_run(
                block_.get(), &xt, static_cast<float>(st->GetScalar(convs_[0].x_scale)), Integer(x_zp) - (minus_128(x_, x, x_zp.dtype()) ? 128 : 0), scales, zero_points,
                static_cast<int32_t>(chainerx::Dtype::kUInt8), flags, sum_.state ? &rt : nullptr, sum_.group.in_scale[1 - sum_.conv_operand], r_zp, sum_.group.out_scale,
                sum_.group.out_zero_point, sum_.group.relu, &ot, chainerx::CurrentStream());
        // (what it refuses, and operands that are in error, are for the instructions)
        if (rc == CHX_HIP_EUNSUPPORTED || rc == CHX_HIP_EINVAL) return false;
        CHECK_EQ(CHX_HIP_OK, rc) << chx_hip_last_error();
        if (st->options().recorded_memory) st->options().recorded_memory->push_back(block_);  // a recording may outlive the program
        // (the depthwise result is code - 128 on its way to the projection)
        CountMinus128Stores((signed_storage ? 1 : 0) + (st->store_minus_128(between_) ? 1 : 0));
        if (sum_.state) {
            sum_.state->fused = true;
            CountResidualFusion();
            st->count_residual_fusion();
        }
        st->SetArray(out_slot, out);
        ++g_inverted_residuals;
        return true;
    }

    std::shared_ptr<chx_hip_inverted_residual> block_;
    int x_, between_, y_;
    std::vector<Quantization> convs_;
    int64_t out_channels_;
    int stride_;
    bool has_bias_;
    Sum sum_;
};

std::atomic<int64_t> g_bottlenecks{0};

// The 3x3 convolution of a bottleneck block, the 1x1 convolution behind it with the residual sum, and the 1x1 convolution that
// reads the sum in the next block (where there is one) as one launch (chx_hip_bottleneck_run).
class BottleneckOp : public GroupOp {
public:
    struct Quantization {  // the variable slots of a convolution
        int x_scale, x_zp, y_scale, y_zp;
    };
    struct Sum {
        chx_hip_residual_group group;
        int conv_operand, other, out;
        std::shared_ptr<ResidualFusionState> state;
    };
    BottleneckOp(const ChxVMInstructionProto& last, std::shared_ptr<chx_hip_bottleneck> block, int x, int between, int next, const std::vector<Quantization>& convs,
                 int64_t wide_channels, int64_t next_channels, bool has_bias, Sum sum, ChxVMSteps steps, std::vector<int> freed)
        : GroupOp(last, std::move(steps), std::move(freed)), block_(std::move(block)), x_(x), between_(between), next_(next), convs_(convs), wide_channels_(wide_channels), next_channels_(next_channels),
          has_bias_(has_bias), sum_(std::move(sum)) {
    }

private:
    bool RunAsOne(ChxVMState* st) override {
        if (st->GetVar(x_)->IsNull() || st->GetVar(sum_.other)->IsNull() || (has_bias_ && !st->options().qlinearconv_onnx_int32_bias)) return false;
        float scales[3] = {1.f, 1.f, 1.f};
        int32_t zero_points[3] = {0, 0, 0};
        const chx_hip_residual_group& g = sum_.group;
        const int k = sum_.conv_operand;
        for (size_t i = 0; i < convs_.size(); ++i) {
            for (int slot : {convs_[i].x_scale, convs_[i].x_zp, convs_[i].y_scale, convs_[i].y_zp})
                if (st->GetVar(slot)->IsNull()) return false;
            const StrictScalar& zp = st->GetScalar(convs_[i].y_zp);
            if (zp.dtype() != chainerx::Dtype::kUInt8) return false;
            scales[i] = static_cast<float>(st->GetScalar(convs_[i].y_scale));
            zero_points[i] = Integer(zp);
            // each reads its input the way it was written: the second the first's result, the third the sum
            const float scale = i == 1 ? scales[0] : g.out_scale;
            const int32_t zero_point = i == 1 ? zero_points[0] : g.out_zero_point;
            if (i > 0 && (static_cast<float>(st->GetScalar(convs_[i].x_scale)) != scale || Integer(st->GetScalar(convs_[i].x_zp)) != zero_point ||
                          st->GetScalar(convs_[i].x_zp).dtype() != chainerx::Dtype::kUInt8))
                return false;
        }
        if (g.in_scale[k] != scales[1] || g.in_zero_point[k] != zero_points[1] || static_cast<chainerx::Dtype>(g.in_dtype[k]) != chainerx::Dtype::kUInt8 ||
            static_cast<chainerx::Dtype>(g.out_dtype) != chainerx::Dtype::kUInt8)
            return false;
        const chainerx::Array x = st->GetArray(x_), r = st->GetArray(sum_.other);
        if (x.ndim() != 4) return false;
        const StrictScalar& x_zp = st->GetScalar(convs_[0].x_zp);
        // a value kept as code - 128 is an int8 tensor with the zero point 128 lower
        auto minus_128 = [&](int slot, const chainerx::Array& a, chainerx::Dtype type_in_program) {
            return st->store_minus_128(slot) && a.dtype() == chainerx::Dtype::kInt8 && type_in_program == chainerx::Dtype::kUInt8;
        };
        const chainerx::Shape shape{x.shape()[0], wide_channels_, x.shape()[2], x.shape()[3]};
        const chainerx::Dtype r_type = static_cast<chainerx::Dtype>(g.in_dtype[1 - k]);
        const bool lowered = minus_128(sum_.other, r, r_type);
        if ((r.dtype() != r_type && !lowered) || r.shape() != shape) return false;
        // (asked before there is memory for the results: on few images most blocks may be faster as their instructions)
        if (chx_hip_bottleneck_takes(block_.get(), x.shape()[0], x.shape()[2], x.shape()[3]) != CHX_HIP_OK) return false;
        const int32_t r_zp = g.in_zero_point[1 - k] - (lowered ? 128 : 0);
        const bool out_signed = st->store_minus_128(sum_.out), next_signed = next_ >= 0 && st->store_minus_128(next_);
        chainerx::Array out = chainerx::EmptyChannelsLastPadded(shape, out_signed ? chainerx::Dtype::kInt8 : chainerx::Dtype::kUInt8), next;
        if (next_ >= 0)
            next = chainerx::EmptyChannelsLastPadded(chainerx::Shape{x.shape()[0], next_channels_, x.shape()[2], x.shape()[3]}, next_signed ? chainerx::Dtype::kInt8 : chainerx::Dtype::kUInt8);
        const chx_hip_tensor xt = x.hip(), rt = r.hip();
        chx_hip_tensor ot = out.hip(), nt;
        if (next_ >= 0) nt = next.hip();
        const uint32_t flags = CHX_HIP_ROUND_REFERENCE | (st->options().qlinearconv_onnx_int32_bias ? CHX_HIP_BIAS_ONNX_INT32 : CHX_HIP_BIAS_REFERENCE_FLOAT);
        const int rc = chx_hip_bottleneck_run(
                block_.get(), &xt, static_cast<float>(st->GetScalar(convs_[0].x_scale)), Integer(x_zp) - (minus_128(x_, x, x_zp.dtype()) ? 128 : 0), scales, zero_points,
                static_cast<int32_t>(chainerx::Dtype::kUInt8), flags, &rt, g.in_scale[1 - k], r_zp, g.out_scale, g.out_zero_point, g.relu,
                out_signed ? CHX_HIP_STORE_MINUS_128 : 0u, &ot, next_signed ? CHX_HIP_STORE_MINUS_128 : 0u, next_ >= 0 ? &nt : nullptr, chainerx::CurrentStream());
        // (what it refuses, and operands that are in error, are for the instructions)
        if (rc == CHX_HIP_EUNSUPPORTED || rc == CHX_HIP_EINVAL) return false;
        CHECK_EQ(CHX_HIP_OK, rc) << chx_hip_last_error();
        if (st->options().recorded_memory) st->options().recorded_memory->push_back(block_);  // a recording may outlive the program
        // (the 3x3 convolution's result is code - 128 on its way to the next)
        CountMinus128Stores((out_signed ? 1 : 0) + (next_signed ? 1 : 0) + (st->store_minus_128(between_) ? 1 : 0));
        sum_.state->fused = true;
        CountResidualFusion();
        st->count_residual_fusion();
        st->SetArray(sum_.out, out);
        if (next_ >= 0) st->SetArray(next_, next);
        ++g_bottlenecks;
        return true;
    }

    std::shared_ptr<chx_hip_bottleneck> block_;
    int x_, between_, next_;
    std::vector<Quantization> convs_;
    int64_t wide_channels_, next_channels_;
    bool has_bias_;
    Sum sum_;
};

// A QLinearConv over constants and the instruction in front of it or behind it as one launch.  The convolution's plan is made when
// the program is loaded, and is the instruction's too where the launch is not taken.
class ConvolutionEndOp : public GroupOp {
public:
    struct Quantization {  // variable slots
        int scale, zp;
    };
    struct Convolution {
        ChxVMState::OfferedPlan plan;
        int32_t device;  // that it is on
        chainerx::Array w;
        int x;
        Quantization in, out;
    };
    ConvolutionEndOp(const ChxVMInstructionProto& last, Convolution conv, ChxVMSteps steps, std::vector<int> freed)
        : GroupOp(last, std::move(steps), std::move(freed)), conv_(std::move(conv)), y_(last.outputs[0]) {
    }

protected:
    static bool IsQ8(chainerx::Dtype t) {
        return t == chainerx::Dtype::kUInt8 || t == chainerx::Dtype::kInt8;
    }
    // The plan's memory is on one device: on another one the instructions run.
    bool OnDevice() const {
        int32_t device = 0;
        return chx_hip_get_device(&device) == CHX_HIP_OK && device == conv_.device;
    }
    void RunSteps(ChxVMState* st) override {
        if (OnDevice()) st->set_offered_plan(&conv_.plan);
        GroupOp::RunSteps(st);
        st->set_offered_plan(nullptr);
    }
    // rc: of the launch.  false: the instructions run (what it refuses, and operands that are in error, are for them)
    bool Launched(ChxVMState* st, int rc) {
        if (rc == CHX_HIP_EUNSUPPORTED || rc == CHX_HIP_EINVAL) return false;
        CHECK_EQ(CHX_HIP_OK, rc) << chx_hip_last_error();
        if (st->options().recorded_memory) st->options().recorded_memory->push_back(conv_.plan.plan);  // a recording may outlive the program
        return true;
    }

    Convolution conv_;
    int y_;
};

std::atomic<int64_t> g_quantized_convolutions{0};

// A QuantizeLinear and the convolution over few channels that reads its result (chx_hip_qconv_plan_run_quantize).
class QuantizedConvolutionOp : public ConvolutionEndOp {
public:
    // x, quantize: of the QuantizeLinear (a zero point of -1: none)
    QuantizedConvolutionOp(const ChxVMInstructionProto& conv, Convolution operands, int x, Quantization quantize, ChxVMSteps steps, std::vector<int> freed)
        : ConvolutionEndOp(conv, std::move(operands), std::move(steps), std::move(freed)), x_(x), quantize_(quantize) {
    }

private:
    bool RunAsOne(ChxVMState* st) override {
        if (!OnDevice()) return false;
        for (int slot : {x_, quantize_.scale, conv_.in.scale, conv_.in.zp, conv_.out.scale, conv_.out.zp})
            if (st->GetVar(slot)->IsNull()) return false;
        if (quantize_.zp >= 0 && st->GetVar(quantize_.zp)->IsNull()) return false;
        const chainerx::Array x = st->GetArray(x_);
        const absl::optional<StrictScalar> q_zp = st->GetOptionalScalar(quantize_.zp);  // (none: uint8 0)
        const StrictScalar &x_zp = st->GetScalar(conv_.in.zp), &y_zp = st->GetScalar(conv_.out.zp);
        if (x.ndim() != 4 || x.dtype() != chainerx::Dtype::kFloat32 || x.shape()[1] != conv_.w.shape()[1] || (q_zp.has_value() && q_zp->dtype() != chainerx::Dtype::kUInt8) ||
            x_zp.dtype() != chainerx::Dtype::kUInt8 || !IsQ8(y_zp.dtype()))
            return false;
        const chainerx::Shape y_shape = ConvOutputShape(x, conv_.w, conv_.plan.params);
        for (int64_t extent : y_shape)
            if (extent <= 0) return false;
        chainerx::Array y = chainerx::EmptyChannelsLastPadded(y_shape, y_zp.dtype());
        const chx_hip_tensor xt = x.hip();
        chx_hip_tensor yt = y.hip();
        const uint32_t flags = CHX_HIP_ROUND_REFERENCE | (st->options().qlinearconv_onnx_int32_bias ? CHX_HIP_BIAS_ONNX_INT32 : CHX_HIP_BIAS_REFERENCE_FLOAT);
        if (!Launched(st, chx_hip_qconv_plan_run_quantize(
                                  conv_.plan.plan.get(), &xt, static_cast<float>(st->GetScalar(quantize_.scale)), q_zp.has_value() ? Integer(*q_zp) : 0, static_cast<float>(st->GetScalar(conv_.in.scale)),
                                  Integer(x_zp), static_cast<float>(st->GetScalar(conv_.out.scale)), Integer(y_zp), flags, &yt, chainerx::CurrentStream())))
            return false;
        st->SetArray(y_, y);
        ++g_quantized_convolutions;
        return true;
    }

    int x_;
    Quantization quantize_;
};

std::atomic<int64_t> g_dequantized_convolutions{0};

// A convolution with 1x1 filters and the DequantizeLinear that reads its result (chx_hip_qconv_plan_run_dequantize).
class DequantizedConvolutionOp : public ConvolutionEndOp {
public:
    // dequantize: of the DequantizeLinear (a zero point of -1: none)
    DequantizedConvolutionOp(const ChxVMInstructionProto& last, Convolution operands, Quantization dequantize, ChxVMSteps steps, std::vector<int> freed)
        : ConvolutionEndOp(last, std::move(operands), std::move(steps), std::move(freed)), dequantize_(dequantize) {
    }

private:
    bool RunAsOne(ChxVMState* st) override {
        if (!OnDevice()) return false;
        for (int slot : {conv_.x, conv_.in.scale, conv_.in.zp, conv_.out.scale, conv_.out.zp, dequantize_.scale})
            if (st->GetVar(slot)->IsNull()) return false;
        if (dequantize_.zp >= 0 && st->GetVar(dequantize_.zp)->IsNull()) return false;
        const chainerx::Array x = st->GetArray(conv_.x);
        const absl::optional<StrictScalar> dq_zp = st->GetOptionalScalar(dequantize_.zp);  // (none: uint8 0)
        const StrictScalar &x_zp = st->GetScalar(conv_.in.zp), &y_zp = st->GetScalar(conv_.out.zp);
        if (x.ndim() != 4 || !IsQ8(x.dtype()) || x.shape()[1] != conv_.w.shape()[1] || !IsQ8(y_zp.dtype()) || (dq_zp.has_value() && !IsQ8(dq_zp->dtype()))) return false;
        const chainerx::Shape shape = ConvOutputShape(x, conv_.w, conv_.plan.params);
        for (int64_t extent : shape)
            if (extent <= 0) return false;
        if (shape[0] * shape[1] * shape[2] * shape[3] > CHX_HIP_MOST_DEQUANTIZED) return false;
        // (an input kept as code - 128 is an int8 tensor with the zero point 128 lower)
        const bool lowered = st->store_minus_128(conv_.x) && x.dtype() == chainerx::Dtype::kInt8 && x_zp.dtype() == chainerx::Dtype::kUInt8;
        // laid out as the DequantizeLinear does: like the convolution's result, which is channels-last with whole 16 bytes per pixel
        const bool contiguous = shape[2] == 1 && shape[3] == 1 && (shape[1] % 16 == 0 || shape[0] == 1);
        chainerx::Array y = contiguous ? chainerx::Empty(shape, chainerx::Dtype::kFloat32) : chainerx::EmptyChannelsLast(shape, chainerx::Dtype::kFloat32);
        const chx_hip_tensor xt = x.hip();
        chx_hip_tensor yt = y.hip();
        const uint32_t flags = CHX_HIP_ROUND_REFERENCE | (st->options().qlinearconv_onnx_int32_bias ? CHX_HIP_BIAS_ONNX_INT32 : CHX_HIP_BIAS_REFERENCE_FLOAT);
        if (!Launched(st, chx_hip_qconv_plan_run_dequantize(
                                  conv_.plan.plan.get(), &xt, static_cast<float>(st->GetScalar(conv_.in.scale)), Integer(x_zp) - (lowered ? 128 : 0), static_cast<float>(st->GetScalar(conv_.out.scale)),
                                  Integer(y_zp), static_cast<int32_t>(y_zp.dtype()), flags, static_cast<float>(st->GetScalar(dequantize_.scale)), dq_zp.has_value() ? Integer(*dq_zp) : 0, &yt,
                                  chainerx::CurrentStream())))
            return false;
        st->SetArray(y_, y);
        ++g_dequantized_convolutions;
        return true;
    }

    Quantization dequantize_;
};

// A fused op followed by the Free instructions of its operands that the program had placed
// between the instructions it replaces.
class SequenceOp : public ChxVMOp {
public:
    SequenceOp(const ChxVMInstructionProto& inst, std::vector<std::unique_ptr<ChxVMOp>> ops) : ChxVMOp(inst), ops_(std::move(ops)) {
    }
    void InitImpl() override {
        for (auto& op : ops_) op->InitImpl();
    }
    void Run(ChxVMState* st) override {
        for (auto& op : ops_) op->Run(st);
    }

private:
    std::vector<std::unique_ptr<ChxVMOp>> ops_;
};

class NopOp : public ChxVMOp {
public:
    explicit NopOp(const ChxVMInstructionProto& inst) : ChxVMOp(inst) {
    }
    void Run(ChxVMState*) override {
    }
};

// Number of times a variable slot is read by the program.
int CountUses(const ChxVMProgramProto& program, int slot) {
    int n = 0;
    for (const ChxVMInstructionProto& inst : program.instructions)
        for (const ChxVMValueProto& v : inst.inputs) {
            if ((v.type == ChxVMValueProto::ARRAY || v.type == ChxVMValueProto::OPTIONAL_ARRAY) && v.array == slot) ++n;
            if (v.type == ChxVMValueProto::ARRAY_LIST)
                for (int id : v.array_list) n += id == slot;
        }
    return n;
}

}  // namespace

ChxVM::ChxVM(const ChxVMProgramProto& program) : input_names_(program.input_names), input_types_(program.input_types) {
    // number of variable slots = highest id mentioned + 1 (runtime/chxvm.cc:104-140)
    int max_id = -1;
    for (const ChxVMInstructionProto& inst : program.instructions) {
        for (int o : inst.outputs) max_id = o > max_id ? o : max_id;
        for (const ChxVMValueProto& v : inst.inputs) {
            for (int id : {v.array, v.sequence, v.opaque, v.shape, v.scalar}) max_id = id > max_id ? id : max_id;
            for (int id : v.array_list) max_id = id > max_id ? id : max_id;
        }
    }
    num_variables_ = max_id + 1;
    // Find the QLinearMatMul sequences: QuantizeLinear <- MatMul <- two DequantizeLinear, every
    // intermediate read exactly once apart from its Free.
    const int n = static_cast<int>(program.instructions.size());
    const int kDequantize = OpNumber("DequantizeLinear"), kMatMul = OpNumber("MatMul"), kQuantize = OpNumber("QuantizeLinear"),
              kFree = OpNumber("Free"), kMaxPool = OpNumber("MaxPool"), kAveragePool = OpNumber("AveragePool");
    std::vector<int> producer(num_variables_ > 0 ? num_variables_ : 1, -1);
    for (int i = 0; i < n; ++i)
        for (int o : program.instructions[i].outputs)
            if (o >= 0) producer[o] = i;
    std::vector<int> role(n, 0);  // 0 plain, 1 dropped, 2 fused product, 3 fused pool (both at the QuantizeLinear)
    std::vector<std::pair<int, int>> fused_inputs(n);
    auto single_use = [&](int slot) {
        // one consumer plus at most one Free
        int frees = 0;
        for (const ChxVMInstructionProto& inst : program.instructions)
            if (inst.op == kFree && inst.inputs.size() == 1 && inst.inputs[0].array == slot) ++frees;
        return CountUses(program, slot) - frees == 1;
    };
    for (int q = 0; q < n; ++q) {
        const ChxVMInstructionProto& qi = program.instructions[q];
        if (qi.op != kQuantize || qi.inputs.size() != 3 || qi.inputs[0].array < 0) continue;
        const int m = producer[qi.inputs[0].array];
        if (m >= 0 && (program.instructions[m].op == kMaxPool || program.instructions[m].op == kAveragePool) &&
            single_use(qi.inputs[0].array)) {
            // DequantizeLinear -> pool -> QuantizeLinear; the pool's opaque context output must be unused
            const ChxVMInstructionProto& pi = program.instructions[m];
            const bool is_max = pi.op == kMaxPool;
            const bool shape_ok = pi.inputs.size() == (is_max ? 6u : 5u) && pi.inputs[0].array >= 0 &&
                                  (pi.outputs.size() < 2 || pi.outputs[1] < 0);
            const int d = shape_ok ? producer[pi.inputs[0].array] : -1;
            if (d >= 0 && program.instructions[d].op == kDequantize && program.instructions[d].inputs.size() == 3 &&
                single_use(pi.inputs[0].array)) {
                role[q] = 3;
                fused_inputs[q] = std::make_pair(d, m);
                role[m] = role[d] = 1;
            }
            continue;
        }
        if (m < 0 || program.instructions[m].op != kMatMul || !single_use(qi.inputs[0].array)) continue;
        const ChxVMInstructionProto& mi = program.instructions[m];
        const int da = producer[mi.inputs[0].array], db = producer[mi.inputs[1].array];
        if (da < 0 || db < 0 || da == db || program.instructions[da].op != kDequantize ||
            program.instructions[db].op != kDequantize)
            continue;
        if (!single_use(mi.inputs[0].array) || !single_use(mi.inputs[1].array)) continue;
        role[q] = 2;
        fused_inputs[q] = std::make_pair(da, db);
        role[m] = role[da] = role[db] = 1;
    }
    // Two QLinearConv that read the same value with the same activation quantization, strides, pads and kernel size
    // (the main-path and the shortcut convolution of a down-sampling block): the second moves up to the first and the
    // two run as one launch (role 6 = the first, now the pair; role 7 = the second, now nothing).  Every operand of the
    // second must exist where the first stands, or be a literal constant that stands between the two (the compiler
    // emits a constant in front of its first reader): those constants move up as well (role 7, run in front of the
    // pair).  The second's result then exists from the first's place on (`position` says where a value is produced
    // after this move).
    const int kQLinearConv = OpNumber("QLinearConv");
    const std::set<int> literal_ops = {OpNumber("FloatScalarConstant"), OpNumber("IntScalarConstant"), OpNumber("FloatConstant"),
                                       OpNumber("IntConstant")};
    std::vector<int> position(n);
    for (int i = 0; i < n; ++i) position[i] = i;
    std::vector<int> pair_second(n, -1);
    std::vector<std::vector<int>> pair_constants(n);
    for (int i = 0; i < n && g_pair_convolutions; ++i) {
        const ChxVMInstructionProto& ai = program.instructions[i];
        if (ai.op != kQLinearConv || role[i] != 0 || ai.inputs.size() != 13 || ai.outputs.empty()) continue;
        for (int j = i + 1; j < n; ++j) {
            const ChxVMInstructionProto& bi = program.instructions[j];
            if (bi.op == kFree && bi.inputs.size() == 1 && bi.inputs[0].array == ai.inputs[0].array) break;  // x ends here
            if (bi.op != kQLinearConv || role[j] != 0 || bi.inputs.size() != 13 || bi.outputs.empty()) continue;
            if (bi.inputs[0].array != ai.inputs[0].array) continue;
            bool same = bi.inputs[9].ints == ai.inputs[9].ints && bi.inputs[10].ints == ai.inputs[10].ints &&
                        bi.inputs[11].i == 1 && ai.inputs[11].i == 1 && bi.inputs[12].s == ai.inputs[12].s;
            // the second one's operands: produced before the first, or literal constants in between that can move up
            std::vector<int> moved;
            auto available = [&](int slot) {
                if (slot < 0 || producer[slot] < 0) return false;
                const int pr = producer[slot];
                if (pr < i) return role[pr] == 0 || position[pr] < i;
                if (pr > j || role[pr] != 0 || !literal_ops.count(program.instructions[pr].op) || program.instructions[pr].outputs.size() != 1) return false;
                moved.push_back(pr);
                return true;
            };
            for (int k : {1, 2, 6, 7}) same = same && available(bi.inputs[k].scalar);
            for (int k : {3, 4, 5}) same = same && available(bi.inputs[k].array);
            if (bi.inputs[8].array >= 0) same = same && available(bi.inputs[8].array);
            // nothing between the two may free one of them (the compiler frees a value after its last reader, which
            // the second convolution is at the latest)
            for (int f = i; f < j && same; ++f) {
                const ChxVMInstructionProto& fi = program.instructions[f];
                if (fi.op != kFree || fi.inputs.size() != 1) continue;
                for (int k : {3, 4, 5, 8}) same = same && fi.inputs[0].array != bi.inputs[k].array;
                for (int k : {1, 2, 6, 7}) same = same && fi.inputs[0].array != bi.inputs[k].scalar;
            }
            if (!same) continue;
            role[i] = 6;
            role[j] = 7;
            pair_second[i] = j;
            position[j] = i;
            std::sort(moved.begin(), moved.end());
            moved.erase(std::unique(moved.begin(), moved.end()), moved.end());
            for (int c : moved) {
                role[c] = 7;
                position[c] = i;
            }
            pair_constants[i] = moved;
            break;
        }
    }
    // Residual sums: an ElementWiseNvrtc group of the form Q(act(DQ(a) + DQ(b))) one of whose operands
    // is the result of a QLinearConv that nobody else reads, with the other operand produced
    // before that convolution.  role 4 = the convolution, role 5 = the group.
    const int kElementWise = OpNumber("ElementWiseNvrtc");
    std::vector<int> partner(n, -1), conv_operand(n, 0);
    std::vector<chx_hip_residual_group> groups(n);
    for (int e = 0; e < n && g_fuse_residual; ++e) {
        const ChxVMInstructionProto& ei = program.instructions[e];
        if (ei.op != kElementWise || role[e] != 0 || ei.inputs.size() != 4 || ei.inputs[0].array_list.size() != 2 ||
            ei.outputs.size() != 1)
            continue;
        int32_t matches = 0;
        chx_hip_residual_group g;
        if (chx_hip_elementwise_match_residual_add(ei.inputs[2].s.c_str(), &matches, &g) != 0 || !matches) continue;
        for (int k = 1; k >= 0; --k) {
            const int slot = ei.inputs[0].array_list[k], other = ei.inputs[0].array_list[1 - k];
            if (slot < 0 || other < 0 || slot == other) continue;
            const int c = producer[slot];
            if (c < 0 || program.instructions[c].op != kQLinearConv || role[c] != 0 || !single_use(slot)) continue;
            if (producer[other] < 0 || position[producer[other]] >= c) continue;  // the other operand must exist when the convolution runs
            bool other_alive = true;             // ... and still exist: no Free of it before the group
            for (int i = c; i < e; ++i)
                if (program.instructions[i].op == kFree && program.instructions[i].inputs[0].array == other) other_alive = false;
            if (!other_alive) continue;
            role[c] = 4;
            role[e] = 5;
            partner[c] = e;
            partner[e] = c;
            conv_operand[c] = k;
            groups[c] = g;
            break;
        }
    }
    // Values that may be kept as code - 128 in int8 arrays (ChxVMState::store_minus_128): every writer is a QLinearConv
    // or a residual-sum group computed inside one (the producers that know the storage; a writer that runs some other
    // way stores plain codes and the readers see that from the array's type), and every reader is a QLinearConv that
    // without groups that takes the value as its input, or a residual-sum group computed inside a convolution that takes it as the other
    // operand (QLinearConvWithResidualOp puts plain codes back when its convolution does not compute the group after
    // all).  A reading convolution with pads above 1 is left out: it pads with its input's zero point, and beyond one
    // row or column per side only a zero point stored as the byte 0 comes from the padding that costs nothing; the
    // codes of a zero point of 0, the usual one behind a Relu, are stored as 0x80.
    minus_128_slots_.assign(num_variables_ > 0 ? num_variables_ : 1, false);
    if (g_store_minus_128) {
        std::vector<int> verdict(minus_128_slots_.size(), 0);  // 0 unseen, 1 possible so far, -1 no
        auto rule_out = [&](int slot) {
            if (slot >= 0 && slot < static_cast<int>(verdict.size())) verdict[slot] = -1;
        };
        auto candidate = [&](int slot) {
            if (slot >= 0 && slot < static_cast<int>(verdict.size()) && verdict[slot] == 0) verdict[slot] = 1;
        };
        for (int i = 0; i < n; ++i) {
            const ChxVMInstructionProto& inst = program.instructions[i];
            const bool conv = inst.op == kQLinearConv && inst.inputs.size() == 13 && !inst.outputs.empty();
            // writers
            for (size_t o = 0; o < inst.outputs.size(); ++o) {
                const bool knows = (conv && o == 0 && role[i] != 1) || (role[i] == 5 && o == 0);
                if (knows) candidate(inst.outputs[o]);
                else rule_out(inst.outputs[o]);
            }
            // readers
            if (inst.op == kFree) continue;
            int conv_input = -1, residual_operand = -1;
            if (conv && role[i] != 1) {
                bool small_pads = inst.inputs[12].s.empty() || inst.inputs[12].s == "NOTSET" || inst.inputs[12].s == "VALID";
                for (int64_t pad : inst.inputs[10].ints) small_pads = small_pads && pad >= 0 && pad <= 1;
                // (a grouped convolution gains nothing from the storage)
                if (small_pads && inst.inputs[11].i == 1) conv_input = inst.inputs[0].array;
            }
            if (role[i] == 5) residual_operand = inst.inputs[0].array_list[1 - conv_operand[partner[i]]];
            for (const ChxVMValueProto& v : inst.inputs) {
                switch (v.type) {
                    case ChxVMValueProto::ARRAY:
                    case ChxVMValueProto::OPTIONAL_ARRAY:
                        if (!(v.array == conv_input && &v == &inst.inputs[0])) rule_out(v.array);
                        break;
                    case ChxVMValueProto::ARRAY_LIST:
                        for (int id : v.array_list)
                            if (!(id == residual_operand && id != inst.inputs[0].array_list[conv_operand[partner[i]]])) rule_out(id);
                        break;
                    case ChxVMValueProto::SEQUENCE: rule_out(v.sequence); break;
                    case ChxVMValueProto::OPAQUE: rule_out(v.opaque); break;
                    case ChxVMValueProto::SHAPE: rule_out(v.shape); break;
                    case ChxVMValueProto::SCALAR:
                    case ChxVMValueProto::OPTIONAL_SCALAR: rule_out(v.scalar); break;
                    default: break;
                }
            }
        }
        for (size_t v = 0; v < verdict.size(); ++v) minus_128_slots_[v] = verdict[v] == 1;
    }
    // A fused op runs where its last instruction stood but reads the operands of the earlier ones: a
    // Free of such an operand between the two (the compiler frees a value right after its last
    // reader) moves behind the fused op.
    std::vector<std::vector<int>> deferred_frees(n);
    std::vector<int> deferred(n, -1);  // the fused op that runs the Free
    for (int q = 0; q < n; ++q) {
        if (role[q] != 2 && role[q] != 3) continue;
        std::vector<int> dropped = {fused_inputs[q].first, fused_inputs[q].second};
        if (role[q] == 2) dropped.push_back(producer[program.instructions[q].inputs[0].array]);
        std::set<int> operands;
        int first = q;
        for (int d : dropped) {
            first = d < first ? d : first;
            for (const ChxVMValueProto& v : program.instructions[d].inputs) {
                if (v.type == ChxVMValueProto::ARRAY || v.type == ChxVMValueProto::OPTIONAL_ARRAY) operands.insert(v.array);
                if (v.type == ChxVMValueProto::SCALAR || v.type == ChxVMValueProto::OPTIONAL_SCALAR) operands.insert(v.scalar);
            }
        }
        for (int i = first; i < q; ++i) {
            const ChxVMInstructionProto& fi = program.instructions[i];
            if (fi.op == kFree && fi.inputs.size() == 1 && fi.inputs[0].array >= 0 && operands.count(fi.inputs[0].array)) {
                deferred[i] = q;
                deferred_frees[q].push_back(i);
            }
        }
    }
    std::vector<std::shared_ptr<ResidualFusionState>> fusion_state(n);
    std::vector<bool> dead(num_variables_ > 0 ? num_variables_ : 1, false);
    for (int i = 0; i < n; ++i)
        if (role[i] == 1)
            for (int o : program.instructions[i].outputs)
                if (o >= 0) dead[o] = true;
    for (int i = 0; i < n; ++i) {
        const ChxVMInstructionProto& inst = program.instructions[i];
        const bool frees_dead = inst.op == kFree && inst.inputs.size() == 1 && inst.inputs[0].array >= 0 && dead[inst.inputs[0].array];
        if (role[i] == 1 || role[i] == 7 || frees_dead || deferred[i] >= 0) {
            program_.emplace_back(new NopOp(inst));
        } else if (role[i] == 6) {
            std::vector<std::unique_ptr<ChxVMOp>> seq;
            for (int c : pair_constants[i]) seq.emplace_back(MakeChxVMOp(program.instructions[c]));
            seq.emplace_back(MakeQLinearConvPairOp(inst, program.instructions[pair_second[i]]));
            program_.emplace_back(new SequenceOp(inst, std::move(seq)));
        } else if (role[i] == 3) {
            const ChxVMInstructionProto& pool = program.instructions[fused_inputs[i].second];
            program_.emplace_back(new FusedQuantizedPoolOp(inst, pool, program.instructions[fused_inputs[i].first], pool.op == kMaxPool));
        } else if (role[i] == 4) {
            fusion_state[i] = std::make_shared<ResidualFusionState>();
            program_.emplace_back(new QLinearConvWithResidualOp(inst, program.instructions[partner[i]], groups[i], conv_operand[i],
                                                                fusion_state[i]));
        } else if (role[i] == 5) {
            program_.emplace_back(new ResidualGroupOp(inst, fusion_state[partner[i]]));
        } else if (role[i] == 2) {
            program_.emplace_back(new FusedQLinearMatMulOp(inst, program.instructions[fused_inputs[i].first],
                                                           program.instructions[fused_inputs[i].second]));
        } else if ((inst.op == kMaxPool || inst.op == kAveragePool) && inst.inputs.size() == (inst.op == kMaxPool ? 6u : 5u) &&
                   inst.inputs[0].array >= 0 && !inst.outputs.empty()) {
            program_.emplace_back(new FloatPoolOp(inst, inst.op == kMaxPool));
        } else {
            program_.emplace_back(MakeChxVMOp(inst));
        }
        if (!deferred_frees[i].empty()) {
            std::vector<std::unique_ptr<ChxVMOp>> seq;
            seq.push_back(std::move(program_.back()));
            for (int f : deferred_frees[i]) seq.emplace_back(MakeChxVMOp(program.instructions[f]));
            program_.back().reset(new SequenceOp(inst, std::move(seq)));
        }
        program_.back()->InitImpl();
    }
    // the constants that one instruction writes, once, as the only one
    std::vector<int> writers(num_variables_ > 0 ? num_variables_ : 1, 0);
    for (const ChxVMInstructionProto& inst : program.instructions)
        for (int o : inst.outputs)
            if (o >= 0) ++writers[o];
    constant_slots_.assign(num_variables_ > 0 ? num_variables_ : 1, nullptr);
    ChxVMState scratch(ChxVMOptions(), num_variables_, InOuts());
    for (int i = 0; i < n; ++i) {
        const ChxVMInstructionProto& inst = program.instructions[i];
        const bool constant = literal_ops.count(inst.op) && inst.outputs.size() == 1 && inst.outputs[0] >= 0 && writers[inst.outputs[0]] == 1;
        if (constant && role[i] == 0) {
            const int slot = inst.outputs[0];
            program_[i]->Run(&scratch);
            constants_.emplace_back(new ChxVMVar(*scratch.GetVar(slot)));
            constant_slots_[slot] = constants_.back().get();
        } else if (!dynamic_cast<NopOp*>(program_[i].get())) {
            remaining_.emplace_back(i, program_[i].get());
        }
    }
    // A group of instructions that runs as one launch stands where its last one stood: the Free's of its operands in front of that
    // wait for it.  Only one of two groups (or of a group and a fused op) can have a Free, so the other is not formed: it would
    // run behind the Free of what it reads.
    struct Group {
        std::set<int> moved;  // the members and their Free's
        ChxVMSteps steps;     // these, in the program's order
        std::vector<int> freed;
    };
    std::vector<bool> taken(n, false);  // Free's that a group runs
    auto gather = [&](const std::set<int>& members, int first, const std::set<int>& slots, Group* group) {
        group->moved = members;
        for (int i = first; i <= *members.rbegin(); ++i) {
            const ChxVMInstructionProto& inst = program.instructions[i];
            if (inst.op == kFree && inst.inputs.size() == 1 && slots.count(inst.inputs[0].array)) {
                if (taken[i] || (deferred[i] >= 0 && !members.count(deferred[i]))) return false;
                group->freed.push_back(inst.inputs[0].array);
                if (deferred[i] < 0) group->moved.insert(i);  // (the others run behind one of the members)
            }
            if (group->moved.count(i)) group->steps.emplace_back(i, program_[i].get());
        }
        return true;
    };
    auto install = [&](const Group& group, int last, ChxVMOp* op) {
        for (int i : group.moved) taken[i] = true;
        std::vector<std::pair<int, ChxVMOp*>> rest;
        for (const auto& r : remaining_) {
            if (r.first == last) rest.emplace_back(last, op);
            else if (!group.moved.count(r.first)) rest.push_back(r);
        }
        remaining_.swap(rest);
    };
    // Chains of fused products, for the same runs: every value between two links has one reader.  All slots involved are
    // written once, so that the links may run where the last one stood.
    std::vector<int> reader(num_variables_ > 0 ? num_variables_ : 1, -1);  // of a value that one instruction reads
    for (int i = 0; i < n; ++i) {
        const ChxVMInstructionProto& inst = program.instructions[i];
        if (inst.op == kDequantize && !inst.inputs.empty() && inst.inputs[0].array >= 0) reader[inst.inputs[0].array] = i;
    }
    auto once = [&](int slot) { return slot < 0 || writers[slot] == 1; };
    auto quantization_once = [&](const ChxVMInstructionProto& inst) {
        return inst.inputs.size() == 3 && inst.inputs[0].array >= 0 && once(inst.inputs[0].array) && inst.inputs[1].scalar >= 0 &&
               once(inst.inputs[1].scalar) && once(inst.inputs[2].scalar) && inst.outputs.size() == 1 && once(inst.outputs[0]);
    };
    std::map<int, std::shared_ptr<chx_hip_chain_weights>> laid_out;
    auto link = [&](int q) {  // a fused product that may be part of a chain: its weights are a constant (laid out here, once)
        if (role[q] != 2 || !quantization_once(program.instructions[q]) || !quantization_once(program.instructions[fused_inputs[q].first]) ||
            !quantization_once(program.instructions[fused_inputs[q].second]))
            return false;
        const ChxVMVar* constant = constant_slots_[program.instructions[fused_inputs[q].second].inputs[0].array];
        if (!constant || constant->kind() != ChxVMVar::Kind::kArray || laid_out.count(q)) return constant && laid_out.count(q) != 0;
        const chainerx::Array& b = constant->GetArray();
        if (b.ndim() != 2 || (b.dtype() != chainerx::Dtype::kUInt8 && b.dtype() != chainerx::Dtype::kInt8)) return false;
        const chx_hip_tensor bt = b.hip();
        chx_hip_chain_weights* w = nullptr;
        const int rc = chx_hip_chain_weights_create(&bt, chainerx::CurrentStream(), &w);
        if (rc == CHX_HIP_EUNSUPPORTED) return false;
        CHECK_EQ(CHX_HIP_OK, rc) << chx_hip_last_error();
        laid_out[q] = std::shared_ptr<chx_hip_chain_weights>(w, chx_hip_chain_weights_destroy);
        return true;
    };
    auto product_of = [&](int q, int slot) {  // the instruction that the value goes to, when that is as the left operand of a product
        for (int next = q + 1; next < n; ++next)
            if (role[next] == 2 && fused_inputs[next].first == reader[slot]) return next;
        return -1;
    };
    constexpr size_t kMostLinks = 6;  // of chx_hip_qlinear_chain
    std::vector<bool> chained(n, false);
    for (int q = 0; q < n; ++q) {
        if (chained[q] || !link(q)) continue;
        std::vector<int> links = {q};
        int y = program.instructions[q].outputs[0];
        for (int next; links.size() < kMostLinks && single_use(y) && reader[y] >= 0 && (next = product_of(links.back(), y)) >= 0 && link(next);) {
            links.push_back(next);
            y = program.instructions[next].outputs[0];
        }
        const int a = program.instructions[fused_inputs[q].first].inputs[0].array, head = producer[a];
        const bool quantize = head >= 0 && head < q && program.instructions[head].op == kQuantize && role[head] == 0 && single_use(a) &&
                              quantization_once(program.instructions[head]);
        const int tail = reader[y];
        const bool dequantize = tail > links.back() && single_use(y) && program.instructions[tail].op == kDequantize && role[tail] == 0 &&
                                quantization_once(program.instructions[tail]);
        if (links.size() + quantize + dequantize < 2) continue;
        std::set<int> members(links.begin(), links.end()), slots = {a};
        if (quantize) members.insert(head);
        if (dequantize) members.insert(tail);
        std::vector<QLinearMatMulChainOp::Layer> layers;
        for (int l : links) {
            const ChxVMInstructionProto &da = program.instructions[fused_inputs[l].first], &db = program.instructions[fused_inputs[l].second], &qi = program.instructions[l];
            layers.push_back({da.inputs[1].scalar, da.inputs[2].scalar, db.inputs[1].scalar, db.inputs[2].scalar, qi.inputs[1].scalar, qi.inputs[2].scalar, laid_out[l]});
            for (int slot : {da.inputs[0].array, da.inputs[1].scalar, da.inputs[2].scalar, db.inputs[0].array, db.inputs[1].scalar, db.inputs[2].scalar, qi.inputs[1].scalar, qi.inputs[2].scalar}) slots.insert(slot);
        }
        for (int end : {quantize ? head : -1, dequantize ? tail : -1}) {
            if (end < 0) continue;
            const ChxVMInstructionProto& inst = program.instructions[end];
            for (int slot : {inst.inputs[0].array, inst.inputs[1].scalar, inst.inputs[2].scalar}) slots.insert(slot);
        }
        const int64_t columns = constant_slots_[program.instructions[fused_inputs[links.back()].second].inputs[0].array]->GetArray().shape()[1];
        // (from the links' dropped instructions on: the Free of a link's operand, which waits for the link, stands behind those)
        int first = *members.begin();
        for (int l : links) first = std::min({first, fused_inputs[l].first, fused_inputs[l].second});
        const int last = *members.rbegin();
        Group group;
        if (!gather(members, first, slots, &group)) continue;
        chains_.emplace_back(new QLinearMatMulChainOp(program.instructions[last], quantize ? &program.instructions[head] : nullptr, std::move(layers), columns, a,
                                                      dequantize ? &program.instructions[tail] : nullptr, group.steps, group.freed));
        for (int m : members) chained[m] = true;
        install(group, last, chains_.back().get());
    }
    // Inverted residual blocks, for the same runs: three convolutions whose results in between have one reader, over constants.
    auto constant_array = [&](int slot) -> const chainerx::Array* {
        return slot >= 0 && constant_slots_[slot] && constant_slots_[slot]->kind() == ChxVMVar::Kind::kArray ? &constant_slots_[slot]->GetArray() : nullptr;
    };
    auto all_are = [](const std::vector<int64_t>& v, int64_t value) { return std::all_of(v.begin(), v.end(), [&](int64_t e) { return e == value; }); };
    auto convolution = [&](int i, bool last) {  // one that may be part of a block
        if (i < 0) return false;
        const ChxVMInstructionProto& inst = program.instructions[i];
        if (inst.op != kQLinearConv || inst.inputs.size() != 13 || inst.outputs.size() != 1 || !(role[i] == 0 || (last && role[i] == 4)) || chained[i]) return false;
        if (!(inst.inputs[12].s.empty() || inst.inputs[12].s == "NOTSET")) return false;
        for (int k : {0, 3, 4, 5, 8})
            if (!once(inst.inputs[k].array) || (k != 8 && inst.inputs[k].array < 0)) return false;
        for (int k : {1, 2, 6, 7})
            if (inst.inputs[k].scalar < 0 || !once(inst.inputs[k].scalar)) return false;
        for (int k : {3, 4, 5})
            if (!constant_array(inst.inputs[k].array)) return false;
        return once(inst.outputs[0]) && (inst.inputs[8].array < 0 || constant_array(inst.inputs[8].array));
    };
    std::vector<int> conv_reader(num_variables_ > 0 ? num_variables_ : 1, -1);
    for (int i = 0; i < n; ++i)
        if (program.instructions[i].op == kQLinearConv && !program.instructions[i].inputs.empty() && program.instructions[i].inputs[0].array >= 0)
            conv_reader[program.instructions[i].inputs[0].array] = i;
    for (int e = 0; e < n; ++e) {
        if (!convolution(e, false)) continue;
        const int h1 = program.instructions[e].outputs[0], d = conv_reader[h1];
        if (d <= e || !single_use(h1) || !convolution(d, false)) continue;
        const int h2 = program.instructions[d].outputs[0], p = conv_reader[h2];
        if (p <= d || !single_use(h2) || !convolution(p, true)) continue;
        const int members[3] = {e, d, p};
        const ChxVMInstructionProto& di = program.instructions[d];
        const int64_t stride = di.inputs[9].ints.empty() ? 1 : di.inputs[9].ints[0];
        bool fits = all_are(di.inputs[9].ints, stride) && !di.inputs[10].ints.empty() && all_are(di.inputs[10].ints, 1) && di.inputs[11].i > 1;
        for (int m : {e, p}) {
            const ChxVMInstructionProto& inst = program.instructions[m];
            fits = fits && all_are(inst.inputs[9].ints, 1) && all_are(inst.inputs[10].ints, 0) && inst.inputs[11].i == 1;
        }
        if (!fits) continue;
        chx_hip_conv_operands stages[3];
        chx_hip_tensor tensors[3][4];
        std::vector<InvertedResidualOp::Quantization> convs;
        std::set<int> slots = {h1, h2, program.instructions[e].inputs[0].array};
        for (int m = 0; m < 3; ++m) {
            const ChxVMInstructionProto& inst = program.instructions[members[m]];
            const int operand[4] = {inst.inputs[3].array, inst.inputs[4].array, inst.inputs[5].array, inst.inputs[8].array};
            for (int k = 0; k < 4; ++k)
                if (operand[k] >= 0) {
                    tensors[m][k] = constant_array(operand[k])->hip();
                    slots.insert(operand[k]);
                }
            stages[m] = {&tensors[m][0], &tensors[m][1], &tensors[m][2], operand[3] >= 0 ? &tensors[m][3] : nullptr};
            convs.push_back({inst.inputs[1].scalar, inst.inputs[2].scalar, inst.inputs[6].scalar, inst.inputs[7].scalar});
            for (int k : {1, 2, 6, 7}) slots.insert(inst.inputs[k].scalar);
        }
        if (tensors[1][0].shape[0] != di.inputs[11].i) continue;  // (as many groups as channels)
        Group group;
        if (!gather(std::set<int>(members, members + 3), e, slots, &group)) continue;
        chx_hip_inverted_residual* block = nullptr;
        const int rc = chx_hip_inverted_residual_create(stages, static_cast<int32_t>(stride), chainerx::CurrentStream(), &block);
        if (rc == CHX_HIP_EUNSUPPORTED || rc == CHX_HIP_EINVAL) continue;
        CHECK_EQ(CHX_HIP_OK, rc) << chx_hip_last_error();
        InvertedResidualOp::Sum sum = {};
        if (role[p] == 4) {
            const ChxVMInstructionProto& add = program.instructions[partner[p]];
            sum.group = groups[p];
            sum.conv_operand = conv_operand[p];
            sum.other = add.inputs[0].array_list[1 - conv_operand[p]];
            sum.out = add.outputs[0];
            sum.state = fusion_state[p];
        }
        chains_.emplace_back(new InvertedResidualOp(program.instructions[p], std::shared_ptr<chx_hip_inverted_residual>(block, chx_hip_inverted_residual_destroy),
                                                    program.instructions[e].inputs[0].array, h2, convs, tensors[2][0].shape[0], static_cast<int>(stride),
                                                    stages[0].bias != nullptr, sum, group.steps, group.freed));
        for (int m : members) chained[m] = true;
        install(group, p, chains_.back().get());
    }
    // Bottleneck blocks, likewise: a 3x3 convolution, the 1x1 convolution behind it that computes the residual sum, and the 1x1
    // convolution that reads the sum, where nothing but constants and Free instructions stands in between.
    for (int d = 0; d < n; ++d) {
        if (!convolution(d, false)) continue;
        const int h = program.instructions[d].outputs[0], p = conv_reader[h];
        if (p <= d || !single_use(h) || role[p] != 4 || !convolution(p, true) || partner[p] <= p) continue;
        const int e = partner[p];
        const ChxVMInstructionProto& add = program.instructions[e];
        const int out = add.outputs[0], other = add.inputs[0].array_list[1 - conv_operand[p]];
        if (!once(out) || !once(other)) continue;
        auto form = [&](int i, int64_t kernel, int64_t pad) {
            const ChxVMInstructionProto& inst = program.instructions[i];
            const chainerx::Array& w = *constant_array(inst.inputs[3].array);
            return all_are(inst.inputs[9].ints, 1) && (pad == 0 || !inst.inputs[10].ints.empty()) && all_are(inst.inputs[10].ints, pad) && inst.inputs[11].i == 1 && w.ndim() == 4 &&
                   w.shape()[2] == kernel && w.shape()[3] == kernel;
        };
        if (!form(d, 3, 1) || !form(p, 1, 0)) continue;
        auto nothing_between = [&](int from, int to) {
            for (int i = from + 1; i < to; ++i) {
                const ChxVMInstructionProto& inst = program.instructions[i];
                const bool constant = inst.outputs.size() == 1 && inst.outputs[0] >= 0 && constant_slots_[inst.outputs[0]] != nullptr;
                if (i != p && i != e && inst.op != kFree && !constant && !dynamic_cast<NopOp*>(program_[i].get())) return false;
            }
            return true;
        };
        if (!nothing_between(d, e)) continue;
        std::vector<int> convs = {d, p};
        for (int c = e + 1; c < n; ++c) {
            const ChxVMInstructionProto& inst = program.instructions[c];
            if (inst.op != kQLinearConv || inst.inputs.empty() || inst.inputs[0].array != out) continue;
            if (convolution(c, false) && form(c, 1, 0) && nothing_between(e, c)) convs.push_back(c);
            break;
        }
        int last = convs.back() > e ? convs.back() : e;
        chx_hip_conv_operands stages[3];
        chx_hip_tensor tensors[3][4];
        std::vector<BottleneckOp::Quantization> quantizations;
        std::set<int> slots = {h, program.instructions[d].inputs[0].array, program.instructions[p].outputs[0], other, out};
        auto take = [&](size_t m) {
            const ChxVMInstructionProto& inst = program.instructions[convs[m]];
            const int operand[4] = {inst.inputs[3].array, inst.inputs[4].array, inst.inputs[5].array, inst.inputs[8].array};
            for (int k = 0; k < 4; ++k)
                if (operand[k] >= 0) {
                    tensors[m][k] = constant_array(operand[k])->hip();
                    slots.insert(operand[k]);
                }
            stages[m] = {&tensors[m][0], &tensors[m][1], &tensors[m][2], operand[3] >= 0 ? &tensors[m][3] : nullptr};
            quantizations.push_back({inst.inputs[1].scalar, inst.inputs[2].scalar, inst.inputs[6].scalar, inst.inputs[7].scalar});
            for (int k : {1, 2, 6, 7}) slots.insert(inst.inputs[k].scalar);
        };
        for (size_t m = 0; m < convs.size(); ++m) take(m);
        chx_hip_bottleneck* block = nullptr;
        int rc = chx_hip_bottleneck_create(stages, static_cast<int32_t>(convs.size()), chainerx::CurrentStream(), &block);
        if (rc == CHX_HIP_EUNSUPPORTED && convs.size() == 3) {  // perhaps without the third
            convs.pop_back();
            quantizations.pop_back();
            last = e;
            rc = chx_hip_bottleneck_create(stages, 2, chainerx::CurrentStream(), &block);
        }
        if (rc == CHX_HIP_EUNSUPPORTED || rc == CHX_HIP_EINVAL) continue;
        CHECK_EQ(CHX_HIP_OK, rc) << chx_hip_last_error();
        std::shared_ptr<chx_hip_bottleneck> kept(block, chx_hip_bottleneck_destroy);
        std::set<int> members(convs.begin(), convs.end());
        members.insert(e);
        Group group;
        if (!gather(members, d, slots, &group)) continue;
        const bool reduced = convs.size() == 3;
        chains_.emplace_back(new BottleneckOp(program.instructions[last], kept, program.instructions[d].inputs[0].array, h,
                                              reduced ? program.instructions[convs[2]].outputs[0] : -1, quantizations, tensors[1][0].shape[0], reduced ? tensors[2][0].shape[0] : 0,
                                              stages[0].bias != nullptr, {groups[p], conv_operand[p], other, out, fusion_state[p]}, group.steps, group.freed));
        for (int m : convs) chained[m] = true;
        install(group, last, chains_.back().get());
    }
    // QuantizeLinear in front of a convolution over few channels, and DequantizeLinear behind one with 1x1 filters, likewise.
    for (int i = 0; i < n; ++i) {
        const ChxVMInstructionProto& other = program.instructions[i];
        const bool in_front = other.op == kQuantize;
        if ((!in_front && other.op != kDequantize) || role[i] != 0 || chained[i] || !quantization_once(other)) continue;
        const int codes = in_front ? other.outputs[0] : other.inputs[0].array;
        const int c = codes < 0 ? -1 : in_front ? conv_reader[codes] : producer[codes];
        if (c < 0 || (in_front ? c <= i : c >= i) || !single_use(codes) || !convolution(c, false)) continue;
        const ChxVMInstructionProto& ci = program.instructions[c];
        const chainerx::Array& w = *constant_array(ci.inputs[3].array);
        if (w.ndim() != 4 || ci.inputs[11].i != 1) continue;
        // (the first kernel's K axis is channels by filter rows)
        if (in_front ? w.shape()[1] * w.shape()[2] > 32 : w.shape()[2] != 1 || w.shape()[3] != 1) continue;
        const std::vector<int64_t>&strides = ci.inputs[9].ints, &pads = ci.inputs[10].ints;
        if ((!strides.empty() && strides.size() != 2) || (!pads.empty() && pads.size() != 2 && pads.size() != 4)) continue;
        auto of = [](const std::vector<int64_t>& v, size_t k, int64_t none) { return static_cast<int32_t>(v.empty() ? none : v[k]); };
        const chx_hip_conv_params params = {of(strides, 0, 1), of(strides, 1, 1), of(pads, 0, 0), of(pads, 1, 0), of(pads, pads.size() == 4 ? 2 : 0, 0), of(pads, pads.size() == 4 ? 3 : 1, 0), 1};
        std::set<int> slots = {codes, other.inputs[0].array, other.inputs[1].scalar, other.inputs[2].scalar};
        for (int k : {0, 3, 4, 5, 8}) slots.insert(ci.inputs[k].array);
        for (int k : {1, 2, 6, 7}) slots.insert(ci.inputs[k].scalar);
        Group group;
        if (!gather({i, c}, std::min(i, c), slots, &group)) continue;
        const int bias = ci.inputs[8].array;
        const chx_hip_tensor wt = w.hip(), scale = constant_array(ci.inputs[4].array)->hip(), zp = constant_array(ci.inputs[5].array)->hip();
        chx_hip_tensor bt;
        if (bias >= 0) bt = constant_array(bias)->hip();
        chx_hip_qconv_plan* plan = nullptr;
        // (operands that are in error, and no memory, are for the instruction)
        if (chx_hip_qconv_plan_create(&wt, &scale, &zp, bias >= 0 ? &bt : nullptr, &params, chainerx::CurrentStream(), &plan) != CHX_HIP_OK) continue;
        ConvolutionEndOp::Convolution conv;
        conv.plan = {std::shared_ptr<chx_hip_qconv_plan>(plan, chx_hip_qconv_plan_destroy), params};
        CHXVM_HIP_CALL(chx_hip_get_device(&conv.device));
        conv.w = w;
        conv.x = ci.inputs[0].array;
        conv.in = {ci.inputs[1].scalar, ci.inputs[2].scalar};
        conv.out = {ci.inputs[6].scalar, ci.inputs[7].scalar};
        const ConvolutionEndOp::Quantization own = {other.inputs[1].scalar, other.inputs[2].scalar};
        if (in_front) chains_.emplace_back(new QuantizedConvolutionOp(ci, std::move(conv), other.inputs[0].array, own, group.steps, group.freed));
        else chains_.emplace_back(new DequantizedConvolutionOp(other, std::move(conv), own, group.steps, group.freed));
        chained[i] = chained[c] = true;
        install(group, std::max(i, c), chains_.back().get());
    }
}

ChxVM::~ChxVM() = default;

int64_t DequantizedConvolutions() {
    return g_dequantized_convolutions.load();
}

int64_t QuantizedConvolutions() {
    return g_quantized_convolutions.load();
}

int64_t Bottlenecks() {
    return g_bottlenecks.load();
}

int64_t InvertedResiduals() {
    return g_inverted_residuals.load();
}

int64_t MatMulChains() {
    return g_matmul_chains.load();
}

void SetFuseResidual(bool on) {
    g_fuse_residual = on;
}

void SetPairConvolutions(bool on) {
    g_pair_convolutions = on;
}

void SetStoreMinus128(bool on) {
    g_store_minus_128 = on;
}

namespace {

// .npy (format 1.0) with the elements in logical (row-major) order, whatever the strides on the device
void SaveNpy(const chainerx::Array& a, const std::string& filename) {
    static const std::map<chainerx::Dtype, const char*> descr = {
            {chainerx::Dtype::kBool, "|b1"},   {chainerx::Dtype::kInt8, "|i1"},     {chainerx::Dtype::kInt16, "<i2"},
            {chainerx::Dtype::kInt32, "<i4"},  {chainerx::Dtype::kInt64, "<i8"},    {chainerx::Dtype::kUInt8, "|u1"},
            {chainerx::Dtype::kFloat16, "<f2"}, {chainerx::Dtype::kFloat32, "<f4"}, {chainerx::Dtype::kFloat64, "<f8"}};
    auto it = descr.find(a.dtype());
    CHECK(it != descr.end()) << "no .npy type for " << a.dtype();
    const int64_t item = a.GetItemSize(), total = a.GetTotalSize();
    // the bytes the array spans on the device, then a gather by strides on the host
    int64_t span = total ? item : 0;
    for (int i = 0; i < a.ndim() && total; ++i) {
        CHECK_LE(0, a.strides()[i]) << "negative strides in an output dump";
        span += (a.shape()[i] - 1) * a.strides()[i];
    }
    std::vector<char> raw(static_cast<size_t>(span)), packed(static_cast<size_t>(total * item));
    if (span) {
        const chx_hip_tensor t = a.hip();
        CHXVM_HIP_CALL(chx_hip_memcpy_d2h(raw.data(), t.data, static_cast<size_t>(span), chainerx::CurrentStream()));
    }
    std::vector<int64_t> index(static_cast<size_t>(a.ndim()), 0);
    for (int64_t flat = 0; flat < total; ++flat) {
        int64_t off = 0;
        for (int i = 0; i < a.ndim(); ++i) off += index[i] * a.strides()[i];
        std::memcpy(&packed[static_cast<size_t>(flat * item)], &raw[static_cast<size_t>(off)], static_cast<size_t>(item));
        for (int i = a.ndim() - 1; i >= 0; --i) {
            if (++index[i] < a.shape()[i]) break;
            index[i] = 0;
        }
    }
    std::ostringstream header;
    header << "{'descr': '" << it->second << "', 'fortran_order': False, 'shape': (";
    for (int i = 0; i < a.ndim(); ++i) header << a.shape()[i] << (a.ndim() == 1 || i + 1 < a.ndim() ? "," : "") << (i + 1 < a.ndim() ? " " : "");
    header << "), }";
    std::string h = header.str();
    while ((10 + h.size() + 1) % 64 != 0) h += ' ';
    h += '\n';
    std::ofstream ofs(filename, std::ios::binary);
    CHECK(ofs) << "cannot write " << filename;
    const unsigned char magic[10] = {0x93, 'N', 'U', 'M', 'P', 'Y', 1, 0, static_cast<unsigned char>(h.size() & 0xff),
                                     static_cast<unsigned char>(h.size() >> 8)};
    ofs.write(reinterpret_cast<const char*>(magic), 10);
    ofs.write(h.data(), static_cast<std::streamsize>(h.size()));
    ofs.write(packed.data(), static_cast<std::streamsize>(packed.size()));
}

// runtime/chxvm.cc:70-92
void DumpOutput(ChxVMState* st, const ChxVMOp* op, const std::string& output_dir) {
    const ChxVMInstructionProto& inst = op->instruction();
    for (size_t i = 0; i < inst.outputs.size() && i < inst.output_names.size(); ++i) {
        const int id = inst.outputs[i];
        const std::string& name = inst.output_names[i];
        if (id <= 0 || name.empty()) continue;
        // an instruction fused away when the program was loaded leaves its named outputs unset
        ChxVMVar* var = st->PeekVar(id);
        if (!var || !var->IsArray()) continue;
        std::string clean = name;
        for (char& c : clean)
            if (c == '/') c = '_';
        std::ostringstream oss;
        oss << output_dir << '/' << std::setfill('0') << std::setw(5) << inst.id << '_' << clean << ".npy";
        SaveNpy(var->GetArray(), oss.str());
    }
}

chainerx::Shape ShapeOf(const ChxVMTypeProto& type) {
    return chainerx::Shape(type.shape.begin(), type.shape.end());
}

// runtime/chxvm.cc:38-64: an instruction that names its outputs also types them; dtype 0 = untyped
void CheckType(ChxVMState* st, const ChxVMOp* op) {
    const ChxVMInstructionProto& inst = op->instruction();
    if (inst.output_names.empty()) return;
    CHECK_EQ(inst.outputs.size(), inst.output_types.size()) << op->name() << ": " << op->debug_info();
    for (size_t i = 0; i < inst.outputs.size(); ++i) {
        const ChxVMTypeProto& type = inst.output_types[i];
        if (type.dtype == 0) continue;
        const int id = inst.outputs[i];
        CHECK_LT(0, id);
        // unset: the instruction was fused into a neighbour when the program was loaded (or its result freed already)
        ChxVMVar* var = st->PeekVar(id);
        if (!var || var->IsNull() || !var->IsArray()) continue;
        const chainerx::Array& a = st->GetArray(id);
        CHECK_EQ(static_cast<chainerx::Dtype>(type.dtype), a.dtype()) << "Dtype check failed in output #" << i << ": " << op->debug_info();
        CHECK_EQ(ShapeOf(type), a.shape()) << "Shape check failed in output #" << i << ": " << op->debug_info();
    }
}

int64_t InMbs(int64_t bytes) {
    return bytes / 1000 / 1000;
}

}  // namespace

InOuts ChxVM::Run(const InOuts& program_inputs, const ChxVMOptions& options) {
    CHECK_EQ(input_names_.size(), input_types_.size());
    for (size_t i = 0; i < input_names_.size(); ++i) {
        const std::string& name = input_names_[i];
        auto found = program_inputs.find(name);
        CHECK(found != program_inputs.end()) << "Input '" << name << "' not found";  // runtime/chxvm.cc:142-143
        if (!options.check_types) continue;
        const ChxVMTypeProto& type = input_types_[i];
        const ChxVMVar& var = *found->second;
        if (var.IsArray()) {
            if (type.dtype == 0) continue;
            const chainerx::Array& a = var.GetArray();
            CHECK_EQ(static_cast<chainerx::Dtype>(type.dtype), a.dtype()) << "Input '" << name << "' has an unexpected dtype";
            CHECK_EQ(ShapeOf(type), a.shape()) << "Input '" << name << "' has an unexpected shape";
        } else {
            CHECK_EQ(0, type.dtype) << "Input '" << name << "' must be a tensor";
        }
    }
    if (options.trace_level == 0 && !options.check_types && !options.check_nans && !options.check_infs && options.dump_memory_usage == 0 &&
        !options.chrome_tracing && options.dump_outputs_dir.empty()) {
        ChxVMState state(options, constant_slots_, program_inputs);
        state.set_minus_128_slots(&minus_128_slots_);
        for (const auto& instruction : remaining_) {
            state.set_pc(instruction.first);
            try {
                instruction.second->Run(&state);
            } catch (...) {
                const ChxVMOp* op = program_[state.pc()].get();  // (one of those that a chain stands for, where it runs them)
                std::cerr << "Exception in " << op->name() << " (pc " << state.pc() << ") " << op->debug_info() << std::endl;
                throw;
            }
        }
        residual_fusions_ += state.residual_fusions();
        return state.GetOutputs();
    }
    ChxVMState state(options, num_variables_, program_inputs);
    // (a run that checks result types against the program's or writes results to files sees plain codes everywhere)
    if (!options.check_types && options.dump_outputs_dir.empty()) state.set_minus_128_slots(&minus_128_slots_);
    int64_t peak_used_mbs = 0;
    while (state.pc() < static_cast<int>(program_.size())) {
        const int pc = state.pc();
        ChxVMOp* op = program_[pc].get();
        size_t event = 0;
        if (options.chrome_tracing) event = options.chrome_tracing->Begin("ChxVM", op->name(), pc, op->instruction().flops);
        try {
            op->Run(&state);
        } catch (...) {
            std::cerr << "Exception in " << op->name() << " (pc " << pc << ") " << op->debug_info() << std::endl;
            throw;
        }
        if (options.chrome_tracing) {
            CHXVM_HIP_CALL(chx_hip_stream_synchronize(chainerx::CurrentStream()));
            options.chrome_tracing->End(event);
        }
        state.set_pc(state.pc() + 1);  // jumps set pc - 1 themselves (runtime/ops/controlflow.cc:7-21)
        if (options.check_types) CheckType(&state, op);
        if (!options.dump_outputs_dir.empty()) DumpOutput(&state, op, options.dump_outputs_dir);
        if (options.dump_memory_usage >= 1) {
            const int64_t used_mbs = InMbs(state.GetTotalVariableSize());
            peak_used_mbs = std::max(peak_used_mbs, used_mbs);
            if (options.dump_memory_usage >= 2) std::cerr << " Memory usage=" << used_mbs << "MB" << std::endl;
        }
    }
    if (options.dump_memory_usage >= 1) {
        state.ShowVariableStatus();
        std::cerr << "Peak memory usage=" << peak_used_mbs << "MB" << std::endl;
    }
    residual_fusions_ += state.residual_fusions();
    return state.GetOutputs();
}

}  // namespace runtime
}  // namespace chainer_compiler

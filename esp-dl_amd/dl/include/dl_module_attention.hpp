// The core of an attention block as one module: what Model::fuse_attention makes of the Transpose, Reshape, Split,
// MatMul, Mul, Softmax, QuantizeLinear and Reshape modules between the convolution that leaves q, k and v and the
// modules that read the block's feature map (espdl_hip_attention_s8).
#pragma once

#include "dl_module_base.hpp"
#include "espdl_hip.h"

namespace dl {
namespace module {

class Attention : public Module {
private:
    espdl_hip_attention_desc m_desc;

public:
    /// Inputs: qkv [N, H, W, channels] and, when the scores are scaled, the one-element constant.  Outputs: the feature
    /// map [N, H, W, heads * head_dim] and, when something else reads it, v in the same form.
    Attention(const char *name, const espdl_hip_attention_desc &desc) :
        Module(name, MODULE_NON_INPLACE, QUANT_TYPE_SYMM_8BIT), m_desc(desc)
    {
    }
    std::vector<std::vector<int>> get_output_shape(std::vector<std::vector<int>> &input_shapes)
    {
        std::vector<int> out = input_shapes[0];
        out.back() = m_desc.heads * m_desc.head_dim;
        return std::vector<std::vector<int>>(m_outputs_index.size(), out);
    }
    int64_t get_macs(std::vector<std::vector<int>> &input_shapes)
    {
        return (int64_t)input_shapes[0][0] * m_desc.heads * m_desc.positions * m_desc.positions *
            (m_desc.key_dim + m_desc.head_dim);
    }
    void forward(ModelContext *context, runtime_mode_t mode = RUNTIME_MODE_AUTO)
    {
        (void)mode;
        TensorBase *qkv = context->get_tensor(m_inputs_index[0]);
        TensorBase *scale = m_inputs_index.size() > 1 ? context->get_tensor(m_inputs_index[1]) : nullptr;
        TensorBase *out = context->get_tensor(m_outputs_index[0]);
        TensorBase *v = m_outputs_index.size() > 1 ? context->get_tensor(m_outputs_index[1]) : nullptr;
        if (!qkv || !out || !qkv->on_device() || !out->on_device() || qkv->shape.size() != 4 ||
            (scale && !scale->on_device()) || (v && !v->on_device())) {
            DL_LOGE("Attention", "%s: needs device tensors", name.c_str());
            return;
        }
        espdl_hip_attention_desc d = m_desc;
        d.batch = qkv->shape[0];
        d.round_mode = context->round_mode == ROUND_MODE_HALF_EVEN ? ESPDL_HIP_ROUND_HALF_EVEN : ESPDL_HIP_ROUND_HALF_UP;
        const int rc = espdl_hip_attention_s8(&d, static_cast<const int8_t *>(qkv->data),
                                              scale ? static_cast<const int8_t *>(scale->data) : nullptr,
                                              static_cast<int8_t *>(out->data), v ? static_cast<int8_t *>(v->data) : nullptr,
                                              context->stream);
        if (rc != ESPDL_HIP_OK)
            DL_LOGE("Attention", "%s: %s", name.c_str(), espdl_hip_last_error());
    }
    void print() { DL_LOGI("Attention", "heads: %d, key_dim: %d, head_dim: %d.", m_desc.heads, m_desc.key_dim, m_desc.head_dim); }
};

} // namespace module
} // namespace dl

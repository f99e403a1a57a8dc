// torch.ops.fa_amd in native code: from the dispatcher to the C ABI without Python.
//
// A decode step issues these operators by the dozen, most of them for kernels of 5 to 30 us, and a call through
// torch.library.custom_op and ctypes costs the host 24 us (10 of them in three Python kernels of the dispatcher,
// 14 in the argument checks and the ctypes call).  Through this file it costs 5 to 6: an append and an attention of four
// short sequences 44 -> 11 us, calls whose kernels take less than the host did 25 to 28 -> 17 to 19 us.
//
// The operators that torch_ops.py defines in Python (namespace fa_amd_py, the same schemas) stay what says which
// calls are valid and what an invalid one raises.  A native kernel makes the same checks, launches what passes
// them, and hands every other call -- a failed check, a status that is not FA_OK, scratch that needs a warning,
// an input that requires grad -- to the Python operator, which raises or does what it always did.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <atomic>
#include <limits>

#include "../../include/fa_kv_cache.h"
#include "../../include/fa_paged_attention.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// The C ABI's entry points, as the process has loaded them (fa_torch_ops_bind); null until then.
struct Entries {
  decltype(&fa_paged_attention_loop) loop, fp8_loop;
  decltype(&fa_paged_attention_reduce) reduce, fp8_reduce;
  decltype(&fa_kv_cache_write) kv_cache_write;
  decltype(&fa_paged_attention_loop_workspace_bytes) workspace_bytes;
};
Entries entries = {};

// The Python operators have given their one warning of scratch that a wide table could outgrow
// (fa_torch_ops_capacity_warned): from then on such a call has nothing to say and is launched here.
std::atomic<bool> capacity_warned{false};

bool fits_int32(int64_t v) { return v >= std::numeric_limits<int32_t>::min() && v <= std::numeric_limits<int32_t>::max(); }

bool is_16bit(at::ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }
bool is_byte_cache(at::ScalarType t) { return t == at::kFloat8_e5m2 || t == at::kFloat8_e4m3fn || t == at::kByte; }

// Block ids, heads and rows are checked against key_cache alone, so value_cache has to hold at least as much.
bool covers(const Tensor &value_cache, const Tensor &key_cache) {
  for (int64_t d = 0; d < key_cache.dim(); ++d)
    if (value_cache.size(d) < key_cache.size(d)) return false;
  return true;
}

bool same_device(const Tensor &anchor, const Tensor &t) { return t.device() == anchor.device(); }
bool same_device(const Tensor &anchor, const OptTensor &t) { return !t.has_value() || t->device() == anchor.device(); }

// k_scales / v_scales into the options; false: not a pair the kernels take.
bool set_scales(fa_paged_attention_options &op, const OptTensor &k_scales, const OptTensor &v_scales, int64_t kv_heads,
                int64_t blocks, const Tensor &anchor) {
  if (!k_scales.has_value() && !v_scales.has_value()) return true;
  if (!k_scales.has_value() || !v_scales.has_value()) return false;
  for (const Tensor *t : {&*k_scales, &*v_scales})
    if (t->scalar_type() != at::kFloat || !t->is_contiguous() || !same_device(anchor, *t) || t->sizes() != k_scales->sizes())
      return false;
  if (k_scales->dim() == 1 && k_scales->size(0) == kv_heads) op.kv_scale_mode = FA_KV_SCALE_HEAD;
  else if (k_scales->dim() == 2 && k_scales->size(0) == blocks && k_scales->size(1) == kv_heads) op.kv_scale_mode = FA_KV_SCALE_BLOCK;
  else return false;
  op.k_scales = static_cast<const float *>(k_scales->const_data_ptr());
  op.v_scales = static_cast<const float *>(v_scales->const_data_ptr());
  return true;
}

struct Scratch { const Tensor &exp_sums, &max_logits, &tmp_out; };

// One attention call; false: the Python operator has to see it.
bool attend(const Tensor &out, const Scratch *scratch, const Tensor &query, const Tensor &key_cache, const Tensor &value_cache,
            const Tensor &block_tables, const Tensor &context_lens, double scale, bool fp8, double fp8_scale,
            int64_t partition_size, const OptTensor &sinks, const OptTensor &alibi_slopes, double softcap, int64_t window_left,
            const OptTensor &k_scales, const OptTensor &v_scales, int64_t max_context_len) {
  if (!entries.loop || !query.is_cuda()) return false;
  for (const Tensor *t : {&out, &key_cache, &value_cache, &block_tables, &context_lens})
    if (!same_device(query, *t)) return false;
  if (!same_device(query, sinks) || !same_device(query, alibi_slopes)) return false;
  if (!query.is_contiguous() || !out.is_contiguous() || !block_tables.is_contiguous() || !context_lens.is_contiguous()) return false;
  const auto q_type = query.scalar_type(), kv_type = key_cache.scalar_type();
  if (!is_16bit(q_type) || out.scalar_type() != q_type) return false;
  if (block_tables.scalar_type() != at::kInt || context_lens.scalar_type() != at::kInt) return false;
  if ((fp8 ? !is_byte_cache(kv_type) : kv_type != q_type) || value_cache.scalar_type() != kv_type) return false;
  if (key_cache.dim() != 4 || key_cache.stride(3) != 1 || value_cache.strides() != key_cache.strides()) return false;
  if (!covers(value_cache, key_cache)) return false;
  if ((query.dim() != 3 && query.dim() != 4) || out.sizes() != query.sizes()) return false;
  const int64_t S = query.size(0), QL = query.dim() == 4 ? query.size(1) : 1, H = query.size(-2), D = query.size(-1);
  const int64_t blocks = key_cache.size(0), block_size = key_cache.size(1), kv_heads = key_cache.size(2);
  if (block_tables.dim() != 2 || block_tables.size(0) != S || context_lens.numel() != S || key_cache.size(3) != D) return false;
  if (kv_heads <= 0 || H % kv_heads != 0) return false;
  for (int64_t v : {S, QL, H, D, blocks, block_size, kv_heads, block_tables.size(1), partition_size, window_left, max_context_len})
    if (!fits_int32(v)) return false;
  if (sinks.has_value() && (sinks->scalar_type() != q_type || sinks->numel() != H || !sinks->is_contiguous())) return false;

  fa_paged_attention_shape sh = FA_PAGED_ATTENTION_SHAPE_INIT;
  sh.num_seqs = (int32_t)S;
  sh.num_heads = (int32_t)H;
  sh.num_kv_heads = (int32_t)kv_heads;
  sh.head_size = (int32_t)D;
  sh.block_size = (int32_t)block_size;
  sh.max_blocks_per_seq = (int32_t)block_tables.size(1);
  sh.max_num_partitions = 1;
  sh.partition_size = (int32_t)partition_size;
  sh.kv_block_stride = key_cache.stride(0);
  sh.kv_token_stride = key_cache.stride(1);
  sh.kv_head_stride = key_cache.stride(2);
  sh.num_pool_blocks = (int32_t)blocks;
  sh.q_dtype = q_type == at::kBFloat16 ? FA_DTYPE_BF16 : FA_DTYPE_F16;

  fa_paged_attention_options_workspace full = FA_PAGED_ATTENTION_OPTIONS_WORKSPACE_INIT;
  fa_paged_attention_options &op = full.options;
  op.sinks = sinks.has_value() ? sinks->const_data_ptr() : nullptr;
  op.softcap = (float)softcap;
  op.fp8_scale = (float)fp8_scale;
  if (alibi_slopes.has_value()) {
    if (alibi_slopes->scalar_type() != at::kFloat || !alibi_slopes->is_contiguous() || alibi_slopes->numel() != H) return false;
    op.alibi_slopes = static_cast<const float *>(alibi_slopes->const_data_ptr());
    op.mask_flags |= FA_MASK_ALIBI;
  }
  if (softcap > 0.0) op.mask_flags |= FA_MASK_SOFTCAP;
  if (window_left >= 0) {
    op.mask_flags |= FA_MASK_WINDOW;
    op.window_left = (int32_t)window_left;
  }
  op.query_len = (int32_t)QL;
  if (!fp8 && (k_scales.has_value() || v_scales.has_value())) return false;
  if (!set_scales(op, k_scales, v_scales, kv_heads, blocks, query)) return false;
  op.kv_fp8_format = kv_type == at::kFloat8_e4m3fn ? FA_FP8_E4M3 : FA_FP8_E5M2;

  if (scratch) {
    for (const Tensor *t : {&scratch->exp_sums, &scratch->max_logits, &scratch->tmp_out})
      if (!same_device(query, *t) || t->scalar_type() != at::kFloat || !t->is_contiguous() || t->dim() < 1) return false;
    const int64_t partitions = scratch->max_logits.size(-1);
    const int64_t slots = S * QL * H * partitions;
    if (!fits_int32(partitions) || scratch->max_logits.numel() != slots || scratch->exp_sums.numel() != slots ||
        scratch->tmp_out.numel() != slots * D)
      return false;
    sh.max_num_partitions = (int32_t)partitions;
    if (max_context_len < 0) {  // unknown: the Python operator warns, once, where the scratch arrays may be too small
      const int64_t size = partition_size > 0 ? partition_size : (D == 64 ? 256 : 512);
      if (scratch->exp_sums.size(-1) * size < block_tables.size(1) * block_size && !capacity_warned.load(std::memory_order_relaxed))
        return false;
      max_context_len = 0;
    }
  }

  const c10::DeviceGuard guard(query.device());
  op.stream = c10::hip::getCurrentHIPStream(query.device().index()).stream();
  const auto *tables = static_cast<const int32_t *>(block_tables.const_data_ptr());
  const auto *lens = static_cast<const int32_t *>(context_lens.const_data_ptr());
  void *o = out.data_ptr();
  const void *q = query.const_data_ptr(), *k = key_cache.const_data_ptr(), *v = value_cache.const_data_ptr();
  if (scratch)
    return (fp8 ? entries.fp8_reduce : entries.reduce)(
               o, q, k, v, tables, lens, (float)scale, (int32_t)max_context_len, static_cast<float *>(scratch->exp_sums.data_ptr()),
               static_cast<float *>(scratch->max_logits.data_ptr()), static_cast<float *>(scratch->tmp_out.data_ptr()), &sh,
               &op) == FA_OK;
  Tensor space;
  if (const int64_t need = entries.workspace_bytes(&sh, &op, fp8); need > 0) {  // see fa_paged_attention_options_workspace
    try {
      space = at::empty({need}, query.options().dtype(at::kByte));
      full.workspace = space.data_ptr();
      full.workspace_bytes = need;
    } catch (const c10::OutOfMemoryError &) {  // the call needs none
    }
  }
  return (fp8 ? entries.fp8_loop : entries.loop)(o, q, k, v, tables, lens, (float)scale, 0, &sh, &op) == FA_OK;
}

bool append(const Tensor &key, const Tensor &value, const Tensor &key_cache, const Tensor &value_cache, const Tensor &slot_mapping,
            double fp8_scale, const OptTensor &k_scales, const OptTensor &v_scales) {
  if (!entries.loop || !key.is_cuda()) return false;
  for (const Tensor *t : {&value, &key_cache, &value_cache, &slot_mapping})
    if (!same_device(key, *t)) return false;
  const auto type = key.scalar_type(), kv_type = key_cache.scalar_type();
  if (!is_16bit(type) || value.scalar_type() != type) return false;
  if (key.dim() != 3 || key.stride(2) != 1 || value.sizes() != key.sizes() || value.strides() != key.strides()) return false;
  const bool fp8 = is_byte_cache(kv_type);
  if ((!fp8 && kv_type != type) || value_cache.scalar_type() != kv_type) return false;
  if (key_cache.dim() != 4 || key_cache.stride(3) != 1 || value_cache.strides() != key_cache.strides() ||
      !covers(value_cache, key_cache) || key_cache.size(2) != key.size(1) || key_cache.size(3) != key.size(2))
    return false;
  if (slot_mapping.scalar_type() != at::kLong || !slot_mapping.is_contiguous() || slot_mapping.numel() != key.size(0)) return false;
  for (int64_t v : {key.size(0), key.size(1), key.size(2), key_cache.size(1)})
    if (!fits_int32(v)) return false;
  fa_kv_cache_write_shape sh = FA_KV_CACHE_WRITE_SHAPE_INIT;
  sh.num_tokens = (int32_t)key.size(0);
  sh.num_kv_heads = (int32_t)key.size(1);
  sh.head_size = (int32_t)key.size(2);
  sh.block_size = (int32_t)key_cache.size(1);
  sh.kv_block_stride = key_cache.stride(0);
  sh.kv_token_stride = key_cache.stride(1);
  sh.kv_head_stride = key_cache.stride(2);
  sh.src_token_stride = key.stride(0);
  sh.src_head_stride = key.stride(1);
  sh.src_dtype = type == at::kBFloat16 ? FA_DTYPE_BF16 : FA_DTYPE_F16;
  sh.cache_dtype = !fp8 ? FA_KV_CACHE_16BIT : kv_type == at::kFloat8_e4m3fn ? FA_KV_CACHE_E4M3 : FA_KV_CACHE_E5M2;
  sh.num_pool_blocks = key_cache.size(0);
  fa_paged_attention_options op = FA_PAGED_ATTENTION_OPTIONS_INIT;
  op.fp8_scale = (float)fp8_scale;
  if (!fp8 && (k_scales.has_value() || v_scales.has_value())) return false;
  if (!set_scales(op, k_scales, v_scales, key.size(1), key_cache.size(0), key)) return false;
  const c10::DeviceGuard guard(key.device());
  op.stream = c10::hip::getCurrentHIPStream(key.device().index()).stream();
  return entries.kv_cache_write(key.const_data_ptr(), value.const_data_ptr(), key_cache.data_ptr(), value_cache.data_ptr(),
                                static_cast<const int64_t *>(slot_mapping.const_data_ptr()), &sh, &op) == FA_OK;
}

// ---- dispatcher kernels -------------------------------------------------------------------------
// Boxed, one for all operators: which arguments there are and which of them are written is the schema's to say.

// The operator of the same name that is written in Python.
c10::OperatorHandle in_python(const c10::OperatorHandle &op) {
  const std::string &name = op.schema().name();  // fa_amd::...
  return c10::Dispatcher::singleton().findSchemaOrThrow(("fa_amd_py" + name.substr(name.find("::"))).c_str(), "");
}

void autograd(const c10::OperatorHandle &op, c10::DispatchKeySet keys, torch::jit::Stack *stack) {
  const size_t n = op.schema().arguments().size();
  if (at::GradMode::is_enabled())
    for (const auto &arg : torch::jit::last(*stack, n))
      if (arg.isTensor() && arg.toTensor().requires_grad()) return in_python(op).callBoxed(stack);
  at::AutoDispatchBelowAutograd below;
  op.redispatchBoxed(keys & c10::after_autograd_keyset, stack);
}

void written_versions(const c10::OperatorHandle &op, c10::DispatchKeySet keys, torch::jit::Stack *stack) {
  const auto &args = op.schema().arguments();
  const auto given = torch::jit::last(*stack, args.size());
  for (size_t k = 0; k < args.size(); ++k)
    if (args[k].alias_info() && args[k].alias_info()->isWrite()) {
      const Tensor &t = given[k].toTensor();
      if (t.is_inference()) {  // (no version to count: what the Python operator says to that)
        return in_python(op).callBoxed(stack);
      }
    }
  for (size_t k = 0; k < args.size(); ++k)
    if (args[k].alias_info() && args[k].alias_info()->isWrite()) given[k].toTensor().unsafeGetTensorImpl()->bump_version();
  at::AutoDispatchBelowADInplaceOrView below;
  op.redispatchBoxed(keys & c10::after_ADInplaceOrView_keyset, stack);
}

// Arguments by name order of the schema; a kernel reads them off the stack, and drops them once they are launched.
struct Args {
  torch::jit::Stack *stack;
  size_t n, at = 0;
  const c10::IValue &next() { return torch::jit::peek(*stack, at++, n); }
  const Tensor &tensor() { return next().toTensor(); }
  OptTensor maybe() { return next().toOptional<Tensor>(); }
  double real() { return next().toDouble(); }
  int64_t integer() { return next().toInt(); }
};

template <bool kSplit, bool kFp8>
void attention(const c10::OperatorHandle &op, torch::jit::Stack *stack) {
  const size_t n = op.schema().arguments().size();
  Args a{stack, n};
  const Tensor &out = a.tensor();
  const Tensor *es = nullptr, *ml = nullptr, *tmp = nullptr;
  if constexpr (kSplit) es = &a.tensor(), ml = &a.tensor(), tmp = &a.tensor();
  const Tensor &query = a.tensor(), &kc = a.tensor(), &vc = a.tensor(), &tables = a.tensor(), &lens = a.tensor();
  const double scale = a.real(), fp8_scale = kFp8 ? a.real() : 1.0;
  const int64_t partition_size = kSplit ? a.integer() : 0;
  const OptTensor sinks = a.maybe(), slopes = a.maybe();
  const double softcap = a.real();
  const int64_t window_left = a.integer();
  OptTensor ks, vs;
  if constexpr (kFp8) ks = a.maybe(), vs = a.maybe();
  const int64_t longest = kSplit ? a.integer() : 0;
  bool done;
  if constexpr (kSplit) {
    const Scratch scratch{*es, *ml, *tmp};
    done = attend(out, &scratch, query, kc, vc, tables, lens, scale, kFp8, fp8_scale, partition_size, sinks, slopes, softcap,
                  window_left, ks, vs, longest);
  } else {
    done = attend(out, nullptr, query, kc, vc, tables, lens, scale, kFp8, fp8_scale, 0, sinks, slopes, softcap, window_left, ks,
                  vs, 0);
  }
  if (!done) return in_python(op).callBoxed(stack);
  torch::jit::drop(*stack, n);
}

void cache_write(const c10::OperatorHandle &op, torch::jit::Stack *stack) {
  const size_t n = op.schema().arguments().size();
  Args a{stack, n};
  const Tensor &key = a.tensor(), &value = a.tensor(), &kc = a.tensor(), &vc = a.tensor(), &slots = a.tensor();
  const double fp8_scale = a.real();
  const OptTensor ks = a.maybe(), vs = a.maybe();
  if (!append(key, value, kc, vc, slots, fp8_scale, ks, vs)) return in_python(op).callBoxed(stack);
  torch::jit::drop(*stack, n);
}

}  // namespace

// table: addresses of the entry points in the order of Entries; 0: not as many as this library was built for.
extern "C" __attribute__((visibility("default"))) int fa_torch_ops_bind(void *const *table, size_t count) {
  if (count * sizeof(void *) != sizeof(Entries)) return 0;
  memcpy(&entries, table, sizeof(Entries));
  return 1;
}

extern "C" __attribute__((visibility("default"))) void fa_torch_ops_capacity_warned() { capacity_warned.store(true); }

TORCH_LIBRARY_FRAGMENT(fa_amd, m) {
  const std::vector<at::Tag> tags = {at::Tag::pt2_compliant_tag};
  m.def("paged_attention_loop(Tensor(a0!) out, Tensor query, Tensor key_cache, Tensor value_cache, Tensor block_tables, "
        "Tensor context_lens, float scale, Tensor? sinks=None, Tensor? alibi_slopes=None, float softcap=0., "
        "SymInt window_left=-1) -> ()", tags);
  m.def("paged_attention_fp8_loop(Tensor(a0!) out, Tensor query, Tensor key_cache, Tensor value_cache, Tensor block_tables, "
        "Tensor context_lens, float scale, float fp8_scale, Tensor? sinks=None, Tensor? alibi_slopes=None, float softcap=0., "
        "SymInt window_left=-1, Tensor? k_scales=None, Tensor? v_scales=None) -> ()", tags);
  m.def("paged_attention_reduce(Tensor(a0!) out, Tensor(a1!) exp_sums, Tensor(a2!) max_logits, Tensor(a3!) tmp_out, "
        "Tensor query, Tensor key_cache, Tensor value_cache, Tensor block_tables, Tensor context_lens, float scale, "
        "SymInt partition_size=0, Tensor? sinks=None, Tensor? alibi_slopes=None, float softcap=0., SymInt window_left=-1, "
        "SymInt max_context_len=-1) -> ()", tags);
  m.def("paged_attention_fp8_reduce(Tensor(a0!) out, Tensor(a1!) exp_sums, Tensor(a2!) max_logits, Tensor(a3!) tmp_out, "
        "Tensor query, Tensor key_cache, Tensor value_cache, Tensor block_tables, Tensor context_lens, float scale, "
        "float fp8_scale, SymInt partition_size=0, Tensor? sinks=None, Tensor? alibi_slopes=None, float softcap=0., "
        "SymInt window_left=-1, Tensor? k_scales=None, Tensor? v_scales=None, SymInt max_context_len=-1) -> ()", tags);
  m.def("kv_cache_write(Tensor key, Tensor value, Tensor(a2!) key_cache, Tensor(a3!) value_cache, Tensor slot_mapping, "
        "float fp8_scale=1., Tensor? k_scales=None, Tensor? v_scales=None) -> ()", tags);
}

TORCH_LIBRARY_IMPL(fa_amd, CUDA, m) {
  m.impl("paged_attention_loop", torch::CppFunction::makeFromBoxedFunction<&attention<false, false>>());
  m.impl("paged_attention_fp8_loop", torch::CppFunction::makeFromBoxedFunction<&attention<false, true>>());
  m.impl("paged_attention_reduce", torch::CppFunction::makeFromBoxedFunction<&attention<true, false>>());
  m.impl("paged_attention_fp8_reduce", torch::CppFunction::makeFromBoxedFunction<&attention<true, true>>());
  m.impl("kv_cache_write", torch::CppFunction::makeFromBoxedFunction<&cache_write>());
}

TORCH_LIBRARY_IMPL(fa_amd, Autograd, m) {
  for (const char *name : {"paged_attention_loop", "paged_attention_fp8_loop", "paged_attention_reduce",
                           "paged_attention_fp8_reduce", "kv_cache_write"})
    m.impl(name, torch::CppFunction::makeFromBoxedFunction<&autograd>());
}

TORCH_LIBRARY_IMPL(fa_amd, ADInplaceOrView, m) {
  for (const char *name : {"paged_attention_loop", "paged_attention_fp8_loop", "paged_attention_reduce",
                           "paged_attention_fp8_reduce", "kv_cache_write"})
    m.impl(name, torch::CppFunction::makeFromBoxedFunction<&written_versions>());
}

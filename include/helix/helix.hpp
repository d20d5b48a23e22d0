// helix.hpp — native C++ host layer over libhelix_hip.so's C ABI, mirroring the reference's
// Rust interface for the SSM path so a C++ caller writes what a HelixML caller writes:
//
//   tensor_core:  Shape, DType, Device, TensorError (crates/tensor-core/src/{shape,dtype,device,
//                 error}.rs), the Tensor trait's constructors and to/from host copies
//                 (tensor.rs:7-59, TensorRandom 212-233) on a device tensor, HipTensor;
//   nn:           Linear (crates/nn/src/lib.rs:53-134), RMSNorm (lib.rs:219-285), the exported
//                 MambaBlock (Linear -> SiLU -> Linear, lib.rs:846-906), ssm::S4Block
//                 (ssm.rs:37-186, checkpoint/restore 331-360), ssm::MambaBlock (ssm.rs:435-483),
//                 and the full selective Mamba block (MambaBlockFused);
//   training:     the checkpoint file of CheckpointManager (training/src/checkpoint.rs:137-198):
//                 u32 big-endian metadata length, metadata JSON, then bincode 1.x of
//                 Vec<CpuTensor> — HipTensors are written in exactly the bytes a CpuTensor with
//                 the same values writes, and read back from them;
//   hal:          ComputeBackend (crates/hal/src/backend.rs:13-70) and ComputeGraph
//                 (hal/src/operations.rs:87-230) for ROCm, the full OperationType enum
//                 (hal/src/device.rs:129-210).
//
// Errors are thrown as helix::TensorError carrying the reference's variant; nothing here
// computes on the host: every value comes from the HIP kernels behind include/helix_hip.h.
#pragma once

#include <cstddef>
#include <cstdint>
#include <map>
#include <memory>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

namespace helix {

// ----------------------------------------------------------------------------- tensor_core
// tensor_core::TensorError variants (crates/tensor-core/src/error.rs:7-37), declaration order.
enum class ErrorKind {
    ShapeMismatch,
    InvalidDimension,
    DeviceMismatch,
    DTypeMismatch,
    UnsupportedOperation,
    AllocationFailed,
    BackendError,
    SerializationError,
    InvalidCheckpoint,
    InvalidInput,
};

class TensorError : public std::runtime_error {
public:
    TensorError(ErrorKind k, const std::string& msg) : std::runtime_error(msg), kind_(k) {}
    ErrorKind kind() const { return kind_; }
    // The variant for a libhelix_hip status code (include/helix_hip.h hx_status).
    static TensorError from_status(int status, const std::string& what);

private:
    ErrorKind kind_;
};

// Throws the TensorError for a non-zero hx status, with the library's last error text.
void check(int status, const char* what);

// tensor_core::DType (dtype.rs:8-37), same variant order (it is the bincode tag).
enum class DType : uint32_t { I8, I16, I32, I64, U8, U16, U32, U64, F16, F32, F64, Bool, C32, C64 };

// tensor_core::Shape (shape.rs:8-97): row-major dims.
class Shape {
public:
    Shape() = default;
    explicit Shape(std::vector<size_t> dims) : dims_(std::move(dims)) {}
    const std::vector<size_t>& as_slice() const { return dims_; }
    size_t ndim() const { return dims_.size(); }
    size_t dim(size_t i) const;
    size_t numel() const;
    bool operator==(const Shape& o) const { return dims_ == o.dims_; }
    bool operator!=(const Shape& o) const { return dims_ != o.dims_; }

private:
    std::vector<size_t> dims_;
};

// tensor_core::Device (device.rs:8-25). The reference has no ROCm variant; a HipTensor lives on
// Custom("rocm:<id>").
struct Device {
    enum class Kind : uint32_t { Cpu, Cuda, Metal, Wgpu, Qpu, Npu, Tpu, Custom } kind = Kind::Cpu;
    uint64_t index = 0;
    std::string name;
    static Device cpu() { return Device{}; }
    static Device rocm(int id) { return Device{Kind::Custom, 0, "rocm:" + std::to_string(id)}; }
    bool operator==(const Device& o) const { return kind == o.kind && index == o.index && name == o.name; }
};

// Storage of a device tensor: fp32, or bf16 (the north-star block's storage; DType has no BF16,
// so such a tensor reports DType::F32 values when copied to the host or serialised).
enum class Storage { F32, BF16 };

// Seeded host generator for the reference's TensorRandom distributions (SplitMix64 with
// Box-Muller normals): the reference's own generator is unseeded thread_rng
// (backend-cpu/src/lib.rs:1209-1257), so only the distributions can match.
class Rng {
public:
    explicit Rng(uint64_t seed) : s_(seed) {}
    uint64_t next_u64();
    float uniform(float lo, float hi);
    float normal(float mean, float std);

private:
    uint64_t s_;
    bool have_spare_ = false;
    double spare_ = 0.0;
};

// A device tensor: the HipTensor a crates/backend-hip would define. Owns device memory
// (hx_malloc/hx_free); the data are row-major contiguous. Beside them it records the strides the
// reference's ndarray array would have (helixml_amd/host/ndlayout.hpp): a transpose keeps permuted
// strides there, and mean's summation order and cat/stack/broadcast_to's failures follow them.
class HipTensor {
public:
    HipTensor() = default;
    HipTensor(Shape shape, Storage st, int device = 0);  // uninitialised
    static HipTensor zeros(Shape shape, Storage st = Storage::F32, int device = 0);
    static HipTensor ones(Shape shape, Storage st = Storage::F32, int device = 0);
    static HipTensor from_host(const std::vector<float>& values, Shape shape,
                               Storage st = Storage::F32, int device = 0);
    static HipTensor random_normal(Shape shape, float mean, float std, Rng& rng,
                                   Storage st = Storage::F32, int device = 0);
    static HipTensor random_uniform(Shape shape, float lo, float hi, Rng& rng,
                                    Storage st = Storage::F32, int device = 0);

    const Shape& shape() const { return shape_; }
    Storage storage() const { return storage_; }
    DType dtype() const { return DType::F32; }
    Device device() const { return Device::rocm(device_); }
    size_t numel() const { return shape_.numel(); }
    size_t nbytes() const { return numel() * (storage_ == Storage::BF16 ? 2 : 4); }
    void* data() const { return buf_ ? buf_->ptr : nullptr; }
    bool defined() const { return buf_ != nullptr; }

    std::vector<float> to_host() const;  // values as f32 (bf16 widened exactly)
    HipTensor to_storage(Storage st) const;
    HipTensor reshape(Shape s) const;  // shares storage
    HipTensor clone() const;

    // ---- TensorOps (tensor.rs:62-134) with CpuTensor's semantics and errors
    // (backend-cpu/src/lib.rs); fp32 storage. Values come from the device primitives of
    // helix_hip.h (hx_binary_f32, hx_unary_f32, hx_mean_axis_f32, hx_copy_strided_f32, ...).
    // matmul: 2-D x 2-D, 1-D x 2-D, 2-D x 1-D (lib.rs:634-757), bit-exact; other ranks
    // UnsupportedOperation as the reference.
    HipTensor matmul(const HipTensor& other) const;
    HipTensor add(const HipTensor& o) const;  // equal shapes (lib.rs:570-632), bit-exact
    HipTensor sub(const HipTensor& o) const;
    HipTensor mul(const HipTensor& o) const;
    HipTensor div(const HipTensor& o) const;
    HipTensor add_scalar(float s) const;  // lib.rs:916-922
    HipTensor mul_scalar(float s) const;  // lib.rs:925-932
    HipTensor neg() const;                // lib.rs:895-902
    HipTensor abs() const;                // lib.rs:822-828
    HipTensor sqrt() const;               // lib.rs:768-775 (correctly rounded)
    HipTensor exp() const;                // lib.rs:777-784 (device libm: within a few ulp)
    HipTensor log() const;                // lib.rs:786-793
    HipTensor sin() const;                // lib.rs:795-801
    HipTensor cos() const;                // lib.rs:803-809
    float to_scalar() const;              // lib.rs:966-974: one element, else InvalidInput
    static HipTensor from_scalar(float value, Shape shape, int device = 0);  // lib.rs:904-914
    static HipTensor eye(size_t n, int device = 0);                          // lib.rs:1303-1323
    // ---- TensorActivation (tensor.rs:191-209)
    HipTensor silu() const;     // x / (1 + exp(-x)), lib.rs:1154-1170
    HipTensor sigmoid() const;  // lib.rs:1172-1178
    // ---- TensorReduce::mean (lib.rs:995-1010): dims (all when null) are removed one by one in
    // reverse order of the list (keepdim is ignored, as in the reference), each by ndarray's
    // mean_axis with its summation order (bit-exact).
    HipTensor mean(const std::vector<size_t>* dims = nullptr, bool keepdim = false) const;
    // ---- TensorBroadcast::broadcast_to (lib.rs:1352-1518; other ranks through the generic
    // index map of lib.rs:511-560, reproduced as written)
    HipTensor broadcast_to(const Shape& shape) const;
    // ---- Tensor shape operations (tensor.rs:7-59): exact copies
    HipTensor transpose(size_t dim0, size_t dim1) const;  // lib.rs:115-137 (materialised)
    HipTensor slice(const std::vector<size_t>& start, const std::vector<size_t>& end) const;  // 2-D, lib.rs:139-183
    static HipTensor cat(const std::vector<HipTensor>& ts, size_t dim);    // 1-D, lib.rs:185-252
    // lib.rs:254-335: for 1..3-D inputs the data are concatenated in input order whatever `dim`,
    // and `dim` only places the count in the shape field; 0-D and >= 4-D inputs are placed by
    // the generic stack (lib.rs:390-467)
    static HipTensor stack(const std::vector<HipTensor>& ts, size_t dim);
    // lib.rs:84-91: to_owned() keeps the array's memory order, so the copy keeps its strides
    HipTensor contiguous() const { return clone(); }
    // lib.rs:80-82: the reference array's standard (row-major) layout
    bool is_contiguous() const;
    // The reference array's strides, in elements (row-major unless set).
    std::vector<int64_t> ref_strides() const;
    // Metadata only: records the strides the reference's array has after the operation that made
    // this tensor (row-major strides clear the record).
    void set_ref_strides(std::vector<int64_t> strides);

private:
    struct Buffer {
        void* ptr = nullptr;
        explicit Buffer(size_t bytes);
        ~Buffer();
        Buffer(const Buffer&) = delete;
        Buffer& operator=(const Buffer&) = delete;
    };
    std::shared_ptr<Buffer> buf_;
    Shape shape_;
    Storage storage_ = Storage::F32;
    int device_ = 0;
    std::vector<int64_t> strides_;  // the reference array's strides; empty = row-major
};

// ----------------------------------------------------------------------------- nn
// nn::Linear (lib.rs:53-134): weight [out, in] ~ N(0, sqrt(2/in)), bias zeros; y = x . W^T + b.
class Linear {
public:
    Linear(size_t in_features, size_t out_features, Rng& rng, int device = 0);
    Linear(HipTensor weight, HipTensor bias) : weight_(std::move(weight)), bias_(std::move(bias)) {}
    HipTensor forward(const HipTensor& x) const;             // fp32, [rows, in]
    HipTensor forward_silu(const HipTensor& x) const;        // silu(x . W^T + b), one launch
    const HipTensor& weight() const { return weight_; }
    const HipTensor& bias() const { return bias_; }

private:
    HipTensor weight_, bias_;
};

// nn::RMSNorm (lib.rs:219-285): weight ones; y = x / sqrt(mean(x^2) + eps) * w over the last dim.
class RMSNorm {
public:
    RMSNorm(size_t d_model, float eps, int device = 0);
    HipTensor forward(const HipTensor& x, Storage out = Storage::F32) const;
    HipTensor& weight() { return weight_; }
    float eps() const { return eps_; }

private:
    HipTensor weight_;
    float eps_;
};

// Exported nn::MambaBlock (lib.rs:846-906): forward = out_proj(silu(gate(x))).
class MambaBlock {
public:
    MambaBlock(size_t d_model, size_t d_state, size_t d_conv, size_t expand, Rng& rng, int device = 0);
    HipTensor forward(const HipTensor& x) const;  // x [seq_len, d_model] fp32
    const Linear& gate() const { return gate_; }
    const Linear& out_proj() const { return out_proj_; }

private:
    Linear gate_, out_proj_;
};

// nn::ssm::S4Block (ssm.rs:37-186): shared-state S4 recurrence, dt = 0.1.
class S4Block {
public:
    S4Block(size_t d_model, size_t d_state, Rng& rng, int device = 0);
    // forward_ssm (ssm.rs:138-186): x [d_model, L] -> y with the reference's memory [L, d_model]
    // and shape field [d_model, L]. parallel = the time-parallel form (equal to rounding).
    // The block keeps discretize(dt)'s decay, computed on the host from A_real / A_imag, for the
    // buffers it was computed from, and a device workspace: forwards on one block must not run
    // concurrently from several threads, and after writing into A_real / A_imag in place (their
    // data() pointers) call parameters_changed(); assigning new tensors or restore() needs nothing.
    HipTensor forward_ssm(const HipTensor& x, const HipTensor* gate = nullptr,
                          bool parallel = false) const;
    // Drops the kept decay: the next forward_ssm discretizes A_real / A_imag again.
    void parameters_changed() { a_disc_ = HipTensor(); a_src_[0] = a_src_[1] = nullptr; }
    // Module::forward (ssm.rs:269-273) = forward_conv (ssm.rs:189-229) with compute_conv_kernel
    // (ssm.rs:232-251), written as the reference writes them over HipTensor ops, so every shape
    // gives the reference's result or error: input [batch, seq_len] (2-D slices), kernel
    // K_0 = C.B, K_k = C.(A_real^k).B through 2-D x 1-D products. As in the reference, no input
    // shape completes (the k = 1 product needs d_model == d_state, k = 2 is a 1-D x 1-D matmul,
    // the stack of K_0 [d, d] with K_1 [d] mismatches, and the L = 1 path reshapes a [1, 1]
    // slice to [d_model] then slices the 2-D kernel with one index); an input of rank < 2
    // (where the reference's unwrap panics) raises InvalidDimension.
    HipTensor forward(const HipTensor& x) const { return forward_conv(x); }
    HipTensor forward_conv(const HipTensor& x) const;
    // checkpoint()/restore() (ssm.rs:331-360): A_real, A_imag, B, C, D, delta, Lambda.
    std::vector<HipTensor> checkpoint() const;
    void restore(const std::vector<HipTensor>& ck);
    size_t d_model() const { return d_model_; }
    size_t d_state() const { return d_state_; }
    HipTensor A_real, A_imag, B, C, D, delta, Lambda;

private:
    size_t d_model_, d_state_;
    // discretize(dt)'s decay (hx_s4_discretize, host libm) for the A_real / A_imag buffers it was
    // computed from (identified by their addresses; parameters_changed() and restore() drop it)
    mutable HipTensor a_disc_;
    mutable const void* a_src_[2] = {nullptr, nullptr};
    mutable HipTensor workspace_;
};

// The exported nn::S4Block (crates/nn/src/lib.rs:674-773): A [d_state, d_state] ~ N(0, 0.1),
// B [d_state, d_model] ~ N(0, 0.1), C [d_model, d_state] ~ N(0, 0.1), D zeros [d_model], delta
// [d_model] ~ U(0.001, 0.1), Lambda [d_state] ~ N(0, 1) (lib.rs:687-726, in that draw order).
// forward = forward_ssm (lib.rs:770-772) returns its input unchanged (a clone, lib.rs:742-756):
// the README's S4 example. dim(0) and dim(1) are read first, so an input of rank < 2 (a panic
// in the reference) raises InvalidDimension.
class ExportedS4Block {
public:
    ExportedS4Block(size_t d_model, size_t d_state, Rng& rng, int device = 0);
    HipTensor forward_ssm(const HipTensor& x) const;
    HipTensor forward(const HipTensor& x) const { return forward_ssm(x); }
    std::vector<const HipTensor*> parameters() const { return {&A, &B, &C, &D, &delta, &Lambda}; }
    size_t d_model() const { return d_model_; }
    size_t d_state() const { return d_state_; }
    HipTensor A, B, C, D, delta, Lambda;

private:
    size_t d_model_, d_state_;
};

// The reference's nn code over the HipTensor primitives alone, each written as the reference
// writes it (the generic Module<T> bodies instantiated for T = HipTensor, no fused kernel):
//   linear       Linear::forward (lib.rs:120-134): x.matmul(W.transpose(0,1)) + broadcast(bias)
//   mamba_mlp    exported MambaBlock::forward_mamba (lib.rs:888-906): linear -> silu -> linear
//   rmsnorm      RMSNorm::forward (lib.rs:258-285) with eps' = eps (the reference draws
//                U[eps, eps + 1e-8) per row)
//   s4_forward_ssm  ssm::S4Block::discretize + forward_ssm (ssm.rs:103-186): per-step slices,
//                GEMVs and stack(., 1)
// They show the primitives are a complete drop-in; the fused entry points are the fast path.
namespace generic {
HipTensor linear(const HipTensor& x, const HipTensor& weight, const HipTensor* bias);
HipTensor mamba_mlp(const HipTensor& x, const Linear& gate, const Linear& out_proj);
HipTensor rmsnorm(const HipTensor& x, const HipTensor& weight, float eps);
HipTensor s4_forward_ssm(const S4Block& s4, const HipTensor& x);
}  // namespace generic

// nn::ssm::MambaBlock::forward_mamba (ssm.rs:435-464): delta = X . delta_proj; y =
// S4.forward_ssm(delta) gated by `gate`. X must be [d_model, d_model] as in the reference.
class SsmMambaBlock {
public:
    SsmMambaBlock(size_t d_model, size_t d_state, Rng& rng, int device = 0);
    HipTensor forward_mamba(const HipTensor& x) const;
    S4Block s4;
    HipTensor delta_proj, B_proj, C_proj, gate;
};

// The selective Mamba block the exported MambaBlock's parameters describe (bf16 storage, fp32
// arithmetic): in_proj -> conv1d+SiLU -> x_proj -> dt_proj -> selective scan -> out_proj.
class MambaBlockFused {
public:
    MambaBlockFused(size_t d_model, size_t d_state, size_t d_conv, size_t expand, Rng& rng,
                    int device = 0, size_t dt_rank = 0);
    HipTensor forward(const HipTensor& x) const;  // x [batch, L, d_model] bf16
    size_t d_model, d_state, d_conv, d_inner, dt_rank;
    HipTensor w_in, conv_w, conv_b, w_x, w_dt, dt_bias, A, D, w_out;

private:
    mutable HipTensor workspace_;
};

// Fused selective scan on HipTensors (hx_selective_scan_fwd).
HipTensor selective_scan(const HipTensor& u, const HipTensor& delta, const HipTensor& A,
                         const HipTensor& B, const HipTensor& C, const HipTensor* D,
                         const HipTensor* z, const HipTensor* dt_bias, bool softplus,
                         HipTensor* last_state = nullptr);

// ----------------------------------------------------------------------------- training
// CheckpointManager's file (training/src/checkpoint.rs:137-198): u32 big-endian metadata
// length, metadata JSON, bincode of Vec<CpuTensor>. The tensor bytes are those a CpuTensor with
// the same values writes (device Cpu, dtype F32), so files move between the two backends.
struct HostTensor {
    std::vector<size_t> shape;
    std::vector<float> values;
};
std::vector<uint8_t> encode_params(const std::vector<HostTensor>& params);
std::vector<HostTensor> decode_params(const std::vector<uint8_t>& bytes);
void save_checkpoint(const std::string& path, const std::string& metadata_json,
                     const std::vector<HostTensor>& params);
std::pair<std::string, std::vector<HostTensor>> load_checkpoint_host(const std::string& path);
// HipTensor forms (device <-> host copies around the above)
void save_checkpoint(const std::string& path, const std::string& metadata_json,
                     const std::vector<HipTensor>& params);
std::pair<std::string, std::vector<HipTensor>> load_checkpoint(const std::string& path,
                                                               int device = 0);

// ----------------------------------------------------------------------------- hal
// hal::DeviceType and DataType (hal/src/device.rs:8-100) in the reference's declaration order.
enum class DeviceType { CPU, CUDA, Metal, ROCm, NPU, TPU, QPU, BCI };
enum class DataType { I8, I16, I32, I64, U8, U16, U32, U64, F16, F32, F64, BF8, BF16, C32, C64, Bool };
// hal::OperationType (hal/src/device.rs:129-210), every variant in the reference's order.
enum class OperationType {
    Add, Sub, Mul, Div, Pow, Sqrt, Abs,
    Sin, Cos, Tan, Asin, Acos, Atan,
    Exp, Log, Log2, Log10,
    MatMul, Transpose, Inverse, Determinant, Eigenvalues, SVD,
    Conv1D, Conv2D, Conv3D, MaxPool, AvgPool,
    FFT, IFFT, RFFT, IRFFT,
    Sum, Mean, Max, Min, Var, Std,
    ReLU, Sigmoid, Tanh, SiLU, GELU, Softmax,
    SSMForward, SSMBackward, StateUpdate,
    TopologicalAnalysis, MotifDetection, CycleDetection, StabilityCalculation,
    QuantumGate, QuantumMeasurement, QuantumEntanglement,
    SpikeEncoding, SpikeDecoding, SignalFiltering,
};
const char* operation_name(OperationType op);  // the variant's name (Debug formatting)

// hal::MemoryHandle (hal/src/memory.rs:11-24).
struct MemoryHandle {
    uint64_t id = 0;
    DeviceType device = DeviceType::ROCm;
    size_t size = 0;  // bytes
    DataType dtype = DataType::F32;
    uintptr_t address = 0;
    std::vector<size_t> shape;  // logical shape of the buffer (empty: size / element bytes, 1-D)
};

// hal::Operation (hal/src/operations.rs:9-28): type, inputs, output, numeric parameters.
struct Operation {
    OperationType op_type;
    std::vector<MemoryHandle> inputs;
    MemoryHandle* output = nullptr;  // optional output: used as the destination when it has memory
                                     // (address != 0); its id names the result in a ComputeGraph
    std::map<std::string, double> params;
    explicit Operation(OperationType t) : op_type(t) {}
};

// hal::ComputeGraph (hal/src/operations.rs:88-231): nodes, dependency edges from -> to,
// build() finds input nodes (no incoming edge) and output nodes (no outgoing edge),
// topological_sort() is the reference's DFS (reverse post-order) and raises on a cycle.
class ComputeGraph {
public:
    size_t add_operation(Operation op);
    void add_dependency(size_t from, size_t to);  // InvalidInput for an unknown node
    const std::vector<Operation>& nodes() const { return nodes_; }
    const std::vector<size_t>* dependencies(size_t node) const;
    void build();
    std::vector<size_t> topological_sort() const;
    const std::vector<size_t>& input_nodes() const { return inputs_; }
    const std::vector<size_t>& output_nodes() const { return outputs_; }

private:
    std::vector<Operation> nodes_;
    std::map<size_t, std::vector<size_t>> deps_;
    std::vector<size_t> inputs_, outputs_;
};

// hal::TopologicalFeatures / AsyncHandle (hal/src/backend.rs:73-123).
struct TopologicalFeatures {
    std::vector<uint64_t> motif_hashes;
    std::vector<std::vector<size_t>> cycles;
    double stability = 0.0;
    double entropy = 0.0;
};
struct AsyncHandle {
    uint64_t id = 0;
    std::string device_id;
    OperationType operation = OperationType::Add;
};

struct DeviceCapabilities {
    DeviceType device_type = DeviceType::ROCm;
    std::string device_id;
    std::vector<OperationType> supported_operations;
    std::vector<DataType> supported_precisions;
    size_t compute_units = 0;
    size_t memory_bytes = 0;
    size_t available_memory = 0;
    double memory_bandwidth_gbs = 0.0;
    bool supports_async = true;
};

// hal::ComputeBackend (hal/src/backend.rs:13-70), every method of the trait.
class ComputeBackend {
public:
    virtual ~ComputeBackend() = default;
    virtual DeviceType device_type() const = 0;
    virtual std::string device_id() const = 0;
    virtual const DeviceCapabilities& capabilities() const = 0;
    virtual bool supports_operation(OperationType op) const = 0;
    virtual size_t optimal_batch_size() const = 0;
    virtual std::vector<DataType> supported_precisions() const = 0;
    virtual double memory_bandwidth() const = 0;
    virtual size_t compute_units() const = 0;
    virtual MemoryHandle allocate(size_t size, DataType dtype) = 0;
    virtual void deallocate(const MemoryHandle& h) = 0;
    virtual void copy_from_host(const MemoryHandle& dst, const void* src, size_t bytes) = 0;
    virtual void copy_to_host(void* dst, const MemoryHandle& src, size_t bytes) const = 0;
    virtual MemoryHandle copy_to(const MemoryHandle& src, ComputeBackend& dst) = 0;
    virtual MemoryHandle execute_op(const Operation& op) = 0;
    virtual std::vector<MemoryHandle> execute_graph(const ComputeGraph& graph) = 0;
    virtual TopologicalFeatures compute_topological_features(const MemoryHandle& data) = 0;
    virtual AsyncHandle execute_async(const Operation& op) = 0;
    virtual MemoryHandle wait(const AsyncHandle& h) = 0;
    virtual bool is_available() const = 0;
    virtual double utilization() const = 0;
    virtual void synchronize() = 0;
};

// ComputeBackend for one ROCm device. execute_op runs on the device:
//   Add/Sub/Mul/Div (2 equal-size inputs), Sqrt/Abs/Sin/Cos/Exp/Log/Sigmoid/SiLU (1 input),
//   Mean (all elements -> 1), Transpose (2-D, shape from the input handle), MatMul (a [M,K],
//   b [K,N] from the handles' shapes), SSMForward (u, delta, A, B, C[, D, z, dt_bias]; params
//   batch, seqlen, dim, dstate, softplus), StateUpdate (state, u, delta, A, B, C[, D, z,
//   dt_bias]; params batch, dim, dstate, softplus). Others: UnsupportedOperation.
// execute_async launches the operation on the device stream and returns at once; wait() blocks
// until it has finished and returns its output. execute_graph runs the nodes in topological
// order, feeding a node's output to the nodes whose inputs carry that output's id, and returns
// the outputs of the output nodes (the reference's substitution rule, operations.rs + the CPU
// backend's execute_graph). utilization() reads the device's busy percentage from sysfs.
class RocmBackend : public ComputeBackend {
public:
    explicit RocmBackend(int device = 0);
    ~RocmBackend() override;
    DeviceType device_type() const override { return DeviceType::ROCm; }
    std::string device_id() const override;
    const DeviceCapabilities& capabilities() const override { return caps_; }
    bool supports_operation(OperationType op) const override;
    size_t optimal_batch_size() const override;
    std::vector<DataType> supported_precisions() const override { return caps_.supported_precisions; }
    double memory_bandwidth() const override { return caps_.memory_bandwidth_gbs; }
    size_t compute_units() const override { return caps_.compute_units; }
    MemoryHandle allocate(size_t size, DataType dtype) override;
    void deallocate(const MemoryHandle& h) override;
    void copy_from_host(const MemoryHandle& dst, const void* src, size_t bytes) override;
    void copy_to_host(void* dst, const MemoryHandle& src, size_t bytes) const override;
    MemoryHandle copy_to(const MemoryHandle& src, ComputeBackend& dst) override;
    MemoryHandle execute_op(const Operation& op) override;
    std::vector<MemoryHandle> execute_graph(const ComputeGraph& graph) override;
    TopologicalFeatures compute_topological_features(const MemoryHandle& data) override;
    AsyncHandle execute_async(const Operation& op) override;
    MemoryHandle wait(const AsyncHandle& h) override;
    bool is_available() const override;
    double utilization() const override;
    void synchronize() override;

private:
    // device scratch of the scan's time segments, kept between SSMForward operations and
    // grown on demand (operations of one backend run in order on the default stream)
    void* scan_workspace(size_t bytes);
    int device_;
    DeviceCapabilities caps_;
    uint64_t next_id_ = 1;
    std::map<uint64_t, void*> live_;
    std::map<uint64_t, MemoryHandle> pending_;  // execute_async outputs by handle id
    void* scan_ws_ = nullptr;
    size_t scan_ws_bytes_ = 0;
};

// Host-side check of an operation's inputs against what RocmBackend::execute_op would touch:
// every input handle that is read must have a device address and hold the bytes the operation
// reads (element counts from its shape, else its size), dtypes must be what the kernels take
// (F32 for the elementwise ops, Mean, Transpose and MatMul; for SSMForward / StateUpdate the
// storage type of u, F32 or BF16, shared by delta, B, C and z, with A, D, dt_bias and the state
// F32), and size parameters must be non-negative integers. Throws the reference's TensorError
// variants (InvalidInput, DTypeMismatch, ShapeMismatch, UnsupportedOperation); launches
// nothing. execute_op calls it first. The reference's CPU backend clamps to the smallest
// handle instead (backend-cpu/src/cpu_backend.rs); a device backend cannot read past a buffer.
void validate_operation(const Operation& op);

}  // namespace helix

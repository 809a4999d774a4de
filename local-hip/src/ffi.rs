// Raw declarations of liblocal_hip.so.  GENERATED by gen_ffi.py from include/local_hip.h: do not edit.
// One item per LH_API function of the header, same order, same argument names.
#![allow(non_camel_case_types, dead_code)]
use core::ffi::{c_char, c_int, c_void};

#[repr(C)] pub struct lh_context { _private: [u8; 0] }
#[repr(C)] pub struct lh_buffer { _private: [u8; 0] }
#[repr(C)] pub struct lh_batch { _private: [u8; 0] }
#[repr(C)] pub struct lh_event { _private: [u8; 0] }
#[repr(C)] pub struct lh_graph { _private: [u8; 0] }

#[repr(C)] #[derive(Clone, Copy, Debug, PartialEq, Eq)]
pub enum lh_dtype { LH_F16 = 0, LH_F32 = 1, LH_BF16 = 2 }
#[repr(C)] #[derive(Clone, Copy, Debug, PartialEq, Eq)]
pub enum lh_quant { LH_Q4_0 = 0, LH_TQ2_0 = 1 }
#[repr(C)] #[derive(Clone, Copy, Debug, PartialEq, Eq)]
pub enum lh_prologue { LH_PROLOGUE_RMS_NORM = 1, LH_PROLOGUE_GELU_MUL = 2 }

// lh_status values (local-metal/src/error.rs:1-32); every fallible call returns one as c_int.
pub const LH_OK: c_int = 0;
pub const LH_ERR_NO_DEVICE: c_int = 1;
pub const LH_ERR_NO_COMMAND_QUEUE: c_int = 2;
pub const LH_ERR_BUFFER_ALLOCATION: c_int = 3;
pub const LH_ERR_LIBRARY_CREATION: c_int = 4;
pub const LH_ERR_PIPELINE_CREATION: c_int = 5;
pub const LH_ERR_SHADER_NOT_FOUND: c_int = 6;
pub const LH_ERR_COMMAND_BUFFER: c_int = 7;
pub const LH_ERR_INVALID_ARGUMENT: c_int = 8;
pub const LH_ERR_IO: c_int = 9;
pub const LH_ROWS_F16: c_int = 2;
pub const LH_TQ_SEED: u64 = 0x7459C0DE;
pub const LH_DEFAULT_KV_BITS: c_int = 2;
pub const LH_ACT_NONE: c_int = 0;
pub const LH_ACT_SILU: c_int = 1;
pub const LH_ACT_GELU_TANH: c_int = 2;
pub const LH_ACT_RELU_SQUARED: c_int = 3;
pub const LH_ACT_SIGMOID: c_int = 4;
pub const LH_ACT_SILU_PAIRS: c_int = 5;
pub const LH_ROWS: c_int = 0;
pub const LH_ROWS_AT_POSITION: c_int = 1;
pub const LH_BLOCKS_AT_POSITION: c_int = 2;
pub const LH_ROWS_F32: c_int = 3;

#[link(name = "local_hip")]
extern "C" {
    pub fn lh_last_error() -> *const c_char;
    pub fn lh_version() -> *const c_char;
    pub fn lh_context_create(device_index: c_int, out: *mut *mut lh_context) -> c_int;
    pub fn lh_context_destroy(ctx: *mut lh_context);
    pub fn lh_context_device_name(ctx: *const lh_context, dst: *mut c_char, dst_len: usize) -> c_int;
    pub fn lh_context_compute_units(ctx: *const lh_context) -> c_int;
    pub fn lh_context_stream(ctx: *const lh_context) -> *mut c_void;
    pub fn lh_context_synchronize(ctx: *mut lh_context) -> c_int;
    pub fn lh_event_create(ctx: *mut lh_context, out: *mut *mut lh_event) -> c_int;
    pub fn lh_event_destroy(ev: *mut lh_event);
    pub fn lh_event_record(ev: *mut lh_event) -> c_int;
    pub fn lh_event_elapsed_ms(start: *mut lh_event, stop: *mut lh_event, ms: *mut f32) -> c_int;
    pub fn lh_buffer_from_bytes(ctx: *mut lh_context, src: *const c_void, len: usize, out: *mut *mut lh_buffer) -> c_int;
    pub fn lh_buffer_empty(ctx: *mut lh_context, len: usize, out: *mut *mut lh_buffer) -> c_int;
    pub fn lh_buffer_pinned(ctx: *mut lh_context, len: usize, out: *mut *mut lh_buffer) -> c_int;
    pub fn lh_buffer_view(parent: *mut lh_buffer, offset: usize, len: usize, out: *mut *mut lh_buffer) -> c_int;
    pub fn lh_buffer_wrap(ctx: *mut lh_context, device_ptr: *mut c_void, len: usize, out: *mut *mut lh_buffer) -> c_int;
    pub fn lh_buffer_free(buf: *mut lh_buffer);
    pub fn lh_buffer_length(buf: *const lh_buffer) -> usize;
    pub fn lh_buffer_device_ptr(buf: *const lh_buffer) -> *mut c_void;
    pub fn lh_buffer_write(buf: *mut lh_buffer, offset: usize, src: *const c_void, len: usize) -> c_int;
    pub fn lh_buffer_read(buf: *const lh_buffer, offset: usize, dst: *mut c_void, len: usize) -> c_int;
    pub fn lh_buffer_fill_zero(buf: *mut lh_buffer) -> c_int;
    pub fn lh_batch_new(ctx: *mut lh_context, out: *mut *mut lh_batch) -> c_int;
    pub fn lh_batch_free(batch: *mut lh_batch);
    pub fn lh_batch_dispatch_count(batch: *const lh_batch) -> u32;
    pub fn lh_batch_blit_copy(batch: *mut lh_batch, src: *const lh_buffer, src_offset: usize, dst: *mut lh_buffer, dst_offset: usize, len: usize) -> c_int;
    pub fn lh_batch_write(batch: *mut lh_batch, dst: *mut lh_buffer, offset: usize, src: *const c_void, len: usize) -> c_int;
    pub fn lh_batch_commit_and_wait(batch: *mut lh_batch) -> c_int;
    pub fn lh_debug_set_tq2_split_spin_limit(polls: u32);
    pub fn lh_debug_set_attention_pair_spin_limit(polls: u32);
    pub fn lh_batch_submit_and_renew(batch: *mut lh_batch) -> c_int;
    pub fn lh_batch_commit_and_renew(batch: *mut lh_batch) -> c_int;
    pub fn lh_batch_begin_capture(batch: *mut lh_batch) -> c_int;
    pub fn lh_batch_end_capture(batch: *mut lh_batch, out: *mut *mut lh_graph) -> c_int;
    pub fn lh_graph_launch(graph: *mut lh_graph) -> c_int;
    pub fn lh_graph_dispatch_count(graph: *const lh_graph) -> u32;
    pub fn lh_graph_free(graph: *mut lh_graph);
    pub fn lh_matvec_q4_0(ctx: *mut lh_context, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_q4_0_into(batch: *mut lh_batch, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_q4_0_f32out(ctx: *mut lh_context, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_q4_0_f32out_into(batch: *mut lh_batch, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_q4_0_copied_into(batch: *mut lh_batch, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, copy: *mut lh_buffer, rows: u32, cols: u32, cap: f32) -> c_int;
    pub fn lh_matvec_tq2_0(ctx: *mut lh_context, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_tq2_0_into(batch: *mut lh_batch, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_tq2_0_f32out(ctx: *mut lh_context, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_tq2_0_f32out_into(batch: *mut lh_batch, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_tq2_0_soa_into(batch: *mut lh_batch, qs: *const lh_buffer, scales: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_quant_typed_into(batch: *mut lh_batch, fmt: lh_quant, matrix: *const lh_buffer, vector: *const lh_buffer, vector_dtype: lh_dtype, output: *mut lh_buffer, output_dtype: lh_dtype, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_quant_grouped_into(batch: *mut lh_batch, fmt: lh_quant, count: u32, matrices: *const *const lh_buffer, vectors: *const *const lh_buffer, vector_dtype: lh_dtype, outputs: *const *mut lh_buffer, output_dtype: lh_dtype, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_quant_norm_chain_into(batch: *mut lh_batch, fmt: lh_quant, count: u32, matrices: *const *const lh_buffer, vector: *const lh_buffer, weight: *const lh_buffer, residual: *const lh_buffer, next_weight: *const lh_buffer, store: *mut lh_buffer, eps: f32, outputs: *const *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_quant_norm_chain_gelu_into(batch: *mut lh_batch, fmt: lh_quant, gate: *const lh_buffer, up: *const lh_buffer, factor: *const lh_buffer, vector: *const lh_buffer, weight: *const lh_buffer, residual: *const lh_buffer, next_weight: *const lh_buffer, store: *mut lh_buffer, eps: f32, out: *mut lh_buffer, up_out: *mut lh_buffer, rows: u32, cols: u32, applied: *mut c_int) -> c_int;
    pub fn lh_matvec_quant_norm_chain_tail_into(batch: *mut lh_batch, fmt: lh_quant, count: u32, matrices: *const *const lh_buffer, vector: *const lh_buffer, weight: *const lh_buffer, residual: *const lh_buffer, apply_scale: c_int, scale: f32, next_weight: *const lh_buffer, store: *mut lh_buffer, eps: f32, outputs: *const *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_quant_rotated_into(batch: *mut lh_batch, fmt: lh_quant, matrix: *const lh_buffer, vector: *const lh_buffer, signs: *const lh_buffer, head_dim: u32, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_quant_fused_into(batch: *mut lh_batch, fmt: lh_quant, count: u32, matrices: *const *const lh_buffer, vector: *const lh_buffer, prologue: c_int, aux: *const lh_buffer, eps: f32, outputs: *const *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matmul_nt_q4_0_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, output: *mut lh_buffer, m: u32, k: u32, n: u32) -> c_int;
    pub fn lh_matmul_nt_tq2_0_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, output: *mut lh_buffer, m: u32, k: u32, n: u32) -> c_int;
    pub fn lh_multivec_nt_q4_0_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, output: *mut lh_buffer, m: u32, k: u32, n: u32) -> c_int;
    pub fn lh_multivec_nt_tq2_0_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, output: *mut lh_buffer, m: u32, k: u32, n: u32) -> c_int;
    pub fn lh_matmul_nt_quant_typed_into(batch: *mut lh_batch, fmt: lh_quant, input: *const lh_buffer, input_dtype: lh_dtype, weight: *const lh_buffer, output: *mut lh_buffer, output_dtype: lh_dtype, m: u32, k: u32, n: u32) -> c_int;
    pub fn lh_matmul_nt_quant_gelu_mul_into(batch: *mut lh_batch, fmt: lh_quant, input: *const lh_buffer, w_gate: *const lh_buffer, w_up: *const lh_buffer, output: *mut lh_buffer, m: u32, k: u32, n: u32) -> c_int;
    pub fn lh_matmul_nt_quant_gelu_mul_strided_into(batch: *mut lh_batch, fmt: lh_quant, input: *const lh_buffer, weight: *const lh_buffer, m: u32, k: u32, n: u32, gate_rows: *const lh_buffer, row_stride: u32, row_offset: u32, output: *mut lh_buffer) -> c_int;
    pub fn lh_matmul_nt_quant_capped_into(batch: *mut lh_batch, fmt: lh_quant, input: *const lh_buffer, input_dtype: lh_dtype, weight: *const lh_buffer, output: *mut lh_buffer, m: u32, k: u32, n: u32, cap: f32) -> c_int;
    pub fn lh_matmul_nt_quant_norm_into(batch: *mut lh_batch, fmt: lh_quant, input: *const lh_buffer, weight: *const lh_buffer, m: u32, k: u32, n: u32, norm_weight: *const lh_buffer, residual: *const lh_buffer, output: *mut lh_buffer, eps: f32, apply_scale: c_int, scale: f32, norm2_weight: *const lh_buffer, output2: *mut lh_buffer) -> c_int;
    pub fn lh_matmul_nt_quant_grouped_into(batch: *mut lh_batch, fmt: lh_quant, count: u32, input: *const lh_buffer, weights: *const *const lh_buffer, outputs: *const *mut lh_buffer, ns: *const u32, m: u32, k: u32) -> c_int;
    pub fn lh_matmul_nt_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, output: *mut lh_buffer, m: u32, k: u32, n: u32) -> c_int;
    pub fn lh_clipped_linear_tiled_nt_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, bias: *const lh_buffer, output: *mut lh_buffer, m: u32, k: u32, n: u32, input_min: f32, input_max: f32, output_min: f32, output_max: f32) -> c_int;
    pub fn lh_matvec(ctx: *mut lh_context, matrix: *const lh_buffer, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_offset_into(batch: *mut lh_batch, matrix: *const lh_buffer, matrix_offset: usize, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_f32out_offset(ctx: *mut lh_context, matrix: *const lh_buffer, matrix_offset: usize, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_f32out_offset_into(batch: *mut lh_batch, matrix: *const lh_buffer, matrix_offset: usize, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_f32in_offset(ctx: *mut lh_context, matrix: *const lh_buffer, matrix_offset: usize, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_matvec_f32in_offset_into(batch: *mut lh_batch, matrix: *const lh_buffer, matrix_offset: usize, vector: *const lh_buffer, output: *mut lh_buffer, rows: u32, cols: u32) -> c_int;
    pub fn lh_rms_norm_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, output: *mut lh_buffer, dim: u32, rows: u32, eps: f32) -> c_int;
    pub fn lh_rms_norm_add_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, residual: *const lh_buffer, output: *mut lh_buffer, dim: u32, rows: u32, eps: f32) -> c_int;
    pub fn lh_rms_norm_residual_scale_into(batch: *mut lh_batch, input: *const lh_buffer, weight: *const lh_buffer, residual: *const lh_buffer, output: *mut lh_buffer, dim: u32, rows: u32, eps: f32, apply_scale: c_int, scale: f32) -> c_int;
    pub fn lh_scale_rms_norm_residual_scale_into(batch: *mut lh_batch, before: f32, input: *const lh_buffer, weight: *const lh_buffer, residual: *const lh_buffer, output: *mut lh_buffer, dim: u32, rows: u32, eps: f32, scale: f32) -> c_int;
    pub fn lh_qk_norm_gpu_into(batch: *mut lh_batch, qk_data: *mut lh_buffer, weight: *const lh_buffer, head_dim: u32, num_heads: u32, eps: f32) -> c_int;
    pub fn lh_qk_norm_offset_into(batch: *mut lh_batch, qk_data: *mut lh_buffer, weight: *const lh_buffer, weight_offset: usize, head_dim: u32, num_heads: u32, eps: f32) -> c_int;
    pub fn lh_qk_norm_rope_available(head_dim: u32) -> c_int;
    pub fn lh_qk_norm_rope_into(batch: *mut lh_batch, input: *const lh_buffer, output: *mut lh_buffer, weight: *const lh_buffer, head_dim: u32, num_heads: u32, eps: f32, position: u32, theta: f32, partial_rotary_factor: f32) -> c_int;
    pub fn lh_rope_into(batch: *mut lh_batch, input: *const lh_buffer, output: *mut lh_buffer, head_dim: u32, position: u32, theta: f32, partial_rotary_factor: f32, num_heads: u32) -> c_int;
    pub fn lh_rope_batch_into(batch: *mut lh_batch, qk: *mut lh_buffer, start_pos: u32, theta: f32, head_dim: u32, num_heads: u32, seq_len: u32, partial_rotary_factor: f32) -> c_int;
    pub fn lh_rope_batch_decode_into(batch: *mut lh_batch, qk: *mut lh_buffer, positions: *const lh_buffer, theta: f32, head_dim: u32, num_heads: u32, seq_len: u32, partial_rotary_factor: f32) -> c_int;
    pub fn lh_gelu_mul_into(batch: *mut lh_batch, a: *const lh_buffer, b: *const lh_buffer, out: *mut lh_buffer, count: u32) -> c_int;
    pub fn lh_residual_add_into(batch: *mut lh_batch, a: *const lh_buffer, b: *const lh_buffer, output: *mut lh_buffer, count: u32) -> c_int;
    pub fn lh_scale_in_place_gpu_into(batch: *mut lh_batch, data: *mut lh_buffer, scalar: f32, count: u32) -> c_int;
    pub fn lh_gather_strided_f16_into(batch: *mut lh_batch, src: *const lh_buffer, dst: *mut lh_buffer, row_stride: u32, base_off: u32, pld: u32, n_rows: u32) -> c_int;
    pub fn lh_gelu_mul_strided_into(batch: *mut lh_batch, a: *const lh_buffer, b: *const lh_buffer, b_row_stride: u32, b_offset: u32, out: *mut lh_buffer, dim: u32, rows: u32) -> c_int;
    pub fn lh_logit_softcap_gpu_into(batch: *mut lh_batch, data: *mut lh_buffer, cap: f32, count: u32) -> c_int;
    pub fn lh_smallm_max_m() -> u32;
    pub fn lh_batchm_max_m() -> u32;
    pub fn lh_multivec_max_m() -> u32;
    pub fn lh_batchm_enabled() -> c_int;
    pub fn lh_mma_enabled() -> c_int;
    pub fn lh_smallm_enabled() -> c_int;
    pub fn lh_dequant_q4_0_into(batch: *mut lh_batch, data: *const lh_buffer, byte_offset: usize, output: *mut lh_buffer, num_elements: usize) -> c_int;
    pub fn lh_dequant_tq2_0_into(batch: *mut lh_batch, data: *const lh_buffer, byte_offset: usize, output: *mut lh_buffer, num_elements: usize) -> c_int;
    pub fn lh_dequant_scaled_into(batch: *mut lh_batch, fmt: lh_quant, data: *const lh_buffer, byte_offset: usize, output: *mut lh_buffer, num_elements: usize, scale: f32) -> c_int;
    pub fn lh_dequant_rows_into(batch: *mut lh_batch, fmt: c_int, table: *const lh_buffer, table_rows: u32, cols: u32, rows: *const lh_buffer, n_rows: u32, scale: f32, output: *mut lh_buffer) -> c_int;
    pub fn lh_tq2_dequant(ctx: *mut lh_context, packed: *const lh_buffer, scales: *const lh_buffer, output: *mut lh_buffer, num_elements: u32) -> c_int;
    pub fn lh_turboquant_levels(dim: u32, bits: u32, levels: *mut f32) -> c_int;
    pub fn lh_turboquant_signs(dim: u32, seed: u64, signs: *mut f32) -> c_int;
    pub fn lh_turboquant_code_bytes(dim: u32, bits: u32) -> u32;
    pub fn lh_swa_ring_capacity(window: usize, max_positions: usize) -> usize;
    pub fn lh_kv_bits_from_env() -> u32;
    pub fn lh_encode_kv_turboquant(ctx: *mut lh_context, input: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, packed: *mut lh_buffer, norms: *mut lh_buffer, head_dim: u32, n_kv_heads: u32, num_tokens: u32, bits: u32, position: u32, ring_capacity: u32) -> c_int;
    pub fn lh_encode_kv_turboquant_into(batch: *mut lh_batch, input: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, packed: *mut lh_buffer, norms: *mut lh_buffer, head_dim: u32, n_kv_heads: u32, num_tokens: u32, bits: u32, position: u32, ring_capacity: u32) -> c_int;
    pub fn lh_encode_kv_turboquant_batched_into(batch: *mut lh_batch, input: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, packed: *mut lh_buffer, norms: *mut lh_buffer, positions: *const lh_buffer, head_dim: u32, n_kv_heads: u32, lane_capacity: u32, bits: u32, n_lanes: u32, ring_capacity: u32) -> c_int;
    pub fn lh_dequantize_kv_turboquant(ctx: *mut lh_context, packed: *const lh_buffer, norms: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, output: *mut lh_buffer, head_dim: u32, n_kv_heads: u32, num_tokens: u32, bits: u32, token_start: u32, ring_capacity: u32) -> c_int;
    pub fn lh_dequantize_kv_turboquant_into(batch: *mut lh_batch, packed: *const lh_buffer, norms: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, output: *mut lh_buffer, head_dim: u32, n_kv_heads: u32, num_tokens: u32, bits: u32, token_start: u32, ring_capacity: u32) -> c_int;
    pub fn lh_decode_qkv_prepare_into(batch: *mut lh_batch, q: *mut lh_buffer, k: *mut lh_buffer, v: *mut lh_buffer, q_norm: *const lh_buffer, k_norm: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, rq: *mut lh_buffer, k_codes: *mut lh_buffer, k_norms: *mut lh_buffer, v_codes: *mut lh_buffer, v_norms: *mut lh_buffer, head_dim: u32, n_q_heads: u32, n_kv_heads: u32, eps: f32, position: u32, theta: f32, partial_rotary_factor: f32, bits: u32, ring_capacity: u32) -> c_int;
    pub fn lh_decode_qkv_prepare_rows_into(batch: *mut lh_batch, q: *mut lh_buffer, k: *mut lh_buffer, v: *mut lh_buffer, q_norm: *const lh_buffer, k_norm: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, rq: *mut lh_buffer, k_codes: *mut lh_buffer, k_norms: *mut lh_buffer, v_codes: *mut lh_buffer, v_norms: *mut lh_buffer, positions: *const lh_buffer, head_dim: u32, n_q_heads: u32, n_kv_heads: u32, rows: u32, eps: f32, start_position: u32, theta: f32, partial_rotary_factor: f32, bits: u32, ring_capacity: u32, lane_capacity: u32) -> c_int;
    pub fn lh_matmul_nt_qkv_prepare_rows_into(batch: *mut lh_batch, fmt: lh_quant, input: *const lh_buffer, w_q: *const lh_buffer, w_k: *const lh_buffer, w_v: *const lh_buffer, k_dim: u32, q: *mut lh_buffer, k: *mut lh_buffer, v: *mut lh_buffer, q_norm: *const lh_buffer, k_norm: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, rq: *mut lh_buffer, k_codes: *mut lh_buffer, k_norms: *mut lh_buffer, v_codes: *mut lh_buffer, v_norms: *mut lh_buffer, positions: *const lh_buffer, head_dim: u32, n_q_heads: u32, n_kv_heads: u32, rows: u32, eps: f32, start_position: u32, theta: f32, partial_rotary_factor: f32, bits: u32, ring_capacity: u32, lane_capacity: u32) -> c_int;
    pub fn lh_matmul_nt_q_prepare_rows_into(batch: *mut lh_batch, fmt: lh_quant, input: *const lh_buffer, w_q: *const lh_buffer, k_dim: u32, q: *mut lh_buffer, q_norm: *const lh_buffer, signs: *const lh_buffer, rq: *mut lh_buffer, positions: *const lh_buffer, head_dim: u32, n_q_heads: u32, rows: u32, eps: f32, start_position: u32, theta: f32, partial_rotary_factor: f32, lane_capacity: u32) -> c_int;
    pub fn lh_hadamard_rotate_into(batch: *mut lh_batch, input: *const lh_buffer, signs: *const lh_buffer, output: *mut lh_buffer, head_dim: u32, num_heads: u32, pre_sign: c_int, post_sign: c_int) -> c_int;
    pub fn lh_hadamard_rotate_hf_into(batch: *mut lh_batch, input: *const lh_buffer, signs: *const lh_buffer, output: *mut lh_buffer, head_dim: u32, num_heads: u32, pre_sign: c_int, post_sign: c_int) -> c_int;
    pub fn lh_hadamard_rotate_fh_into(batch: *mut lh_batch, input: *const lh_buffer, signs: *const lh_buffer, output: *mut lh_buffer, head_dim: u32, num_heads: u32, pre_sign: c_int, post_sign: c_int) -> c_int;
    pub fn lh_flash_attention_tq_into(batch: *mut lh_batch, rq: *const lh_buffer, k_codes: *const lh_buffer, k_norms: *const lh_buffer, v_codes: *const lh_buffer, v_norms: *const lh_buffer, levels: *const lh_buffer, out: *mut lh_buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> c_int;
    pub fn lh_flash_attention_tq_static_into(batch: *mut lh_batch, rq: *const lh_buffer, k_codes: *const lh_buffer, k_norms: *const lh_buffer, v_codes: *const lh_buffer, v_norms: *const lh_buffer, levels: *const lh_buffer, out: *mut lh_buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> c_int;
    pub fn lh_flash_attention_tq_prefill_into(batch: *mut lh_batch, rq: *const lh_buffer, k_codes: *const lh_buffer, k_norms: *const lh_buffer, v_codes: *const lh_buffer, v_norms: *const lh_buffer, levels: *const lh_buffer, out: *mut lh_buffer, head_dim: u32, kv_len: u32, start_pos: u32, n_rows: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> c_int;
    pub fn lh_flash_attention_tq_prefill_tiled_into(batch: *mut lh_batch, rq: *const lh_buffer, k_codes: *const lh_buffer, k_norms: *const lh_buffer, v_codes: *const lh_buffer, v_norms: *const lh_buffer, levels: *const lh_buffer, out: *mut lh_buffer, head_dim: u32, kv_len: u32, start_pos: u32, n_rows: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> c_int;
    pub fn lh_flash_attention_tq_batched_into(batch: *mut lh_batch, rq: *const lh_buffer, k_codes: *const lh_buffer, k_norms: *const lh_buffer, v_codes: *const lh_buffer, v_norms: *const lh_buffer, levels: *const lh_buffer, out: *mut lh_buffer, positions: *const lh_buffer, head_dim: u32, lane_capacity: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, n_lanes: u32, ring_capacity: u32) -> c_int;
    pub fn lh_flash_attention_tq_rotated_into(batch: *mut lh_batch, rq: *const lh_buffer, k_codes: *const lh_buffer, k_norms: *const lh_buffer, v_codes: *const lh_buffer, v_norms: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, out: *mut lh_buffer, out_f16: *mut lh_buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> c_int;
    pub fn lh_flash_attention_tq_rotated_lazy_into(batch: *mut lh_batch, rq: *const lh_buffer, k_codes: *const lh_buffer, k_norms: *const lh_buffer, v_codes: *const lh_buffer, v_norms: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, out: *mut lh_buffer, out_f16: *mut lh_buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32, rotated: *mut c_int) -> c_int;
    pub fn lh_matmul_nt_qkv_attention_lanes_into(batch: *mut lh_batch, fmt: lh_quant, input: *const lh_buffer, w_q: *const lh_buffer, w_k: *const lh_buffer, w_v: *const lh_buffer, k_dim: u32, q: *mut lh_buffer, k: *mut lh_buffer, v: *mut lh_buffer, q_norm: *const lh_buffer, k_norm: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, rq: *mut lh_buffer, k_codes: *mut lh_buffer, k_norms: *mut lh_buffer, v_codes: *mut lh_buffer, v_norms: *mut lh_buffer, positions: *const lh_buffer, out: *mut lh_buffer, out_f16: *mut lh_buffer, head_dim: u32, n_q_heads: u32, n_kv_heads: u32, lanes: u32, eps: f32, theta: f32, partial_rotary_factor: f32, window: u32, bits: u32, ring_capacity: u32, lane_capacity: u32) -> c_int;
    pub fn lh_token_attention_tq_into(batch: *mut lh_batch, q_raw: *const lh_buffer, k_raw: *const lh_buffer, v_raw: *const lh_buffer, q: *mut lh_buffer, k: *mut lh_buffer, v: *mut lh_buffer, q_norm: *const lh_buffer, k_norm: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, rq: *mut lh_buffer, k_codes: *mut lh_buffer, k_norms: *mut lh_buffer, v_codes: *mut lh_buffer, v_norms: *mut lh_buffer, out: *mut lh_buffer, out_f16: *mut lh_buffer, head_dim: u32, num_q_heads: u32, num_kv_heads: u32, eps: f32, position: u32, theta: f32, partial_rotary_factor: f32, window: u32, bits: u32, ring_capacity: u32, rotated: *mut c_int) -> c_int;
    pub fn lh_flash_attention_tq_batched_rotated_into(batch: *mut lh_batch, rq: *const lh_buffer, k_codes: *const lh_buffer, k_norms: *const lh_buffer, v_codes: *const lh_buffer, v_norms: *const lh_buffer, levels: *const lh_buffer, signs: *const lh_buffer, out: *mut lh_buffer, out_f16: *mut lh_buffer, positions: *const lh_buffer, head_dim: u32, lane_capacity: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, n_lanes: u32, ring_capacity: u32) -> c_int;
    pub fn lh_flash_decoding_into(batch: *mut lh_batch, q: *const lh_buffer, k: *const lh_buffer, v: *const lh_buffer, output: *mut lh_buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32) -> c_int;
    pub fn lh_flash_attention_windowed_split_into(batch: *mut lh_batch, q: *const lh_buffer, k: *const lh_buffer, v: *const lh_buffer, output: *mut lh_buffer, partial_max: *mut lh_buffer, partial_sum: *mut lh_buffer, partial_acc: *mut lh_buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, num_splits: u32) -> c_int;
    pub fn lh_flash_split_count(eff_seq_len: u32) -> u32;
    pub fn lh_embed_rows_bf16_into(batch: *mut lh_batch, table: *const lh_buffer, table_rows: u32, cols: u32, rows: *const lh_buffer, n_rows: u32, output: *mut lh_buffer) -> c_int;
    pub fn lh_embed_token_bf16_into(batch: *mut lh_batch, table: *const lh_buffer, table_rows: u32, cols: u32, token: u32, position: u32, output: *mut lh_buffer, at: *mut lh_buffer, next: *mut lh_buffer) -> c_int;
    pub fn lh_norm_rows_f32_into(batch: *mut lh_batch, input: *const lh_buffer, add: *const lh_buffer, weight: *const lh_buffer, store: *mut lh_buffer, row_index: *const lh_buffer, output: *mut lh_buffer, output_dtype: c_int, dim: u32, rows: u32, eps: f32) -> c_int;
    pub fn lh_residual_rows_into(batch: *mut lh_batch, input: *const lh_buffer, branch: *const lh_buffer, weight: *const lh_buffer, store: *mut lh_buffer, output: *mut lh_buffer, output_dtype: c_int, dim: u32, rows: u32, eps: f32) -> c_int;
    pub fn lh_gated_norm_rows_into(batch: *mut lh_batch, input: *const lh_buffer, gate: *const lh_buffer, gate_act: u32, gate_first: c_int, weight: *const lh_buffer, output: *mut lh_buffer, dtype: c_int, dim: u32, group: u32, rows: u32, eps: f32) -> c_int;
    pub fn lh_softcap_f32_into(batch: *mut lh_batch, logits: *mut lh_buffer, n: usize, cap: f32) -> c_int;
    pub fn lh_linear_rows_into(batch: *mut lh_batch, input: *const lh_buffer, input_dtype: c_int, weight: *const lh_buffer, bias: *const lh_buffer, m: u32, k: u32, count: u32, ns: *const u32, acts: *const u32, heads: *const u32, padded: *const u32, layouts: *const u32, outputs: *const *mut lh_buffer, output_dtype: c_int, accumulate: c_int, position: *const lh_buffer) -> c_int;
    pub fn lh_linear_vector_into(batch: *mut lh_batch, input: *const lh_buffer, input_dtype: c_int, weight: *const lh_buffer, bias: *const lh_buffer, k: u32, count: u32, ns: *const u32, acts: *const u32, heads: *const u32, padded: *const u32, layouts: *const u32, outputs: *const *mut lh_buffer, output_dtype: c_int, accumulate: c_int, position: *const lh_buffer) -> c_int;
    pub fn lh_linear_norm_vector_into(batch: *mut lh_batch, input: *const lh_buffer, add: *const lh_buffer, store: *mut lh_buffer, norm_weight: *const lh_buffer, eps: f32, weight: *const lh_buffer, bias: *const lh_buffer, k: u32, count: u32, ns: *const u32, acts: *const u32, heads: *const u32, padded: *const u32, layouts: *const u32, outputs: *const *mut lh_buffer, output_dtype: c_int, accumulate: c_int, position: *const lh_buffer) -> c_int;
    pub fn lh_linear_norm_vector_capped_into(batch: *mut lh_batch, input: *const lh_buffer, norm_weight: *const lh_buffer, eps: f32, weight: *const lh_buffer, bias: *const lh_buffer, k: u32, n: u32, output: *mut lh_buffer, cap: f32) -> c_int;
    pub fn lh_linear_norm_vector_copied_into(batch: *mut lh_batch, input: *const lh_buffer, norm_weight: *const lh_buffer, eps: f32, weight: *const lh_buffer, bias: *const lh_buffer, k: u32, n: u32, output: *mut lh_buffer, copy: *mut lh_buffer, cap: f32) -> c_int;
    pub fn lh_linear_residual_norm_vector_copied_into(batch: *mut lh_batch, input: *mut lh_buffer, branch: *const lh_buffer, branch_weight: *const lh_buffer, branch_eps: f32, norm_weight: *const lh_buffer, eps: f32, weight: *const lh_buffer, bias: *const lh_buffer, k: u32, n: u32, output: *mut lh_buffer, copy: *mut lh_buffer, cap: f32) -> c_int;
    pub fn lh_linear_residual_vector_into(batch: *mut lh_batch, input: *const lh_buffer, branch: *const lh_buffer, store: *mut lh_buffer, norm_weight: *const lh_buffer, eps: f32, weight: *const lh_buffer, bias: *const lh_buffer, k: u32, count: u32, ns: *const u32, acts: *const u32, heads: *const u32, padded: *const u32, layouts: *const u32, outputs: *const *mut lh_buffer, output_dtype: c_int, accumulate: c_int, position: *const lh_buffer) -> c_int;
    pub fn lh_gated_vector_fits(k: u32, group: u32) -> u32;
    pub fn lh_linear_gated_vector_into(batch: *mut lh_batch, input: *const lh_buffer, gate: *const lh_buffer, gate_dtype: c_int, gate_act: u32, gate_first: c_int, norm_weight: *const lh_buffer, group: u32, eps: f32, weight: *const lh_buffer, bias: *const lh_buffer, k: u32, count: u32, ns: *const u32, acts: *const u32, heads: *const u32, padded: *const u32, layouts: *const u32, outputs: *const *mut lh_buffer, output_dtype: c_int, accumulate: c_int, position: *const lh_buffer) -> c_int;
    pub fn lh_attention_padded_dim(dim: u32) -> u32;
    pub fn lh_attention_padded_vdim(vdim: u32) -> u32;
    pub fn lh_attention_rows_into(batch: *mut lh_batch, q: *const lh_buffer, keys: *const lh_buffer, values: *const lh_buffer, output: *mut lh_buffer, dtype: c_int, position: *const lh_buffer, max_position: u32, rows: u32, heads: u32, kv_heads: u32, maps: u32, dim: u32, vdim: u32, capacity: u32, scale: f32, lambda: f32, out_scale: f32, eps: f32, sink: *const lh_buffer, gate: *const lh_buffer) -> c_int;
    pub fn lh_latent_padded_rank(rank: u32) -> u32;
    pub fn lh_latent_row(rank: u32, rot: u32) -> u32;
    pub fn lh_latent_prepare_into(batch: *mut lh_batch, q_rot: *const lh_buffer, down: *const lh_buffer, norm_weight: *const lh_buffer, frequencies: *const lh_buffer, position: *const lh_buffer, q: *mut lh_buffer, q_dtype: c_int, cache: *mut lh_buffer, dtype: c_int, rows: u32, heads: u32, rank: u32, rot: u32, q_ld: u32, rot_column: u32, clear_column: u32, capacity: u32, eps: f32) -> c_int;
    pub fn lh_head_linear_into(batch: *mut lh_batch, input: *const lh_buffer, dtype: c_int, weight: *const lh_buffer, output: *mut lh_buffer, output_dtype: c_int, rows: u32, heads: u32, n: u32, k: u32, output_ld: u32) -> c_int;
    pub fn lh_latent_expand_into(batch: *mut lh_batch, cache: *const lh_buffer, dtype: c_int, weight: *const lh_buffer, keys: *mut lh_buffer, values: *mut lh_buffer, positions: u32, heads: u32, dim: u32, rot: u32, vdim: u32, rank: u32) -> c_int;
    pub fn lh_latent_attention_rows_into(batch: *mut lh_batch, q: *const lh_buffer, cache: *const lh_buffer, output: *mut lh_buffer, dtype: c_int, position: *const lh_buffer, max_position: u32, rows: u32, heads: u32, rank: u32, rot: u32, capacity: u32, scale: f32, sink: *const lh_buffer, gate: *const lh_buffer) -> c_int;
    pub fn lh_latent_attention_values_into(batch: *mut lh_batch, q: *const lh_buffer, cache: *const lh_buffer, latent: *mut lh_buffer, dtype: c_int, position: *const lh_buffer, max_position: u32, rows: u32, heads: u32, rank: u32, rot: u32, capacity: u32, scale: f32, sink: *const lh_buffer, gate: *const lh_buffer, value_weight: *const lh_buffer, vdim: u32, output: *mut lh_buffer) -> c_int;
    pub fn lh_latent_queries_into(batch: *mut lh_batch, q: *const lh_buffer, key_weight: *const lh_buffer, q_rot: *const lh_buffer, down: *const lh_buffer, norm_weight: *const lh_buffer, frequencies: *const lh_buffer, position: *const lh_buffer, output: *mut lh_buffer, cache: *mut lh_buffer, dtype: c_int, rows: u32, heads: u32, dim: u32, rank: u32, rot: u32, capacity: u32, eps: f32) -> c_int;
    pub fn lh_linear_attention_padded_dim(dim: u32) -> u32;
    pub fn lh_linear_attention_workspace_bytes(rows: u32, heads: u32, dim: u32, vdim: u32) -> usize;
    pub fn lh_linear_attention_recurrent_into(batch: *mut lh_batch, q: *const lh_buffer, k: *const lh_buffer, v: *const lh_buffer, dtype: c_int, state: *mut lh_buffer, decay: *const lh_buffer, output: *mut lh_buffer, rows: u32, heads: u32, dim: u32, vdim: u32, scale: f32) -> c_int;
    pub fn lh_linear_attention_chunked_into(batch: *mut lh_batch, q: *const lh_buffer, k: *const lh_buffer, v: *const lh_buffer, state: *mut lh_buffer, decay_powers: *const lh_buffer, workspace: *mut lh_buffer, output: *mut lh_buffer, rows: u32, heads: u32, dim: u32, vdim: u32, scale: f32) -> c_int;
    pub fn lh_selective_steps_bytes(rows: u32, heads: u32) -> usize;
    pub fn lh_selective_conv_into(batch: *mut lh_batch, input: *const lh_buffer, dtype: c_int, ring: *mut lh_buffer, taps_weight: *const lh_buffer, bias: *const lh_buffer, position: *const lh_buffer, x: *mut lh_buffer, b: *mut lh_buffer, c: *mut lh_buffer, rows: u32, heads: u32, vdim: u32, groups: u32, state: u32, taps: u32) -> c_int;
    pub fn lh_selective_recurrent_into(batch: *mut lh_batch, x: *const lh_buffer, b: *const lh_buffer, c: *const lh_buffer, dtype: c_int, dt_raw: *const lh_buffer, dt_bias: *const lh_buffer, a_log: *const lh_buffer, skip: *const lh_buffer, memory: *mut lh_buffer, output: *mut lh_buffer, rows: u32, heads: u32, vdim: u32, groups: u32, state: u32) -> c_int;
    pub fn lh_selective_chunked_into(batch: *mut lh_batch, x: *const lh_buffer, b: *const lh_buffer, c: *const lh_buffer, dt_raw: *const lh_buffer, dt_bias: *const lh_buffer, a_log: *const lh_buffer, skip: *const lh_buffer, memory: *mut lh_buffer, steps: *mut lh_buffer, workspace: *mut lh_buffer, output: *mut lh_buffer, rows: u32, heads: u32, vdim: u32, groups: u32, state: u32) -> c_int;
    pub fn lh_selective_step_into(batch: *mut lh_batch, input: *const lh_buffer, ring: *mut lh_buffer, taps_weight: *const lh_buffer, bias: *const lh_buffer, position: *const lh_buffer, dt_raw: *const lh_buffer, dt_bias: *const lh_buffer, a_log: *const lh_buffer, skip: *const lh_buffer, memory: *mut lh_buffer, output: *mut lh_buffer, heads: u32, vdim: u32, groups: u32, state: u32, taps: u32) -> c_int;
    pub fn lh_moe_plan_words(rows: u32, experts: u32, top: u32) -> u32;
    pub fn lh_moe_route_into(batch: *mut lh_batch, logits: *const lh_buffer, plan: *mut lh_buffer, rows: u32, experts: u32, top: u32) -> c_int;
    pub fn lh_moe_up_into(batch: *mut lh_batch, input: *const lh_buffer, dtype: c_int, plan: *const lh_buffer, up: *const lh_buffer, hidden: *mut lh_buffer, rows: u32, experts: u32, top: u32, width: u32, ff: u32, act: u32) -> c_int;
    pub fn lh_moe_down_into(batch: *mut lh_batch, hidden: *const lh_buffer, dtype: c_int, plan: *const lh_buffer, down: *const lh_buffer, slots: *mut lh_buffer, residual: *mut lh_buffer, rows: u32, experts: u32, top: u32, width: u32, ff: u32) -> c_int;
    pub fn lh_moe_vector_up_into(batch: *mut lh_batch, input: *const lh_buffer, norm_weight: *const lh_buffer, eps: f32, logits: *const lh_buffer, up: *const lh_buffer, hidden: *mut lh_buffer, experts: u32, top: u32, width: u32, ff: u32, act: u32) -> c_int;
    pub fn lh_moe_vector_routed_up_into(batch: *mut lh_batch, input: *const lh_buffer, norm_weight: *const lh_buffer, eps: f32, router: *const lh_buffer, logits: *mut lh_buffer, up: *const lh_buffer, hidden: *mut lh_buffer, experts: u32, top: u32, width: u32, ff: u32, act: u32) -> c_int;
    pub fn lh_moe_vector_down_into(batch: *mut lh_batch, hidden: *const lh_buffer, logits: *const lh_buffer, down: *const lh_buffer, residual: *mut lh_buffer, experts: u32, top: u32, width: u32, ff: u32) -> c_int;
    pub fn lh_advance_position_into(batch: *mut lh_batch, position: *mut lh_buffer, by: u32) -> c_int;
    pub fn lh_argmax_rows_f32_into(batch: *mut lh_batch, logits: *const lh_buffer, index: *mut lh_buffer, rows: u32, n: u32) -> c_int;
    pub fn lh_argmax_advance_f32_into(batch: *mut lh_batch, logits: *const lh_buffer, index: *mut lh_buffer, n: u32, position: *mut lh_buffer, by: u32) -> c_int;
}

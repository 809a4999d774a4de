// The kernel-dispatch layer: `Kernels`, one method per operation of liblocal_hip.so, with the names and the argument
// order that local-engine calls on local-metal (local-metal/src/kernels.rs).  GENERATED by gen_safe.py from
// include/local_hip.h: do not edit.  Operations with host pointers and the helpers of the codec are wrapped by hand in lib.rs: lh_matvec_quant_norm_chain_gelu_into, lh_turboquant_levels, lh_turboquant_signs, lh_turboquant_code_bytes, lh_swa_ring_capacity, lh_flash_attention_tq_rotated_lazy_into, lh_token_attention_tq_into, lh_flash_split_count.
// Other host-side helpers are reached through `ffi`: lh_qk_norm_rope_available, lh_smallm_max_m, lh_batchm_max_m, lh_multivec_max_m, lh_batchm_enabled, lh_mma_enabled, lh_smallm_enabled, lh_kv_bits_from_env, lh_gated_vector_fits, lh_attention_padded_dim, lh_attention_padded_vdim, lh_latent_padded_rank, lh_latent_row, lh_linear_attention_padded_dim, lh_linear_attention_workspace_bytes, lh_selective_steps_bytes, lh_moe_plan_words.
use core::ffi::c_int;

use crate::batch::CommandBatch;
use crate::buffer::Buffer;
use crate::context::Context;
use crate::error::{check, Result};
use crate::ffi;

/// Stand-in for `local_metal::Kernels` (kernels.rs:116-219 builds ~95 Metal pipelines there; the HIP kernels are
/// linked into the library, so this type holds nothing and `new` cannot fail for a missing shader).
#[derive(Debug, Default, Clone, Copy)]
pub struct Kernels;

impl Kernels {
    /// `Kernels::new(ctx, library)` of the reference; the context only proves that a gfx950 device was opened.
    pub fn new(_ctx: &Context) -> Result<Self> {
        Ok(Kernels)
    }

    /// `lh_matvec_q4_0` (include/local_hip.h).
    pub fn matvec_q4_0(&self, ctx: &Context, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_q4_0(ctx.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_q4_0_into` (include/local_hip.h).
    pub fn matvec_q4_0_into(&self, batch: &mut CommandBatch, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_q4_0_into(batch.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_q4_0_f32out` (include/local_hip.h).
    pub fn matvec_q4_0_f32out(&self, ctx: &Context, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_q4_0_f32out(ctx.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_q4_0_f32out_into` (include/local_hip.h).
    pub fn matvec_q4_0_f32out_into(&self, batch: &mut CommandBatch, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_q4_0_f32out_into(batch.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_q4_0_copied_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matvec_q4_0_copied_into(&self, batch: &mut CommandBatch, matrix: &Buffer, vector: &Buffer, output: &Buffer, copy: &Buffer, rows: u32, cols: u32, cap: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_q4_0_copied_into(batch.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), copy.as_ptr(), rows, cols, cap) })
    }

    /// `lh_matvec_tq2_0` (include/local_hip.h).
    pub fn matvec_tq2_0(&self, ctx: &Context, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_tq2_0(ctx.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_tq2_0_into` (include/local_hip.h).
    pub fn matvec_tq2_0_into(&self, batch: &mut CommandBatch, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_tq2_0_into(batch.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_tq2_0_f32out` (include/local_hip.h).
    pub fn matvec_tq2_0_f32out(&self, ctx: &Context, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_tq2_0_f32out(ctx.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_tq2_0_f32out_into` (include/local_hip.h).
    pub fn matvec_tq2_0_f32out_into(&self, batch: &mut CommandBatch, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_tq2_0_f32out_into(batch.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_tq2_0_soa_into` (include/local_hip.h).
    pub fn matvec_tq2_0_soa_into(&self, batch: &mut CommandBatch, qs: &Buffer, scales: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_tq2_0_soa_into(batch.as_ptr(), qs.as_ptr(), scales.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_quant_typed_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matvec_quant_typed_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, matrix: &Buffer, vector: &Buffer, vector_dtype: ffi::lh_dtype, output: &Buffer, output_dtype: ffi::lh_dtype, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_quant_typed_into(batch.as_ptr(), fmt, matrix.as_ptr(), vector.as_ptr(), vector_dtype, output.as_ptr(), output_dtype, rows, cols) })
    }

    /// `lh_matvec_quant_grouped_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matvec_quant_grouped_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, count: u32, matrices: &[&Buffer], vectors: &[&Buffer], vector_dtype: ffi::lh_dtype, outputs: &[&Buffer], output_dtype: ffi::lh_dtype, rows: u32, cols: u32) -> Result<()> {
        let matrices_raw: Vec<*const ffi::lh_buffer> = matrices.iter().map(|b| b.as_ptr() as *const ffi::lh_buffer).collect();
        let vectors_raw: Vec<*const ffi::lh_buffer> = vectors.iter().map(|b| b.as_ptr() as *const ffi::lh_buffer).collect();
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_quant_grouped_into(batch.as_ptr(), fmt, count, matrices_raw.as_ptr(), vectors_raw.as_ptr(), vector_dtype, outputs_raw.as_ptr(), output_dtype, rows, cols) })
    }

    /// `lh_matvec_quant_norm_chain_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matvec_quant_norm_chain_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, count: u32, matrices: &[&Buffer], vector: &Buffer, weight: &Buffer, residual: &Buffer, next_weight: &Buffer, store: &Buffer, eps: f32, outputs: &[&Buffer], rows: u32, cols: u32) -> Result<()> {
        let matrices_raw: Vec<*const ffi::lh_buffer> = matrices.iter().map(|b| b.as_ptr() as *const ffi::lh_buffer).collect();
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_quant_norm_chain_into(batch.as_ptr(), fmt, count, matrices_raw.as_ptr(), vector.as_ptr(), weight.as_ptr(), residual.as_ptr(), next_weight.as_ptr(), store.as_ptr(), eps, outputs_raw.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_quant_norm_chain_tail_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matvec_quant_norm_chain_tail_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, count: u32, matrices: &[&Buffer], vector: &Buffer, weight: &Buffer, residual: &Buffer, apply_scale: c_int, scale: f32, next_weight: &Buffer, store: &Buffer, eps: f32, outputs: &[&Buffer], rows: u32, cols: u32) -> Result<()> {
        let matrices_raw: Vec<*const ffi::lh_buffer> = matrices.iter().map(|b| b.as_ptr() as *const ffi::lh_buffer).collect();
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_quant_norm_chain_tail_into(batch.as_ptr(), fmt, count, matrices_raw.as_ptr(), vector.as_ptr(), weight.as_ptr(), residual.as_ptr(), apply_scale, scale, next_weight.as_ptr(), store.as_ptr(), eps, outputs_raw.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_quant_rotated_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matvec_quant_rotated_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, matrix: &Buffer, vector: &Buffer, signs: &Buffer, head_dim: u32, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_quant_rotated_into(batch.as_ptr(), fmt, matrix.as_ptr(), vector.as_ptr(), signs.as_ptr(), head_dim, output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_quant_fused_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matvec_quant_fused_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, count: u32, matrices: &[&Buffer], vector: &Buffer, prologue: c_int, aux: &Buffer, eps: f32, outputs: &[&Buffer], rows: u32, cols: u32) -> Result<()> {
        let matrices_raw: Vec<*const ffi::lh_buffer> = matrices.iter().map(|b| b.as_ptr() as *const ffi::lh_buffer).collect();
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_quant_fused_into(batch.as_ptr(), fmt, count, matrices_raw.as_ptr(), vector.as_ptr(), prologue, aux.as_ptr(), eps, outputs_raw.as_ptr(), rows, cols) })
    }

    /// `lh_matmul_nt_q4_0_into` (include/local_hip.h).
    pub fn matmul_nt_q4_0_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, output: &Buffer, m: u32, k: u32, n: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_q4_0_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), output.as_ptr(), m, k, n) })
    }

    /// `lh_matmul_nt_tq2_0_into` (include/local_hip.h).
    pub fn matmul_nt_tq2_0_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, output: &Buffer, m: u32, k: u32, n: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_tq2_0_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), output.as_ptr(), m, k, n) })
    }

    /// `lh_multivec_nt_q4_0_into` (include/local_hip.h).
    pub fn multivec_nt_q4_0_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, output: &Buffer, m: u32, k: u32, n: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_multivec_nt_q4_0_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), output.as_ptr(), m, k, n) })
    }

    /// `lh_multivec_nt_tq2_0_into` (include/local_hip.h).
    pub fn multivec_nt_tq2_0_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, output: &Buffer, m: u32, k: u32, n: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_multivec_nt_tq2_0_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), output.as_ptr(), m, k, n) })
    }

    /// `lh_matmul_nt_quant_typed_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_quant_typed_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, input: &Buffer, input_dtype: ffi::lh_dtype, weight: &Buffer, output: &Buffer, output_dtype: ffi::lh_dtype, m: u32, k: u32, n: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_quant_typed_into(batch.as_ptr(), fmt, input.as_ptr(), input_dtype, weight.as_ptr(), output.as_ptr(), output_dtype, m, k, n) })
    }

    /// `lh_matmul_nt_quant_gelu_mul_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_quant_gelu_mul_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, input: &Buffer, w_gate: &Buffer, w_up: &Buffer, output: &Buffer, m: u32, k: u32, n: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_quant_gelu_mul_into(batch.as_ptr(), fmt, input.as_ptr(), w_gate.as_ptr(), w_up.as_ptr(), output.as_ptr(), m, k, n) })
    }

    /// `lh_matmul_nt_quant_gelu_mul_strided_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_quant_gelu_mul_strided_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, input: &Buffer, weight: &Buffer, m: u32, k: u32, n: u32, gate_rows: &Buffer, row_stride: u32, row_offset: u32, output: &Buffer) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_quant_gelu_mul_strided_into(batch.as_ptr(), fmt, input.as_ptr(), weight.as_ptr(), m, k, n, gate_rows.as_ptr(), row_stride, row_offset, output.as_ptr()) })
    }

    /// `lh_matmul_nt_quant_capped_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_quant_capped_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, input: &Buffer, input_dtype: ffi::lh_dtype, weight: &Buffer, output: &Buffer, m: u32, k: u32, n: u32, cap: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_quant_capped_into(batch.as_ptr(), fmt, input.as_ptr(), input_dtype, weight.as_ptr(), output.as_ptr(), m, k, n, cap) })
    }

    /// `lh_matmul_nt_quant_norm_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_quant_norm_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, input: &Buffer, weight: &Buffer, m: u32, k: u32, n: u32, norm_weight: &Buffer, residual: &Buffer, output: &Buffer, eps: f32, apply_scale: c_int, scale: f32, norm2_weight: &Buffer, output2: &Buffer) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_quant_norm_into(batch.as_ptr(), fmt, input.as_ptr(), weight.as_ptr(), m, k, n, norm_weight.as_ptr(), residual.as_ptr(), output.as_ptr(), eps, apply_scale, scale, norm2_weight.as_ptr(), output2.as_ptr()) })
    }

    /// `lh_matmul_nt_quant_grouped_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_quant_grouped_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, count: u32, input: &Buffer, weights: &[&Buffer], outputs: &[&Buffer], ns: &[u32], m: u32, k: u32) -> Result<()> {
        let weights_raw: Vec<*const ffi::lh_buffer> = weights.iter().map(|b| b.as_ptr() as *const ffi::lh_buffer).collect();
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_quant_grouped_into(batch.as_ptr(), fmt, count, input.as_ptr(), weights_raw.as_ptr(), outputs_raw.as_ptr(), ns.as_ptr(), m, k) })
    }

    /// `lh_matmul_nt_into` (include/local_hip.h).
    pub fn matmul_nt_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, output: &Buffer, m: u32, k: u32, n: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), output.as_ptr(), m, k, n) })
    }

    /// `lh_clipped_linear_tiled_nt_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn clipped_linear_tiled_nt_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, bias: &Buffer, output: &Buffer, m: u32, k: u32, n: u32, input_min: f32, input_max: f32, output_min: f32, output_max: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_clipped_linear_tiled_nt_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), bias.as_ptr(), output.as_ptr(), m, k, n, input_min, input_max, output_min, output_max) })
    }

    /// `lh_matvec` (include/local_hip.h).
    pub fn matvec(&self, ctx: &Context, matrix: &Buffer, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec(ctx.as_ptr(), matrix.as_ptr(), vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_offset_into` (include/local_hip.h).
    pub fn matvec_offset_into(&self, batch: &mut CommandBatch, matrix: &Buffer, matrix_offset: usize, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_offset_into(batch.as_ptr(), matrix.as_ptr(), matrix_offset, vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_f32out_offset` (include/local_hip.h).
    pub fn matvec_f32out_offset(&self, ctx: &Context, matrix: &Buffer, matrix_offset: usize, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_f32out_offset(ctx.as_ptr(), matrix.as_ptr(), matrix_offset, vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_f32out_offset_into` (include/local_hip.h).
    pub fn matvec_f32out_offset_into(&self, batch: &mut CommandBatch, matrix: &Buffer, matrix_offset: usize, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_f32out_offset_into(batch.as_ptr(), matrix.as_ptr(), matrix_offset, vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_f32in_offset` (include/local_hip.h).
    pub fn matvec_f32in_offset(&self, ctx: &Context, matrix: &Buffer, matrix_offset: usize, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_f32in_offset(ctx.as_ptr(), matrix.as_ptr(), matrix_offset, vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_matvec_f32in_offset_into` (include/local_hip.h).
    pub fn matvec_f32in_offset_into(&self, batch: &mut CommandBatch, matrix: &Buffer, matrix_offset: usize, vector: &Buffer, output: &Buffer, rows: u32, cols: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matvec_f32in_offset_into(batch.as_ptr(), matrix.as_ptr(), matrix_offset, vector.as_ptr(), output.as_ptr(), rows, cols) })
    }

    /// `lh_rms_norm_into` (include/local_hip.h).
    pub fn rms_norm_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, output: &Buffer, dim: u32, rows: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_rms_norm_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), output.as_ptr(), dim, rows, eps) })
    }

    /// `lh_rms_norm_add_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn rms_norm_add_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, residual: &Buffer, output: &Buffer, dim: u32, rows: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_rms_norm_add_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), residual.as_ptr(), output.as_ptr(), dim, rows, eps) })
    }

    /// `lh_rms_norm_residual_scale_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn rms_norm_residual_scale_into(&self, batch: &mut CommandBatch, input: &Buffer, weight: &Buffer, residual: &Buffer, output: &Buffer, dim: u32, rows: u32, eps: f32, apply_scale: c_int, scale: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_rms_norm_residual_scale_into(batch.as_ptr(), input.as_ptr(), weight.as_ptr(), residual.as_ptr(), output.as_ptr(), dim, rows, eps, apply_scale, scale) })
    }

    /// `lh_scale_rms_norm_residual_scale_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn scale_rms_norm_residual_scale_into(&self, batch: &mut CommandBatch, before: f32, input: &Buffer, weight: &Buffer, residual: &Buffer, output: &Buffer, dim: u32, rows: u32, eps: f32, scale: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_scale_rms_norm_residual_scale_into(batch.as_ptr(), before, input.as_ptr(), weight.as_ptr(), residual.as_ptr(), output.as_ptr(), dim, rows, eps, scale) })
    }

    /// `lh_qk_norm_gpu_into` (include/local_hip.h).
    pub fn qk_norm_gpu_into(&self, batch: &mut CommandBatch, qk_data: &Buffer, weight: &Buffer, head_dim: u32, num_heads: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_qk_norm_gpu_into(batch.as_ptr(), qk_data.as_ptr(), weight.as_ptr(), head_dim, num_heads, eps) })
    }

    /// `lh_qk_norm_offset_into` (include/local_hip.h).
    pub fn qk_norm_offset_into(&self, batch: &mut CommandBatch, qk_data: &Buffer, weight: &Buffer, weight_offset: usize, head_dim: u32, num_heads: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_qk_norm_offset_into(batch.as_ptr(), qk_data.as_ptr(), weight.as_ptr(), weight_offset, head_dim, num_heads, eps) })
    }

    /// `lh_qk_norm_rope_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn qk_norm_rope_into(&self, batch: &mut CommandBatch, input: &Buffer, output: &Buffer, weight: &Buffer, head_dim: u32, num_heads: u32, eps: f32, position: u32, theta: f32, partial_rotary_factor: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_qk_norm_rope_into(batch.as_ptr(), input.as_ptr(), output.as_ptr(), weight.as_ptr(), head_dim, num_heads, eps, position, theta, partial_rotary_factor) })
    }

    /// `lh_rope_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn rope_into(&self, batch: &mut CommandBatch, input: &Buffer, output: &Buffer, head_dim: u32, position: u32, theta: f32, partial_rotary_factor: f32, num_heads: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_rope_into(batch.as_ptr(), input.as_ptr(), output.as_ptr(), head_dim, position, theta, partial_rotary_factor, num_heads) })
    }

    /// `lh_rope_batch_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn rope_batch_into(&self, batch: &mut CommandBatch, qk: &Buffer, start_pos: u32, theta: f32, head_dim: u32, num_heads: u32, seq_len: u32, partial_rotary_factor: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_rope_batch_into(batch.as_ptr(), qk.as_ptr(), start_pos, theta, head_dim, num_heads, seq_len, partial_rotary_factor) })
    }

    /// `lh_rope_batch_decode_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn rope_batch_decode_into(&self, batch: &mut CommandBatch, qk: &Buffer, positions: &Buffer, theta: f32, head_dim: u32, num_heads: u32, seq_len: u32, partial_rotary_factor: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_rope_batch_decode_into(batch.as_ptr(), qk.as_ptr(), positions.as_ptr(), theta, head_dim, num_heads, seq_len, partial_rotary_factor) })
    }

    /// `lh_gelu_mul_into` (include/local_hip.h).
    pub fn gelu_mul_into(&self, batch: &mut CommandBatch, a: &Buffer, b: &Buffer, out: &Buffer, count: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_gelu_mul_into(batch.as_ptr(), a.as_ptr(), b.as_ptr(), out.as_ptr(), count) })
    }

    /// `lh_residual_add_into` (include/local_hip.h).
    pub fn residual_add_into(&self, batch: &mut CommandBatch, a: &Buffer, b: &Buffer, output: &Buffer, count: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_residual_add_into(batch.as_ptr(), a.as_ptr(), b.as_ptr(), output.as_ptr(), count) })
    }

    /// `lh_scale_in_place_gpu_into` (include/local_hip.h).
    pub fn scale_in_place_gpu_into(&self, batch: &mut CommandBatch, data: &Buffer, scalar: f32, count: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_scale_in_place_gpu_into(batch.as_ptr(), data.as_ptr(), scalar, count) })
    }

    /// `lh_gather_strided_f16_into` (include/local_hip.h).
    pub fn gather_strided_f16_into(&self, batch: &mut CommandBatch, src: &Buffer, dst: &Buffer, row_stride: u32, base_off: u32, pld: u32, n_rows: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_gather_strided_f16_into(batch.as_ptr(), src.as_ptr(), dst.as_ptr(), row_stride, base_off, pld, n_rows) })
    }

    /// `lh_gelu_mul_strided_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn gelu_mul_strided_into(&self, batch: &mut CommandBatch, a: &Buffer, b: &Buffer, b_row_stride: u32, b_offset: u32, out: &Buffer, dim: u32, rows: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_gelu_mul_strided_into(batch.as_ptr(), a.as_ptr(), b.as_ptr(), b_row_stride, b_offset, out.as_ptr(), dim, rows) })
    }

    /// `lh_logit_softcap_gpu_into` (include/local_hip.h).
    pub fn logit_softcap_gpu_into(&self, batch: &mut CommandBatch, data: &Buffer, cap: f32, count: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_logit_softcap_gpu_into(batch.as_ptr(), data.as_ptr(), cap, count) })
    }

    /// `lh_dequant_q4_0_into` (include/local_hip.h).
    pub fn dequant_q4_0_into(&self, batch: &mut CommandBatch, data: &Buffer, byte_offset: usize, output: &Buffer, num_elements: usize) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_dequant_q4_0_into(batch.as_ptr(), data.as_ptr(), byte_offset, output.as_ptr(), num_elements) })
    }

    /// `lh_dequant_tq2_0_into` (include/local_hip.h).
    pub fn dequant_tq2_0_into(&self, batch: &mut CommandBatch, data: &Buffer, byte_offset: usize, output: &Buffer, num_elements: usize) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_dequant_tq2_0_into(batch.as_ptr(), data.as_ptr(), byte_offset, output.as_ptr(), num_elements) })
    }

    /// `lh_dequant_scaled_into` (include/local_hip.h).
    pub fn dequant_scaled_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, data: &Buffer, byte_offset: usize, output: &Buffer, num_elements: usize, scale: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_dequant_scaled_into(batch.as_ptr(), fmt, data.as_ptr(), byte_offset, output.as_ptr(), num_elements, scale) })
    }

    /// `lh_dequant_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn dequant_rows_into(&self, batch: &mut CommandBatch, fmt: c_int, table: &Buffer, table_rows: u32, cols: u32, rows: &Buffer, n_rows: u32, scale: f32, output: &Buffer) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_dequant_rows_into(batch.as_ptr(), fmt, table.as_ptr(), table_rows, cols, rows.as_ptr(), n_rows, scale, output.as_ptr()) })
    }

    /// `lh_tq2_dequant` (include/local_hip.h).
    pub fn tq2_dequant(&self, ctx: &Context, packed: &Buffer, scales: &Buffer, output: &Buffer, num_elements: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_tq2_dequant(ctx.as_ptr(), packed.as_ptr(), scales.as_ptr(), output.as_ptr(), num_elements) })
    }

    /// `lh_encode_kv_turboquant` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn encode_kv_turboquant(&self, ctx: &Context, input: &Buffer, levels: &Buffer, signs: &Buffer, packed: &Buffer, norms: &Buffer, head_dim: u32, n_kv_heads: u32, num_tokens: u32, bits: u32, position: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_encode_kv_turboquant(ctx.as_ptr(), input.as_ptr(), levels.as_ptr(), signs.as_ptr(), packed.as_ptr(), norms.as_ptr(), head_dim, n_kv_heads, num_tokens, bits, position, ring_capacity) })
    }

    /// `lh_encode_kv_turboquant_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn encode_kv_turboquant_into(&self, batch: &mut CommandBatch, input: &Buffer, levels: &Buffer, signs: &Buffer, packed: &Buffer, norms: &Buffer, head_dim: u32, n_kv_heads: u32, num_tokens: u32, bits: u32, position: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_encode_kv_turboquant_into(batch.as_ptr(), input.as_ptr(), levels.as_ptr(), signs.as_ptr(), packed.as_ptr(), norms.as_ptr(), head_dim, n_kv_heads, num_tokens, bits, position, ring_capacity) })
    }

    /// `lh_encode_kv_turboquant_batched_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn encode_kv_turboquant_batched_into(&self, batch: &mut CommandBatch, input: &Buffer, levels: &Buffer, signs: &Buffer, packed: &Buffer, norms: &Buffer, positions: &Buffer, head_dim: u32, n_kv_heads: u32, lane_capacity: u32, bits: u32, n_lanes: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_encode_kv_turboquant_batched_into(batch.as_ptr(), input.as_ptr(), levels.as_ptr(), signs.as_ptr(), packed.as_ptr(), norms.as_ptr(), positions.as_ptr(), head_dim, n_kv_heads, lane_capacity, bits, n_lanes, ring_capacity) })
    }

    /// `lh_dequantize_kv_turboquant` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn dequantize_kv_turboquant(&self, ctx: &Context, packed: &Buffer, norms: &Buffer, levels: &Buffer, signs: &Buffer, output: &Buffer, head_dim: u32, n_kv_heads: u32, num_tokens: u32, bits: u32, token_start: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_dequantize_kv_turboquant(ctx.as_ptr(), packed.as_ptr(), norms.as_ptr(), levels.as_ptr(), signs.as_ptr(), output.as_ptr(), head_dim, n_kv_heads, num_tokens, bits, token_start, ring_capacity) })
    }

    /// `lh_dequantize_kv_turboquant_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn dequantize_kv_turboquant_into(&self, batch: &mut CommandBatch, packed: &Buffer, norms: &Buffer, levels: &Buffer, signs: &Buffer, output: &Buffer, head_dim: u32, n_kv_heads: u32, num_tokens: u32, bits: u32, token_start: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_dequantize_kv_turboquant_into(batch.as_ptr(), packed.as_ptr(), norms.as_ptr(), levels.as_ptr(), signs.as_ptr(), output.as_ptr(), head_dim, n_kv_heads, num_tokens, bits, token_start, ring_capacity) })
    }

    /// `lh_decode_qkv_prepare_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn decode_qkv_prepare_into(&self, batch: &mut CommandBatch, q: &Buffer, k: &Buffer, v: &Buffer, q_norm: &Buffer, k_norm: &Buffer, levels: &Buffer, signs: &Buffer, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, head_dim: u32, n_q_heads: u32, n_kv_heads: u32, eps: f32, position: u32, theta: f32, partial_rotary_factor: f32, bits: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_decode_qkv_prepare_into(batch.as_ptr(), q.as_ptr(), k.as_ptr(), v.as_ptr(), q_norm.as_ptr(), k_norm.as_ptr(), levels.as_ptr(), signs.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), head_dim, n_q_heads, n_kv_heads, eps, position, theta, partial_rotary_factor, bits, ring_capacity) })
    }

    /// `lh_decode_qkv_prepare_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn decode_qkv_prepare_rows_into(&self, batch: &mut CommandBatch, q: &Buffer, k: &Buffer, v: &Buffer, q_norm: &Buffer, k_norm: &Buffer, levels: &Buffer, signs: &Buffer, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, positions: &Buffer, head_dim: u32, n_q_heads: u32, n_kv_heads: u32, rows: u32, eps: f32, start_position: u32, theta: f32, partial_rotary_factor: f32, bits: u32, ring_capacity: u32, lane_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_decode_qkv_prepare_rows_into(batch.as_ptr(), q.as_ptr(), k.as_ptr(), v.as_ptr(), q_norm.as_ptr(), k_norm.as_ptr(), levels.as_ptr(), signs.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), positions.as_ptr(), head_dim, n_q_heads, n_kv_heads, rows, eps, start_position, theta, partial_rotary_factor, bits, ring_capacity, lane_capacity) })
    }

    /// `lh_matmul_nt_qkv_prepare_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_qkv_prepare_rows_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, input: &Buffer, w_q: &Buffer, w_k: &Buffer, w_v: &Buffer, k_dim: u32, q: &Buffer, k: &Buffer, v: &Buffer, q_norm: &Buffer, k_norm: &Buffer, levels: &Buffer, signs: &Buffer, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, positions: &Buffer, head_dim: u32, n_q_heads: u32, n_kv_heads: u32, rows: u32, eps: f32, start_position: u32, theta: f32, partial_rotary_factor: f32, bits: u32, ring_capacity: u32, lane_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_qkv_prepare_rows_into(batch.as_ptr(), fmt, input.as_ptr(), w_q.as_ptr(), w_k.as_ptr(), w_v.as_ptr(), k_dim, q.as_ptr(), k.as_ptr(), v.as_ptr(), q_norm.as_ptr(), k_norm.as_ptr(), levels.as_ptr(), signs.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), positions.as_ptr(), head_dim, n_q_heads, n_kv_heads, rows, eps, start_position, theta, partial_rotary_factor, bits, ring_capacity, lane_capacity) })
    }

    /// `lh_matmul_nt_q_prepare_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_q_prepare_rows_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, input: &Buffer, w_q: &Buffer, k_dim: u32, q: &Buffer, q_norm: &Buffer, signs: &Buffer, rq: &Buffer, positions: &Buffer, head_dim: u32, n_q_heads: u32, rows: u32, eps: f32, start_position: u32, theta: f32, partial_rotary_factor: f32, lane_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_q_prepare_rows_into(batch.as_ptr(), fmt, input.as_ptr(), w_q.as_ptr(), k_dim, q.as_ptr(), q_norm.as_ptr(), signs.as_ptr(), rq.as_ptr(), positions.as_ptr(), head_dim, n_q_heads, rows, eps, start_position, theta, partial_rotary_factor, lane_capacity) })
    }

    /// `lh_hadamard_rotate_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn hadamard_rotate_into(&self, batch: &mut CommandBatch, input: &Buffer, signs: &Buffer, output: &Buffer, head_dim: u32, num_heads: u32, pre_sign: c_int, post_sign: c_int) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_hadamard_rotate_into(batch.as_ptr(), input.as_ptr(), signs.as_ptr(), output.as_ptr(), head_dim, num_heads, pre_sign, post_sign) })
    }

    /// `lh_hadamard_rotate_hf_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn hadamard_rotate_hf_into(&self, batch: &mut CommandBatch, input: &Buffer, signs: &Buffer, output: &Buffer, head_dim: u32, num_heads: u32, pre_sign: c_int, post_sign: c_int) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_hadamard_rotate_hf_into(batch.as_ptr(), input.as_ptr(), signs.as_ptr(), output.as_ptr(), head_dim, num_heads, pre_sign, post_sign) })
    }

    /// `lh_hadamard_rotate_fh_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn hadamard_rotate_fh_into(&self, batch: &mut CommandBatch, input: &Buffer, signs: &Buffer, output: &Buffer, head_dim: u32, num_heads: u32, pre_sign: c_int, post_sign: c_int) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_hadamard_rotate_fh_into(batch.as_ptr(), input.as_ptr(), signs.as_ptr(), output.as_ptr(), head_dim, num_heads, pre_sign, post_sign) })
    }

    /// `lh_flash_attention_tq_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_attention_tq_into(&self, batch: &mut CommandBatch, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, levels: &Buffer, out: &Buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_attention_tq_into(batch.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), levels.as_ptr(), out.as_ptr(), head_dim, kv_len, current_pos, num_q_heads, num_kv_heads, window, bits, ring_capacity) })
    }

    /// `lh_flash_attention_tq_static_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_attention_tq_static_into(&self, batch: &mut CommandBatch, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, levels: &Buffer, out: &Buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_attention_tq_static_into(batch.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), levels.as_ptr(), out.as_ptr(), head_dim, kv_len, current_pos, num_q_heads, num_kv_heads, window, bits, ring_capacity) })
    }

    /// `lh_flash_attention_tq_prefill_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_attention_tq_prefill_into(&self, batch: &mut CommandBatch, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, levels: &Buffer, out: &Buffer, head_dim: u32, kv_len: u32, start_pos: u32, n_rows: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_attention_tq_prefill_into(batch.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), levels.as_ptr(), out.as_ptr(), head_dim, kv_len, start_pos, n_rows, num_q_heads, num_kv_heads, window, bits, ring_capacity) })
    }

    /// `lh_flash_attention_tq_prefill_tiled_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_attention_tq_prefill_tiled_into(&self, batch: &mut CommandBatch, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, levels: &Buffer, out: &Buffer, head_dim: u32, kv_len: u32, start_pos: u32, n_rows: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_attention_tq_prefill_tiled_into(batch.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), levels.as_ptr(), out.as_ptr(), head_dim, kv_len, start_pos, n_rows, num_q_heads, num_kv_heads, window, bits, ring_capacity) })
    }

    /// `lh_flash_attention_tq_batched_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_attention_tq_batched_into(&self, batch: &mut CommandBatch, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, levels: &Buffer, out: &Buffer, positions: &Buffer, head_dim: u32, lane_capacity: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, n_lanes: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_attention_tq_batched_into(batch.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), levels.as_ptr(), out.as_ptr(), positions.as_ptr(), head_dim, lane_capacity, num_q_heads, num_kv_heads, window, bits, n_lanes, ring_capacity) })
    }

    /// `lh_flash_attention_tq_rotated_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_attention_tq_rotated_into(&self, batch: &mut CommandBatch, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, levels: &Buffer, signs: &Buffer, out: &Buffer, out_f16: &Buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_attention_tq_rotated_into(batch.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), levels.as_ptr(), signs.as_ptr(), out.as_ptr(), out_f16.as_ptr(), head_dim, kv_len, current_pos, num_q_heads, num_kv_heads, window, bits, ring_capacity) })
    }

    /// `lh_matmul_nt_qkv_attention_lanes_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn matmul_nt_qkv_attention_lanes_into(&self, batch: &mut CommandBatch, fmt: ffi::lh_quant, input: &Buffer, w_q: &Buffer, w_k: &Buffer, w_v: &Buffer, k_dim: u32, q: &Buffer, k: &Buffer, v: &Buffer, q_norm: &Buffer, k_norm: &Buffer, levels: &Buffer, signs: &Buffer, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, positions: &Buffer, out: &Buffer, out_f16: &Buffer, head_dim: u32, n_q_heads: u32, n_kv_heads: u32, lanes: u32, eps: f32, theta: f32, partial_rotary_factor: f32, window: u32, bits: u32, ring_capacity: u32, lane_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_matmul_nt_qkv_attention_lanes_into(batch.as_ptr(), fmt, input.as_ptr(), w_q.as_ptr(), w_k.as_ptr(), w_v.as_ptr(), k_dim, q.as_ptr(), k.as_ptr(), v.as_ptr(), q_norm.as_ptr(), k_norm.as_ptr(), levels.as_ptr(), signs.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), positions.as_ptr(), out.as_ptr(), out_f16.as_ptr(), head_dim, n_q_heads, n_kv_heads, lanes, eps, theta, partial_rotary_factor, window, bits, ring_capacity, lane_capacity) })
    }

    /// `lh_flash_attention_tq_batched_rotated_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_attention_tq_batched_rotated_into(&self, batch: &mut CommandBatch, rq: &Buffer, k_codes: &Buffer, k_norms: &Buffer, v_codes: &Buffer, v_norms: &Buffer, levels: &Buffer, signs: &Buffer, out: &Buffer, out_f16: &Buffer, positions: &Buffer, head_dim: u32, lane_capacity: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, bits: u32, n_lanes: u32, ring_capacity: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_attention_tq_batched_rotated_into(batch.as_ptr(), rq.as_ptr(), k_codes.as_ptr(), k_norms.as_ptr(), v_codes.as_ptr(), v_norms.as_ptr(), levels.as_ptr(), signs.as_ptr(), out.as_ptr(), out_f16.as_ptr(), positions.as_ptr(), head_dim, lane_capacity, num_q_heads, num_kv_heads, window, bits, n_lanes, ring_capacity) })
    }

    /// `lh_flash_decoding_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_decoding_into(&self, batch: &mut CommandBatch, q: &Buffer, k: &Buffer, v: &Buffer, output: &Buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_decoding_into(batch.as_ptr(), q.as_ptr(), k.as_ptr(), v.as_ptr(), output.as_ptr(), head_dim, kv_len, current_pos, num_q_heads, num_kv_heads) })
    }

    /// `lh_flash_attention_windowed_split_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn flash_attention_windowed_split_into(&self, batch: &mut CommandBatch, q: &Buffer, k: &Buffer, v: &Buffer, output: &Buffer, partial_max: &Buffer, partial_sum: &Buffer, partial_acc: &Buffer, head_dim: u32, kv_len: u32, current_pos: u32, num_q_heads: u32, num_kv_heads: u32, window: u32, num_splits: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_flash_attention_windowed_split_into(batch.as_ptr(), q.as_ptr(), k.as_ptr(), v.as_ptr(), output.as_ptr(), partial_max.as_ptr(), partial_sum.as_ptr(), partial_acc.as_ptr(), head_dim, kv_len, current_pos, num_q_heads, num_kv_heads, window, num_splits) })
    }

    /// `lh_embed_rows_bf16_into` (include/local_hip.h).
    pub fn embed_rows_bf16_into(&self, batch: &mut CommandBatch, table: &Buffer, table_rows: u32, cols: u32, rows: &Buffer, n_rows: u32, output: &Buffer) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_embed_rows_bf16_into(batch.as_ptr(), table.as_ptr(), table_rows, cols, rows.as_ptr(), n_rows, output.as_ptr()) })
    }

    /// `lh_embed_token_bf16_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn embed_token_bf16_into(&self, batch: &mut CommandBatch, table: &Buffer, table_rows: u32, cols: u32, token: u32, position: u32, output: &Buffer, at: &Buffer, next: &Buffer) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_embed_token_bf16_into(batch.as_ptr(), table.as_ptr(), table_rows, cols, token, position, output.as_ptr(), at.as_ptr(), next.as_ptr()) })
    }

    /// `lh_norm_rows_f32_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn norm_rows_f32_into(&self, batch: &mut CommandBatch, input: &Buffer, add: &Buffer, weight: &Buffer, store: &Buffer, row_index: &Buffer, output: &Buffer, output_dtype: c_int, dim: u32, rows: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_norm_rows_f32_into(batch.as_ptr(), input.as_ptr(), add.as_ptr(), weight.as_ptr(), store.as_ptr(), row_index.as_ptr(), output.as_ptr(), output_dtype, dim, rows, eps) })
    }

    /// `lh_residual_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn residual_rows_into(&self, batch: &mut CommandBatch, input: &Buffer, branch: &Buffer, weight: &Buffer, store: &Buffer, output: &Buffer, output_dtype: c_int, dim: u32, rows: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_residual_rows_into(batch.as_ptr(), input.as_ptr(), branch.as_ptr(), weight.as_ptr(), store.as_ptr(), output.as_ptr(), output_dtype, dim, rows, eps) })
    }

    /// `lh_gated_norm_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn gated_norm_rows_into(&self, batch: &mut CommandBatch, input: &Buffer, gate: &Buffer, gate_act: u32, gate_first: c_int, weight: &Buffer, output: &Buffer, dtype: c_int, dim: u32, group: u32, rows: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_gated_norm_rows_into(batch.as_ptr(), input.as_ptr(), gate.as_ptr(), gate_act, gate_first, weight.as_ptr(), output.as_ptr(), dtype, dim, group, rows, eps) })
    }

    /// `lh_softcap_f32_into` (include/local_hip.h).
    pub fn softcap_f32_into(&self, batch: &mut CommandBatch, logits: &Buffer, n: usize, cap: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_softcap_f32_into(batch.as_ptr(), logits.as_ptr(), n, cap) })
    }

    /// `lh_linear_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_rows_into(&self, batch: &mut CommandBatch, input: &Buffer, input_dtype: c_int, weight: &Buffer, bias: &Buffer, m: u32, k: u32, count: u32, ns: &[u32], acts: &[u32], heads: &[u32], padded: &[u32], layouts: &[u32], outputs: &[&Buffer], output_dtype: c_int, accumulate: c_int, position: &Buffer) -> Result<()> {
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_rows_into(batch.as_ptr(), input.as_ptr(), input_dtype, weight.as_ptr(), bias.as_ptr(), m, k, count, ns.as_ptr(), acts.as_ptr(), heads.as_ptr(), padded.as_ptr(), layouts.as_ptr(), outputs_raw.as_ptr(), output_dtype, accumulate, position.as_ptr()) })
    }

    /// `lh_linear_vector_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_vector_into(&self, batch: &mut CommandBatch, input: &Buffer, input_dtype: c_int, weight: &Buffer, bias: &Buffer, k: u32, count: u32, ns: &[u32], acts: &[u32], heads: &[u32], padded: &[u32], layouts: &[u32], outputs: &[&Buffer], output_dtype: c_int, accumulate: c_int, position: &Buffer) -> Result<()> {
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_vector_into(batch.as_ptr(), input.as_ptr(), input_dtype, weight.as_ptr(), bias.as_ptr(), k, count, ns.as_ptr(), acts.as_ptr(), heads.as_ptr(), padded.as_ptr(), layouts.as_ptr(), outputs_raw.as_ptr(), output_dtype, accumulate, position.as_ptr()) })
    }

    /// `lh_linear_norm_vector_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_norm_vector_into(&self, batch: &mut CommandBatch, input: &Buffer, add: &Buffer, store: &Buffer, norm_weight: &Buffer, eps: f32, weight: &Buffer, bias: &Buffer, k: u32, count: u32, ns: &[u32], acts: &[u32], heads: &[u32], padded: &[u32], layouts: &[u32], outputs: &[&Buffer], output_dtype: c_int, accumulate: c_int, position: &Buffer) -> Result<()> {
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_norm_vector_into(batch.as_ptr(), input.as_ptr(), add.as_ptr(), store.as_ptr(), norm_weight.as_ptr(), eps, weight.as_ptr(), bias.as_ptr(), k, count, ns.as_ptr(), acts.as_ptr(), heads.as_ptr(), padded.as_ptr(), layouts.as_ptr(), outputs_raw.as_ptr(), output_dtype, accumulate, position.as_ptr()) })
    }

    /// `lh_linear_norm_vector_capped_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_norm_vector_capped_into(&self, batch: &mut CommandBatch, input: &Buffer, norm_weight: &Buffer, eps: f32, weight: &Buffer, bias: &Buffer, k: u32, n: u32, output: &Buffer, cap: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_norm_vector_capped_into(batch.as_ptr(), input.as_ptr(), norm_weight.as_ptr(), eps, weight.as_ptr(), bias.as_ptr(), k, n, output.as_ptr(), cap) })
    }

    /// `lh_linear_norm_vector_copied_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_norm_vector_copied_into(&self, batch: &mut CommandBatch, input: &Buffer, norm_weight: &Buffer, eps: f32, weight: &Buffer, bias: &Buffer, k: u32, n: u32, output: &Buffer, copy: &Buffer, cap: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_norm_vector_copied_into(batch.as_ptr(), input.as_ptr(), norm_weight.as_ptr(), eps, weight.as_ptr(), bias.as_ptr(), k, n, output.as_ptr(), copy.as_ptr(), cap) })
    }

    /// `lh_linear_residual_norm_vector_copied_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_residual_norm_vector_copied_into(&self, batch: &mut CommandBatch, input: &Buffer, branch: &Buffer, branch_weight: &Buffer, branch_eps: f32, norm_weight: &Buffer, eps: f32, weight: &Buffer, bias: &Buffer, k: u32, n: u32, output: &Buffer, copy: &Buffer, cap: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_residual_norm_vector_copied_into(batch.as_ptr(), input.as_ptr(), branch.as_ptr(), branch_weight.as_ptr(), branch_eps, norm_weight.as_ptr(), eps, weight.as_ptr(), bias.as_ptr(), k, n, output.as_ptr(), copy.as_ptr(), cap) })
    }

    /// `lh_linear_residual_vector_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_residual_vector_into(&self, batch: &mut CommandBatch, input: &Buffer, branch: &Buffer, store: &Buffer, norm_weight: &Buffer, eps: f32, weight: &Buffer, bias: &Buffer, k: u32, count: u32, ns: &[u32], acts: &[u32], heads: &[u32], padded: &[u32], layouts: &[u32], outputs: &[&Buffer], output_dtype: c_int, accumulate: c_int, position: &Buffer) -> Result<()> {
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_residual_vector_into(batch.as_ptr(), input.as_ptr(), branch.as_ptr(), store.as_ptr(), norm_weight.as_ptr(), eps, weight.as_ptr(), bias.as_ptr(), k, count, ns.as_ptr(), acts.as_ptr(), heads.as_ptr(), padded.as_ptr(), layouts.as_ptr(), outputs_raw.as_ptr(), output_dtype, accumulate, position.as_ptr()) })
    }

    /// `lh_linear_gated_vector_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_gated_vector_into(&self, batch: &mut CommandBatch, input: &Buffer, gate: &Buffer, gate_dtype: c_int, gate_act: u32, gate_first: c_int, norm_weight: &Buffer, group: u32, eps: f32, weight: &Buffer, bias: &Buffer, k: u32, count: u32, ns: &[u32], acts: &[u32], heads: &[u32], padded: &[u32], layouts: &[u32], outputs: &[&Buffer], output_dtype: c_int, accumulate: c_int, position: &Buffer) -> Result<()> {
        let outputs_raw: Vec<*mut ffi::lh_buffer> = outputs.iter().map(|b| b.as_ptr()).collect();
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_gated_vector_into(batch.as_ptr(), input.as_ptr(), gate.as_ptr(), gate_dtype, gate_act, gate_first, norm_weight.as_ptr(), group, eps, weight.as_ptr(), bias.as_ptr(), k, count, ns.as_ptr(), acts.as_ptr(), heads.as_ptr(), padded.as_ptr(), layouts.as_ptr(), outputs_raw.as_ptr(), output_dtype, accumulate, position.as_ptr()) })
    }

    /// `lh_attention_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn attention_rows_into(&self, batch: &mut CommandBatch, q: &Buffer, keys: &Buffer, values: &Buffer, output: &Buffer, dtype: c_int, position: &Buffer, max_position: u32, rows: u32, heads: u32, kv_heads: u32, maps: u32, dim: u32, vdim: u32, capacity: u32, scale: f32, lambda: f32, out_scale: f32, eps: f32, sink: &Buffer, gate: &Buffer) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_attention_rows_into(batch.as_ptr(), q.as_ptr(), keys.as_ptr(), values.as_ptr(), output.as_ptr(), dtype, position.as_ptr(), max_position, rows, heads, kv_heads, maps, dim, vdim, capacity, scale, lambda, out_scale, eps, sink.as_ptr(), gate.as_ptr()) })
    }

    /// `lh_latent_prepare_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn latent_prepare_into(&self, batch: &mut CommandBatch, q_rot: &Buffer, down: &Buffer, norm_weight: &Buffer, frequencies: &Buffer, position: &Buffer, q: &Buffer, q_dtype: c_int, cache: &Buffer, dtype: c_int, rows: u32, heads: u32, rank: u32, rot: u32, q_ld: u32, rot_column: u32, clear_column: u32, capacity: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_latent_prepare_into(batch.as_ptr(), q_rot.as_ptr(), down.as_ptr(), norm_weight.as_ptr(), frequencies.as_ptr(), position.as_ptr(), q.as_ptr(), q_dtype, cache.as_ptr(), dtype, rows, heads, rank, rot, q_ld, rot_column, clear_column, capacity, eps) })
    }

    /// `lh_head_linear_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn head_linear_into(&self, batch: &mut CommandBatch, input: &Buffer, dtype: c_int, weight: &Buffer, output: &Buffer, output_dtype: c_int, rows: u32, heads: u32, n: u32, k: u32, output_ld: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_head_linear_into(batch.as_ptr(), input.as_ptr(), dtype, weight.as_ptr(), output.as_ptr(), output_dtype, rows, heads, n, k, output_ld) })
    }

    /// `lh_latent_expand_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn latent_expand_into(&self, batch: &mut CommandBatch, cache: &Buffer, dtype: c_int, weight: &Buffer, keys: &Buffer, values: &Buffer, positions: u32, heads: u32, dim: u32, rot: u32, vdim: u32, rank: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_latent_expand_into(batch.as_ptr(), cache.as_ptr(), dtype, weight.as_ptr(), keys.as_ptr(), values.as_ptr(), positions, heads, dim, rot, vdim, rank) })
    }

    /// `lh_latent_attention_rows_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn latent_attention_rows_into(&self, batch: &mut CommandBatch, q: &Buffer, cache: &Buffer, output: &Buffer, dtype: c_int, position: &Buffer, max_position: u32, rows: u32, heads: u32, rank: u32, rot: u32, capacity: u32, scale: f32, sink: &Buffer, gate: &Buffer) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_latent_attention_rows_into(batch.as_ptr(), q.as_ptr(), cache.as_ptr(), output.as_ptr(), dtype, position.as_ptr(), max_position, rows, heads, rank, rot, capacity, scale, sink.as_ptr(), gate.as_ptr()) })
    }

    /// `lh_latent_attention_values_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn latent_attention_values_into(&self, batch: &mut CommandBatch, q: &Buffer, cache: &Buffer, latent: &Buffer, dtype: c_int, position: &Buffer, max_position: u32, rows: u32, heads: u32, rank: u32, rot: u32, capacity: u32, scale: f32, sink: &Buffer, gate: &Buffer, value_weight: &Buffer, vdim: u32, output: &Buffer) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_latent_attention_values_into(batch.as_ptr(), q.as_ptr(), cache.as_ptr(), latent.as_ptr(), dtype, position.as_ptr(), max_position, rows, heads, rank, rot, capacity, scale, sink.as_ptr(), gate.as_ptr(), value_weight.as_ptr(), vdim, output.as_ptr()) })
    }

    /// `lh_latent_queries_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn latent_queries_into(&self, batch: &mut CommandBatch, q: &Buffer, key_weight: &Buffer, q_rot: &Buffer, down: &Buffer, norm_weight: &Buffer, frequencies: &Buffer, position: &Buffer, output: &Buffer, cache: &Buffer, dtype: c_int, rows: u32, heads: u32, dim: u32, rank: u32, rot: u32, capacity: u32, eps: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_latent_queries_into(batch.as_ptr(), q.as_ptr(), key_weight.as_ptr(), q_rot.as_ptr(), down.as_ptr(), norm_weight.as_ptr(), frequencies.as_ptr(), position.as_ptr(), output.as_ptr(), cache.as_ptr(), dtype, rows, heads, dim, rank, rot, capacity, eps) })
    }

    /// `lh_linear_attention_recurrent_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_attention_recurrent_into(&self, batch: &mut CommandBatch, q: &Buffer, k: &Buffer, v: &Buffer, dtype: c_int, state: &Buffer, decay: &Buffer, output: &Buffer, rows: u32, heads: u32, dim: u32, vdim: u32, scale: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_attention_recurrent_into(batch.as_ptr(), q.as_ptr(), k.as_ptr(), v.as_ptr(), dtype, state.as_ptr(), decay.as_ptr(), output.as_ptr(), rows, heads, dim, vdim, scale) })
    }

    /// `lh_linear_attention_chunked_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn linear_attention_chunked_into(&self, batch: &mut CommandBatch, q: &Buffer, k: &Buffer, v: &Buffer, state: &Buffer, decay_powers: &Buffer, workspace: &Buffer, output: &Buffer, rows: u32, heads: u32, dim: u32, vdim: u32, scale: f32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_linear_attention_chunked_into(batch.as_ptr(), q.as_ptr(), k.as_ptr(), v.as_ptr(), state.as_ptr(), decay_powers.as_ptr(), workspace.as_ptr(), output.as_ptr(), rows, heads, dim, vdim, scale) })
    }

    /// `lh_selective_conv_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn selective_conv_into(&self, batch: &mut CommandBatch, input: &Buffer, dtype: c_int, ring: &Buffer, taps_weight: &Buffer, bias: &Buffer, position: &Buffer, x: &Buffer, b: &Buffer, c: &Buffer, rows: u32, heads: u32, vdim: u32, groups: u32, state: u32, taps: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_selective_conv_into(batch.as_ptr(), input.as_ptr(), dtype, ring.as_ptr(), taps_weight.as_ptr(), bias.as_ptr(), position.as_ptr(), x.as_ptr(), b.as_ptr(), c.as_ptr(), rows, heads, vdim, groups, state, taps) })
    }

    /// `lh_selective_recurrent_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn selective_recurrent_into(&self, batch: &mut CommandBatch, x: &Buffer, b: &Buffer, c: &Buffer, dtype: c_int, dt_raw: &Buffer, dt_bias: &Buffer, a_log: &Buffer, skip: &Buffer, memory: &Buffer, output: &Buffer, rows: u32, heads: u32, vdim: u32, groups: u32, state: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_selective_recurrent_into(batch.as_ptr(), x.as_ptr(), b.as_ptr(), c.as_ptr(), dtype, dt_raw.as_ptr(), dt_bias.as_ptr(), a_log.as_ptr(), skip.as_ptr(), memory.as_ptr(), output.as_ptr(), rows, heads, vdim, groups, state) })
    }

    /// `lh_selective_chunked_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn selective_chunked_into(&self, batch: &mut CommandBatch, x: &Buffer, b: &Buffer, c: &Buffer, dt_raw: &Buffer, dt_bias: &Buffer, a_log: &Buffer, skip: &Buffer, memory: &Buffer, steps: &Buffer, workspace: &Buffer, output: &Buffer, rows: u32, heads: u32, vdim: u32, groups: u32, state: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_selective_chunked_into(batch.as_ptr(), x.as_ptr(), b.as_ptr(), c.as_ptr(), dt_raw.as_ptr(), dt_bias.as_ptr(), a_log.as_ptr(), skip.as_ptr(), memory.as_ptr(), steps.as_ptr(), workspace.as_ptr(), output.as_ptr(), rows, heads, vdim, groups, state) })
    }

    /// `lh_selective_step_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn selective_step_into(&self, batch: &mut CommandBatch, input: &Buffer, ring: &Buffer, taps_weight: &Buffer, bias: &Buffer, position: &Buffer, dt_raw: &Buffer, dt_bias: &Buffer, a_log: &Buffer, skip: &Buffer, memory: &Buffer, output: &Buffer, heads: u32, vdim: u32, groups: u32, state: u32, taps: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_selective_step_into(batch.as_ptr(), input.as_ptr(), ring.as_ptr(), taps_weight.as_ptr(), bias.as_ptr(), position.as_ptr(), dt_raw.as_ptr(), dt_bias.as_ptr(), a_log.as_ptr(), skip.as_ptr(), memory.as_ptr(), output.as_ptr(), heads, vdim, groups, state, taps) })
    }

    /// `lh_moe_route_into` (include/local_hip.h).
    pub fn moe_route_into(&self, batch: &mut CommandBatch, logits: &Buffer, plan: &Buffer, rows: u32, experts: u32, top: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_moe_route_into(batch.as_ptr(), logits.as_ptr(), plan.as_ptr(), rows, experts, top) })
    }

    /// `lh_moe_up_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn moe_up_into(&self, batch: &mut CommandBatch, input: &Buffer, dtype: c_int, plan: &Buffer, up: &Buffer, hidden: &Buffer, rows: u32, experts: u32, top: u32, width: u32, ff: u32, act: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_moe_up_into(batch.as_ptr(), input.as_ptr(), dtype, plan.as_ptr(), up.as_ptr(), hidden.as_ptr(), rows, experts, top, width, ff, act) })
    }

    /// `lh_moe_down_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn moe_down_into(&self, batch: &mut CommandBatch, hidden: &Buffer, dtype: c_int, plan: &Buffer, down: &Buffer, slots: &Buffer, residual: &Buffer, rows: u32, experts: u32, top: u32, width: u32, ff: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_moe_down_into(batch.as_ptr(), hidden.as_ptr(), dtype, plan.as_ptr(), down.as_ptr(), slots.as_ptr(), residual.as_ptr(), rows, experts, top, width, ff) })
    }

    /// `lh_moe_vector_up_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn moe_vector_up_into(&self, batch: &mut CommandBatch, input: &Buffer, norm_weight: &Buffer, eps: f32, logits: &Buffer, up: &Buffer, hidden: &Buffer, experts: u32, top: u32, width: u32, ff: u32, act: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_moe_vector_up_into(batch.as_ptr(), input.as_ptr(), norm_weight.as_ptr(), eps, logits.as_ptr(), up.as_ptr(), hidden.as_ptr(), experts, top, width, ff, act) })
    }

    /// `lh_moe_vector_routed_up_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn moe_vector_routed_up_into(&self, batch: &mut CommandBatch, input: &Buffer, norm_weight: &Buffer, eps: f32, router: &Buffer, logits: &Buffer, up: &Buffer, hidden: &Buffer, experts: u32, top: u32, width: u32, ff: u32, act: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_moe_vector_routed_up_into(batch.as_ptr(), input.as_ptr(), norm_weight.as_ptr(), eps, router.as_ptr(), logits.as_ptr(), up.as_ptr(), hidden.as_ptr(), experts, top, width, ff, act) })
    }

    /// `lh_moe_vector_down_into` (include/local_hip.h).
    #[allow(clippy::too_many_arguments)]
    pub fn moe_vector_down_into(&self, batch: &mut CommandBatch, hidden: &Buffer, logits: &Buffer, down: &Buffer, residual: &Buffer, experts: u32, top: u32, width: u32, ff: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_moe_vector_down_into(batch.as_ptr(), hidden.as_ptr(), logits.as_ptr(), down.as_ptr(), residual.as_ptr(), experts, top, width, ff) })
    }

    /// `lh_advance_position_into` (include/local_hip.h).
    pub fn advance_position_into(&self, batch: &mut CommandBatch, position: &Buffer, by: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_advance_position_into(batch.as_ptr(), position.as_ptr(), by) })
    }

    /// `lh_argmax_rows_f32_into` (include/local_hip.h).
    pub fn argmax_rows_f32_into(&self, batch: &mut CommandBatch, logits: &Buffer, index: &Buffer, rows: u32, n: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_argmax_rows_f32_into(batch.as_ptr(), logits.as_ptr(), index.as_ptr(), rows, n) })
    }

    /// `lh_argmax_advance_f32_into` (include/local_hip.h).
    pub fn argmax_advance_f32_into(&self, batch: &mut CommandBatch, logits: &Buffer, index: &Buffer, n: u32, position: &Buffer, by: u32) -> Result<()> {
        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.
        check(unsafe { ffi::lh_argmax_advance_f32_into(batch.as_ptr(), logits.as_ptr(), index.as_ptr(), n, position.as_ptr(), by) })
    }
}

/* Prototypes of the prebuilt launchers (libtf_<entry>.so, one object per entry).
 * Each replaces one generated `launcher_kernel_<md5>` of the reference
 * (tensorforge/generators/generator.py:426-436) with the same name and parameters.
 * The name hashes the description, which does not hold the floating type or the
 * sparsity pattern: chains differing only there share a name with different
 * parameter types. Such prototypes are guarded: define TF_CATALOG_<ENTRY> (the
 * object's entry name in capitals) for the object you link.
 * Generated by tensorforge_amd/catalog_header.py; do not edit. */
#ifndef TENSORFORGE_CATALOG_H
#define TENSORFORGE_CATALOG_H
#include <stddef.h>
#ifdef __cplusplus
extern "C" {
#endif
/* ader7_f64_mfma_bf16x3, ader7_f64_mfma_fp32, ader7_f64_plain, ader7_f64_tuned */
void launcher_kernel_76924ee264(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, size_t numElements, unsigned* flags, void* streamPtr);
#if defined(TF_CATALOG_ADER_DENSE_F32_PLAIN) || defined(TF_CATALOG_ADER_DENSE_F32_TUNED) || defined(TF_CATALOG_ADER_F32_PLAIN) || defined(TF_CATALOG_ADER_F32_TUNED)
void launcher_kernel_b053681baa(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, float* m2, unsigned m2_extraOffset, const float* m3, const float* m4, unsigned m4_extraOffset, const float* m5, const float* m6, unsigned m6_extraOffset, const float* m7, size_t numElements, unsigned* flags, void* streamPtr);
#elif defined(TF_CATALOG_ADER_DENSE_F64_MFMA_FP64) || defined(TF_CATALOG_ADER_DENSE_F64_PLAIN) || defined(TF_CATALOG_ADER_DENSE_F64_TUNED) || defined(TF_CATALOG_ADER_F64_PLAIN) || defined(TF_CATALOG_ADER_F64_TUNED) || defined(TF_CATALOG_OPT_ADER_DENSE_F64_UNROLLED) || defined(TF_CATALOG_OPT_ADER_F64_DMA) || defined(TF_CATALOG_OPT_ADER_F64_K4) || defined(TF_CATALOG_OPT_ADER_F64_LA0) || defined(TF_CATALOG_OPT_ADER_F64_PAIR) || defined(TF_CATALOG_OPT_ADER_F64_PF2) || defined(TF_CATALOG_OPT_ADER_F64_ROWS) || defined(TF_CATALOG_OPT_ADER_F64_W4)
void launcher_kernel_b053681baa(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, size_t numElements, unsigned* flags, void* streamPtr);
#endif
/* deriv_f64_plain, deriv_f64_tuned */
void launcher_kernel_7d2f2effa5(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, size_t numElements, unsigned* flags, void* streamPtr);
/* deriv_na_f64_plain, deriv_na_f64_tuned */
void launcher_kernel_e957b6379b(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, unsigned m5_extraOffset, const double* m6, const double* m7, unsigned m7_extraOffset, const double* m8, unsigned m8_extraOffset, const double* m9, size_t numElements, unsigned* flags, void* streamPtr);
/* few_empty_term */
void launcher_kernel_cca5f863e5(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, const double* m8, unsigned m8_extraOffset, const double* m9, size_t numElements, unsigned* flags, void* streamPtr);
/* flux_local_mod_f64_plain, flux_local_mod_f64_tuned */
void launcher_kernel_28ade16a80(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, double* m3, unsigned m3_extraOffset, const double* m4, size_t numElements, unsigned* flags, void* streamPtr);
/* flux_local_orig_f64_plain, flux_local_orig_f64_tuned */
void launcher_kernel_695e8244f6(const double* m0, const double* m1, unsigned m1_extraOffset, const double* m2, unsigned m2_extraOffset, double* m3, unsigned m3_extraOffset, const double* m4, size_t numElements, unsigned* flags, void* streamPtr);
/* flux_neigh_mod_f64_plain, flux_neigh_mod_f64_tuned */
void launcher_kernel_4d655b5e57(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, const double* m3, double* m4, unsigned m4_extraOffset, const double* m5, size_t numElements, unsigned* flags, void* streamPtr);
/* flux_neigh_orig_f64_plain, flux_neigh_orig_f64_tuned */
void launcher_kernel_24cdb11734(const double* m0, const double* m1, unsigned m1_extraOffset, const double* m2, const double* m3, unsigned m3_extraOffset, double* m4, unsigned m4_extraOffset, const double* m5, size_t numElements, unsigned* flags, void* streamPtr);
#if defined(TF_CATALOG_GEMM_F32_PLAIN) || defined(TF_CATALOG_GEMM_F32_TUNED)
void launcher_kernel_368dd01f68(float* m0, unsigned m0_extraOffset, const float* m1, const float* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
#elif defined(TF_CATALOG_GEMM_F64_MFMA_FP64) || defined(TF_CATALOG_GEMM_F64_PLAIN) || defined(TF_CATALOG_GEMM_F64_TUNED) || defined(TF_CATALOG_OPT_GEMM_F64_K4) || defined(TF_CATALOG_OPT_GEMM_F64_LA0) || defined(TF_CATALOG_OPT_GEMM_F64_MFMA64W4K8REGS) || defined(TF_CATALOG_OPT_GEMM_F64_MFMA64W8K8ACC) || defined(TF_CATALOG_OPT_GEMM_F64_MFMA64W8K8END) || defined(TF_CATALOG_OPT_GEMM_F64_PAIR) || defined(TF_CATALOG_OPT_GEMM_F64_PF2) || defined(TF_CATALOG_OPT_GEMM_F64_W4)
void launcher_kernel_368dd01f68(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
#endif
/* inplace_chain_20x70 */
void launcher_kernel_50ca05ee0c(double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, const double* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* inplace_gemm_41_sparse */
void launcher_kernel_2e103479a9(double* m0, unsigned m0_extraOffset, const double* m1, size_t numElements, unsigned* flags, void* streamPtr);
/* inplace_gemm_56 */
void launcher_kernel_79587ab2d2(double* m0, unsigned m0_extraOffset, const double* m1, size_t numElements, unsigned* flags, void* streamPtr);
/* inplace_gemm_70_q30 */
void launcher_kernel_60bfedee1e(double* m0, unsigned m0_extraOffset, const double* m1, size_t numElements, unsigned* flags, void* streamPtr);
#if defined(TF_CATALOG_INPLACE_GEMM_84_Q13)
void launcher_kernel_ef20024dca(double* m0, unsigned m0_extraOffset, const double* m1, size_t numElements, unsigned* flags, void* streamPtr);
#elif defined(TF_CATALOG_INPLACE_GEMM_84_Q13_F32)
void launcher_kernel_ef20024dca(float* m0, unsigned m0_extraOffset, const float* m1, size_t numElements, unsigned* flags, void* streamPtr);
#endif
/* inplace_volume_20 */
void launcher_kernel_b042afe2ce(double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, size_t numElements, unsigned* flags, void* streamPtr);
/* inplace_volume_70_f32 */
void launcher_kernel_00f28504d5(float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, const float* m2, size_t numElements, unsigned* flags, void* streamPtr);
/* inplace_volume_84 */
void launcher_kernel_db3b423e76(double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_chain_13x6x29_q4, matrix_staged_chain_13x6x29_q4, t_matrix_chain_13x6x29_q4_auto, t_matrix_chain_13x6x29_q4_plain */
void launcher_kernel_83309835bc(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, double* m3, unsigned m3_extraOffset, const double* m4, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_chain_20x70x20, matrix_staged_chain_20x70x20, opt_t_matrix_chain_20x70x20_vector, t_matrix_chain_20x70x20_auto, t_matrix_chain_20x70x20_plain */
void launcher_kernel_4507257447(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, double* m3, unsigned m3_extraOffset, const double* m4, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_chain_37x18x50_f32, matrix_staged_chain_37x18x50_f32, t_matrix_chain_37x18x50_f32_auto, t_matrix_chain_37x18x50_f32_plain */
void launcher_kernel_3986b41b4e(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, const float* m2, float* m3, unsigned m3_extraOffset, const float* m4, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_chain_56x21x56, matrix_staged_chain_56x21x56, t_matrix_chain_56x21x56_auto, t_matrix_chain_56x21x56_plain */
void launcher_kernel_286f279ee6(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, double* m3, unsigned m3_extraOffset, const double* m4, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_gemm_16x16_q1, matrix_staged_gemm_16x16_q1, t_matrix_gemm_16x16_q1_auto, t_matrix_gemm_16x16_q1_plain */
void launcher_kernel_62a7014a00(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_gemm_18x21_q8, matrix_staged_gemm_18x21_q8, t_matrix_gemm_18x21_q8_auto, t_matrix_gemm_18x21_q8_plain */
void launcher_kernel_1e872f8b7f(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_gemm_33x35_q10, matrix_staged_gemm_33x35_q10, t_matrix_gemm_33x35_q10_auto, t_matrix_gemm_33x35_q10_plain */
void launcher_kernel_52fd62987d(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_gemm_50x33_q16_f32, matrix_staged_gemm_50x33_q16_f32, t_matrix_gemm_50x33_q16_f32_auto, t_matrix_gemm_50x33_q16_f32_plain */
void launcher_kernel_0101b257e7(float* m0, unsigned m0_extraOffset, const float* m1, const float* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_gemm_57x60, matrix_staged_gemm_57x60, t_matrix_gemm_57x60_auto, t_matrix_gemm_57x60_plain */
void launcher_kernel_a48511a2a0(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_gemm_5x3, matrix_staged_gemm_5x3, t_matrix_gemm_5x3_auto, t_matrix_gemm_5x3_plain */
void launcher_kernel_c2a08e2d8b(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_gemm_7x5_f32, matrix_staged_gemm_7x5_f32, t_matrix_gemm_7x5_f32_auto, t_matrix_gemm_7x5_f32_plain */
void launcher_kernel_d47df54798(float* m0, unsigned m0_extraOffset, const float* m1, const float* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_gemm_84x83, matrix_staged_gemm_84x83, t_matrix_gemm_84x83_auto, t_matrix_gemm_84x83_plain */
void launcher_kernel_d6949a2e25(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_volume_12, matrix_staged_volume_12, t_matrix_volume_12_auto, t_matrix_volume_12_plain */
void launcher_kernel_df0187eec2(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_volume_35, matrix_staged_volume_35, t_matrix_volume_35_auto, t_matrix_volume_35_plain */
void launcher_kernel_86fefd5e47(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_volume_41x47_q5, matrix_staged_volume_41x47_q5, t_matrix_volume_41x47_q5_auto, t_matrix_volume_41x47_q5_plain */
void launcher_kernel_f4590f8b42(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_volume_61x59_f32, matrix_staged_volume_61x59_f32, t_matrix_volume_61x59_f32_auto, t_matrix_volume_61x59_f32_plain */
void launcher_kernel_187c9a7d18(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, float* m2, unsigned m2_extraOffset, const float* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_volume_84x84, matrix_staged_volume_84x84, t_matrix_volume_84x84_auto, t_matrix_volume_84x84_plain */
void launcher_kernel_11f23039a7(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* matrix_direct_volume_90x30_f32, matrix_staged_volume_90x30_f32, t_matrix_volume_90x30_f32_auto, t_matrix_volume_90x30_f32_plain */
void launcher_kernel_5319ef52cf(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, float* m2, unsigned m2_extraOffset, const float* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* pw_clamp_scale_f64 */
void launcher_kernel_b29a95e19f(double* m0, unsigned m0_extraOffset, double m1, size_t numElements, unsigned* flags, void* streamPtr);
/* pw_plastic_f64 */
void launcher_kernel_fdf3bc3ba2(double* m0, unsigned m0_extraOffset, double m1, double m2, size_t numElements, unsigned* flags, void* streamPtr);
#if defined(TF_CATALOG_PW_UPDATE_F32)
void launcher_kernel_7f0eba5235(float* m0, unsigned m0_extraOffset, float m1, const float* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
#elif defined(TF_CATALOG_PW_UPDATE_F64)
void launcher_kernel_7f0eba5235(double* m0, unsigned m0_extraOffset, double m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
#endif
/* t_a_atrans_bc_auto, t_a_atrans_bc_plain */
void launcher_kernel_76147a2fe4(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, const float* m2, unsigned m2_extraOffset, float* m3, unsigned m3_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_ab_transb_auto, t_ab_transb_plain */
void launcher_kernel_29e2cb8b24(const float* m0, const float* m1, unsigned m1_extraOffset, float** m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_abb_trans_auto, t_abb_trans_plain */
void launcher_kernel_69ab6e1327(const float* m0, const float* m1, unsigned m1_extraOffset, float** m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_bbox_auto, t_bbox_plain */
void launcher_kernel_9ebda1b851(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_csa_auto, t_csa_plain */
void launcher_kernel_2304a85efa(float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, const float* m2, unsigned m2_extraOffset, float m3, size_t numElements, unsigned* flags, void* streamPtr);
/* t_dense_sparse_auto, t_dense_sparse_plain */
void launcher_kernel_54b5fd2a96(double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, size_t numElements, unsigned* flags, void* streamPtr);
/* t_few_gemm_41x38_auto, t_few_gemm_41x38_plain */
void launcher_kernel_5b78b5f2a0(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_few_gemm_70x30_q13_f32_auto, t_few_gemm_70x30_q13_f32_plain */
void launcher_kernel_e68807b4c9(float* m0, unsigned m0_extraOffset, const float* m1, const float* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_few_gemm_9x4_q1_auto, t_few_gemm_9x4_q1_plain */
void launcher_kernel_4c6db7f131(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_few_volume_10_auto, t_few_volume_10_plain */
void launcher_kernel_a4ac5f0ee0(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* t_few_volume_35x29_q6_auto, t_few_volume_35x29_q6_plain */
void launcher_kernel_4ad28f7e1c(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* t_few_volume_57x58_f32_auto, t_few_volume_57x58_f32_plain */
void launcher_kernel_97f4bb87ef(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, float* m2, unsigned m2_extraOffset, const float* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* t_few_volume_83x84_f32_auto, t_few_volume_83x84_f32_plain */
void launcher_kernel_bafcf4791a(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, float* m2, unsigned m2_extraOffset, const float* m3, size_t numElements, unsigned* flags, void* streamPtr);
/* t_five_multiplies_auto, t_five_multiplies_plain */
void launcher_kernel_b3ac723cd6(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, const float* m2, unsigned m2_extraOffset, float* m3, unsigned m3_extraOffset, const float* m4, unsigned m4_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_four_matrices_auto, t_four_matrices_plain */
void launcher_kernel_91fe0bc499(const float** m0, unsigned m0_extraOffset, const float** m1, unsigned m1_extraOffset, const float** m2, unsigned m2_extraOffset, float** m3, unsigned m3_extraOffset, const float** m4, unsigned m4_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_fused_ader_pw */
void launcher_kernel_94a4439897(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, size_t numElements, unsigned* flags, void* streamPtr);
/* t_fused_ader_update */
void launcher_kernel_6446c327d1(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, double m8, size_t numElements, unsigned* flags, void* streamPtr);
/* t_fused_gemm_pw */
void launcher_kernel_b29192cb71(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, double m3, size_t numElements, unsigned* flags, void* streamPtr);
/* t_gemm_NN_auto, t_gemm_NN_plain */
void launcher_kernel_6e01ab8126(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
#if defined(TF_CATALOG_T_GEMM_NT_AUTO) || defined(TF_CATALOG_T_GEMM_NT_PLAIN)
void launcher_kernel_96432036d0(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
#elif defined(TF_CATALOG_T_GEMM_OVERWRITE_F32_AUTO) || defined(TF_CATALOG_T_GEMM_OVERWRITE_F32_PLAIN)
void launcher_kernel_96432036d0(float* m0, unsigned m0_extraOffset, const float* m1, const float* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
#endif
/* t_gemm_TN_auto, t_gemm_TN_plain */
void launcher_kernel_a779e024e5(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_gemm_TT_auto, t_gemm_TT_plain */
void launcher_kernel_d87115cd03(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_gemm_alpha_beta_auto, t_gemm_alpha_beta_plain, t_gemm_alpha_runtime_auto, t_gemm_alpha_runtime_plain */
void launcher_kernel_e4b6145dcf(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, double m3, size_t numElements, unsigned* flags, void* streamPtr);
/* t_gemm_ptr_auto, t_gemm_ptr_plain */
void launcher_kernel_b980bf180b(double** m0, unsigned m0_extraOffset, const double** m1, unsigned m1_extraOffset, const double** m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_gemm_strided_a_auto, t_gemm_strided_a_plain */
void launcher_kernel_2a2994fb98(double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_lane_wide_auto, t_lane_wide_plain */
void launcher_kernel_6fedf5eca0(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_mat_vec_auto, t_mat_vec_plain */
void launcher_kernel_090c1dade6(float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, const float* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_pw_big */
void launcher_kernel_0ed654b475(double* m0, unsigned m0_extraOffset, const double** m1, unsigned m1_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_pw_math_f32 */
void launcher_kernel_dd6bffcae1(const float* m0, unsigned m0_extraOffset, float* m1, unsigned m1_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_pw_types */
void launcher_kernel_aaf02c8336(const double** m0, unsigned m0_extraOffset, const double* m1, const double* m2, double m3, double* m4, unsigned m4_extraOffset, const int* m5, unsigned m5_extraOffset, int* m6, unsigned m6_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_redundant_load_opt_auto, t_redundant_load_opt_plain */
void launcher_kernel_ed08ba6408(const float* m0, const float* m1, unsigned m1_extraOffset, const float* m2, float* m3, unsigned m3_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_sparse_dense_auto, t_sparse_dense_plain */
void launcher_kernel_36af273b53(double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_three_index_auto, t_three_index_plain */
void launcher_kernel_adf4365f94(double* m0, unsigned m0_extraOffset, const double* m1, const double* m2, unsigned m2_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* t_three_matrices_auto, t_three_matrices_plain */
void launcher_kernel_b25546c4ce(const float* m0, unsigned m0_extraOffset, const float* m1, unsigned m1_extraOffset, float* m2, unsigned m2_extraOffset, const float* m3, unsigned m3_extraOffset, size_t numElements, unsigned* flags, void* streamPtr);
/* ader_mixed_f64: per-order chains (libtf_ader_mixed_f64_tuned.so and libtf_ader_mixed_f64_plain.so) */
void launcher_kernel_ccc1657a1a(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, size_t numElements, unsigned* flags, void* streamPtr);
void launcher_kernel_a81cd80dd1(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, size_t numElements, unsigned* flags, void* streamPtr);
void launcher_kernel_9672d80e8e(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, size_t numElements, unsigned* flags, void* streamPtr);
void launcher_kernel_85279e58a1(const double* m0, unsigned m0_extraOffset, const double* m1, unsigned m1_extraOffset, double* m2, unsigned m2_extraOffset, const double* m3, const double* m4, unsigned m4_extraOffset, const double* m5, const double* m6, unsigned m6_extraOffset, const double* m7, size_t numElements, unsigned* flags, void* streamPtr);
/* ader_mixed_f64: one persistent launch over all orders (libtf_ader_mixed_f64_tuned.so); no counterpart in the reference */
void launcher_grouped_33116b924b(const double* g0_m0, unsigned g0_m0_extraOffset, const double* g0_m1, unsigned g0_m1_extraOffset, double* g0_m2, unsigned g0_m2_extraOffset, const double* g0_m3, const double* g0_m4, unsigned g0_m4_extraOffset, const double* g0_m5, const double* g0_m6, unsigned g0_m6_extraOffset, const double* g0_m7, size_t g0_numElements, unsigned* g0_flags, const double* g1_m0, unsigned g1_m0_extraOffset, const double* g1_m1, unsigned g1_m1_extraOffset, double* g1_m2, unsigned g1_m2_extraOffset, const double* g1_m3, const double* g1_m4, unsigned g1_m4_extraOffset, const double* g1_m5, const double* g1_m6, unsigned g1_m6_extraOffset, const double* g1_m7, size_t g1_numElements, unsigned* g1_flags, const double* g2_m0, unsigned g2_m0_extraOffset, const double* g2_m1, unsigned g2_m1_extraOffset, double* g2_m2, unsigned g2_m2_extraOffset, const double* g2_m3, const double* g2_m4, unsigned g2_m4_extraOffset, const double* g2_m5, const double* g2_m6, unsigned g2_m6_extraOffset, const double* g2_m7, size_t g2_numElements, unsigned* g2_flags, const double* g3_m0, unsigned g3_m0_extraOffset, const double* g3_m1, unsigned g3_m1_extraOffset, double* g3_m2, unsigned g3_m2_extraOffset, const double* g3_m3, const double* g3_m4, unsigned g3_m4_extraOffset, const double* g3_m5, const double* g3_m6, unsigned g3_m6_extraOffset, const double* g3_m7, size_t g3_numElements, unsigned* g3_flags, const double* g4_m0, unsigned g4_m0_extraOffset, const double* g4_m1, unsigned g4_m1_extraOffset, double* g4_m2, unsigned g4_m2_extraOffset, const double* g4_m3, const double* g4_m4, unsigned g4_m4_extraOffset, const double* g4_m5, const double* g4_m6, unsigned g4_m6_extraOffset, const double* g4_m7, size_t g4_numElements, unsigned* g4_flags, const double* g5_m0, unsigned g5_m0_extraOffset, const double* g5_m1, unsigned g5_m1_extraOffset, double* g5_m2, unsigned g5_m2_extraOffset, const double* g5_m3, const double* g5_m4, unsigned g5_m4_extraOffset, const double* g5_m5, const double* g5_m6, unsigned g5_m6_extraOffset, const double* g5_m7, size_t g5_numElements, unsigned* g5_flags, void* streamPtr);
#ifdef __cplusplus
}
#endif
#endif

// 16 x 16 x 4 matrix-core products of the M -> G kernels (gfx950).
#ifndef G4ACC_MFMA16_HPP
#define G4ACC_MFMA16_HPP

namespace g4acc {

template <typename Real>
struct Mfma16;
// Output row of register i of a lane in lane group jl = lane / 16 (the column is lane % 16). The
// two instructions differ (measured on gfx950): FP32 holds four consecutive rows per lane, FP64
// rows strided by four.
template <>
struct Mfma16<float> {
  typedef float acc_t __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int jl, int i) { return 4 * jl + i; }
};
template <>
struct Mfma16<double> {
  typedef double acc_t __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int jl, int i) { return jl + 4 * i; }
};

}  // namespace g4acc

#endif

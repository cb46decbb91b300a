#include "lfw_xpar64_mm.hpp"
namespace t2fw {
template<bool F> __global__ __launch_bounds__(256,3) void kf(XparFwdArgs p){ extern __shared__ __align__(16) unsigned char s[]; mm::forward_chunk<F>(p,*reinterpret_cast<mm::Smem*>(s),blockIdx.x%p.B,(int)(blockIdx.x/p.B)); }
template<int S,bool F,int O> __global__ __launch_bounds__(256,O) void kb(XparBwdArgs p){ extern __shared__ __align__(16) unsigned char s[]; mm::backward_chunk<S,F>(p,*reinterpret_cast<mm::Smem*>(s),blockIdx.x%p.B,(int)(blockIdx.x/p.B)); }
template __global__ void kf<true>(XparFwdArgs);
template __global__ void kf<false>(XparFwdArgs);
template __global__ void kb<0,true,2>(XparBwdArgs);
template __global__ void kb<1,true,2>(XparBwdArgs);
template __global__ void kb<0,false,2>(XparBwdArgs);
template __global__ void kb<0,true,3>(XparBwdArgs);
}

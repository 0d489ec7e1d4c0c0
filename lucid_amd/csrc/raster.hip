// Tile rasterisation, per-pixel depth ordering and front-to-back blending
// (≙ data/shaders/raster_low.glsl, raster_high.glsl, shared/raster.glsl, shared/shading.glsl).
//
// Kernels (wave64; an 8x8 block of pixels is one wave, one lane per pixel):
//   rowgen_low   one work-group per bin with fewer than 1024 triangles: block lists with the
//                reference's 8-row scanline rule; promotes the bin to the high path when an 8x8
//                block holds more than 256 triangles (raster_low.glsl:39-106,229-237), and
//                generates it again as a high bin.
//   rowgen_high  kRowgenSplitThreads threads per high bin (eight work-groups, or four larger ones
//                in the launch that takes low and high bins, rowgen_fused): block lists with the
//                4-row rule of raster_high.glsl:54-90. (Their space is the bin categories' work.)
//   high_finalize  long block lists of high bins are sorted by centroid depth (bitonic, in
//                registers and LDS, whole work-group) and split into depth ranges so that several
//                waves share a dense block; lists beyond 2048 entries in high_finalize_long.
//   block_raster one wave per block: sorts short lists itself in registers, turns the coverage
//                masks into per-pixel entry bitmaps, shades and blends front to back; pre-sorted
//                blocks take one wave per depth range (block_raster_big; both kinds in one launch:
//                block_raster_fused).
//   fallback     exact per-pixel sort for pixels whose speculative order was violated.
//
// Exact ordering: triangles of a block are pre-sorted by the depth at their covered-pixel
// centroid. Each pixel lane consumes its fragments in that order through a K-entry insertion
// window keyed by (depth at the pixel, triangle id) and checks every arrival against the last
// emitted key. If no arrival is ever smaller than the last emitted key, the emitted sequence is
// exactly the per-pixel sorted order; otherwise the pixel is queued for the fallback kernel,
// which sorts its full fragment list (LDS bitonic, global-memory spill for deep pixels).
// Ties in depth are ordered by triangle id.
#include "lucid_device.h"

namespace lucid {

constexpr int kSortThreads = 256;
constexpr int kFallbackThreads = 256;
constexpr int kWindow = 4;
// The narrow ordering window (tuning window 1) of flat records: one slot, in the register-sorted
// blocks and in the pre-sorted ones (whose depth ranks keep 32 - log2 of the padded list length
// bits). Other records keep four: where surfaces cross, fewer send too many pixels to the exact sort,
// which costs them more (640 x 360, 250 crossing planes, four slots against one with plain records
// and two with general ones: 465 against 2275 us a frame, 486 against 665).
constexpr int kNarrowWindow = 1;
constexpr int kFallbackCap = 512; // fragments per pixel sorted in LDS by the fallback kernel

// ------------------------------------------------------------------ shading

__device__ __forceinline__ float srgb_to_linear(float x) {
	return x < 0.04045f ? (1.0f / 12.92f) * x : glsl_pow((x + 0.055f) * (1.0f / 1.055f), 2.4f);
}
__device__ __forceinline__ float linear_to_srgb(float x) {
	return x < 0.0031308f ? 12.92f * x : 1.055f * glsl_pow(x, 1.0f / 2.4f) - 0.055f;
}

__device__ __forceinline__ float sample_inv_depth(const FrameBufs &b, uint32_t t, float px,
												  float py) {
	uint4 d = b.tri_depth[tri_rec(b, t)];
	return bits2f(d.x) * px + (bits2f(d.y) * py + bits2f(d.z));
}

// Shaded sample colour: RGBA8 word in the reference's quantised mode (0 = contributes
// nothing, shading.glsl:167-168,274) or fp32 with LUCID_OPT_FP32_SAMPLES.
template <bool FP32> struct SampleColor;
template <> struct SampleColor<false> {
	uint32_t enc;
	// component-wise select (keeps struct selects in registers)
	static __device__ __forceinline__ SampleColor sel(bool p, SampleColor a, SampleColor b) {
		SampleColor o;
		o.enc = p ? a.enc : b.enc;
		return o;
	}
	__device__ __forceinline__ bool contributes() const { return enc != 0; }
	__device__ __forceinline__ float4 rgba() const { return decode_rgba8(enc); }
	__device__ __forceinline__ void zero() { enc = 0; }
	__device__ __forceinline__ SampleColor read(int src) const {
		SampleColor o;
		o.enc = wave_read(enc, src);
		return o;
	}
};
template <> struct SampleColor<true> {
	float4 col;
	static __device__ __forceinline__ SampleColor sel(bool p, SampleColor a, SampleColor b) {
		SampleColor o;
		o.col.x = p ? a.col.x : b.col.x;
		o.col.y = p ? a.col.y : b.col.y;
		o.col.z = p ? a.col.z : b.col.z;
		o.col.w = p ? a.col.w : b.col.w;
		return o;
	}
	__device__ __forceinline__ bool contributes() const { return col.w != 0.0f; }
	__device__ __forceinline__ float4 rgba() const { return col; }
	__device__ __forceinline__ void zero() { col = make_float4(0, 0, 0, 0); }
	__device__ __forceinline__ SampleColor read(int src) const {
		SampleColor o;
		o.col.x = wave_read(col.x, src), o.col.y = wave_read(col.y, src);
		o.col.z = wave_read(col.z, src), o.col.w = wave_read(col.w, src);
		return o;
	}
};

// sRGB round trip of finalShading, s = L2S(S2L(x) * f), unclamped. fp = f^(1/2.4).
// Above both linear segments the two powers cancel: L2S(S2L(x) f) = (x + 0.055) fp - 0.055
// exactly (the threshold S2L(x) f >= 0.0031308 is (x + 0.055) fp >= kSrgbHiU); below both,
// s = 12.92 ((x / 12.92) f) with the reference's own operations. Only lanes in neither
// case (or in a NaN case) evaluate the powers, in a branch the wave skips when none is.
constexpr float kSrgbHiU = 0.09544991f; // 1.055 * 0.0031308^(1/2.4)
struct LitChannel {
	float s;     // L2S(S2L(x) f) before the clamp
	float deriv; // ds/dx
};
template <bool DERIV>
__device__ __forceinline__ LitChannel lit_channel(float x, float f, float fp) {
	const float u = (x + 0.055f) * fp;
	const float lin_lo = (1.0f / 12.92f) * x;
	const bool hi = x >= 0.04045f && u >= kSrgbHiU;
	const bool lo = x < 0.04045f && lin_lo * f < 0.0031308f;
	LitChannel o;
	o.s = hi ? u - 0.055f : 12.92f * (lin_lo * f);
	o.deriv = hi ? fp : f;
	if(!hi && !lo) {
		const float lin = srgb_to_linear(x);
		const float y = lin * f;
		o.s = linear_to_srgb(y);
		if constexpr(DERIV) {
			// S2L'(x) = 2.4 S2L(x) / (x + 0.055), L2S'(y) = (L2S(y) + 0.055) / (2.4 y) above
			// their linear segments; no further powers
			const float d_lin = x < 0.04045f
									? (1.0f / 12.92f)
									: 2.4f * lin * __builtin_amdgcn_rcpf(x + 0.055f);
			const float d_srgb = y < 0.0031308f
									 ? 12.92f
									 : (o.s + 0.055f) * __builtin_amdgcn_rcpf(2.4f * y);
			o.deriv = d_srgb * f * d_lin;
		}
	}
	return o;
}

// ------------------------------------------------------------------ albedo textures
//
// textureGrad (shading.glsl:145-150) on an RGBA8 atlas with the reference's sampler
// (src/lucid_base.h:30: linear magnification, minification and mip filter, repeat
// addressing), restated from the Vulkan sampling rules: the scale factors are the texture
// coordinate derivatives times the level-0 size, lambda = log2(max(|d/dx|, |d/dy|))
// (isotropic), the level is clamped to [0, levels - 1] and the two nearest levels are
// blended by its fraction; within a level, bilinear weights at u = s * size - 0.5 with the
// texel indices wrapped (repeat). s is reduced to [0, 1] first (repeat is periodic).

//
// The mip levels of both atlases sit in a small LDS table (fill_tex_table), one row per atlas
// and level: a lane picks its level's size and texels with two LDS loads. Selecting them from
// the kernel arguments instead took a chain of fifteen compares and selects per level and atlas.
// The filtering is bound by VALU issue (about 70 operations per level go into the bilinear
// filter itself); 96 textured planes at 1024 x 768 (26 M fragments): 316 -> 256 us for the
// block rasteriser.
constexpr int kTexTable = 2 * 2 * kMaxTexLevels; // two uint4 per level, opaque atlas first
// Row of a level: {width, height as floats, width, height}, {texels (64 bits), number of levels of
// the atlas, its last level as a float}.

__device__ __forceinline__ void fill_tex_table(const FrameBufs &b, uint4 *s_tex) {
	const int i = threadIdx.x;
	if(i < 2 * kMaxTexLevels) {
		const int level = i % kMaxTexLevels;
		const bool second = i >= kMaxTexLevels;
		uint32_t off = 0; // (the offsets are kernel arguments: no dynamic indexing)
#pragma unroll
		for(int l = 1; l < kMaxTexLevels; l++)
			off = level == l ? (second ? b.tex[1].offset[l] : b.tex[0].offset[l]) : off;
		const int w = max(1, (second ? b.tex[1].width : b.tex[0].width) >> level);
		const int h = max(1, (second ? b.tex[1].height : b.tex[0].height) >> level);
		const int levels = second ? b.tex[1].levels : b.tex[0].levels;
		const uint64_t at = (uint64_t)((second ? b.tex[1].texels : b.tex[0].texels) + off);
		s_tex[2 * i] = make_uint4(f2bits((float)w), f2bits((float)h), (uint32_t)w, (uint32_t)h);
		s_tex[2 * i + 1] = make_uint4((uint32_t)at, (uint32_t)(at >> 32), (uint32_t)levels,
									  f2bits((float)(levels - 1)));
	}
}

// The level of table rows l: su, sv are the texture coordinates reduced to [0, 1].
__device__ __forceinline__ float4 tex_bilinear(const uint4 *l, float su, float sv) {
	const uint4 d = l[0], at = l[1];
	const int w = (int)d.z, h = (int)d.w;
	const uint32_t *texels = (const uint32_t *)(((uint64_t)at.y << 32) | at.x);
	const float u = su * bits2f(d.x) - 0.5f, uv = sv * bits2f(d.y) - 0.5f;
	const float fu = floorf(u), fv = floorf(uv);
	const float au = u - fu, av = uv - fv;
	int x0 = (int)fu, y0 = (int)fv; // in [-1, size - 1]
	x0 = x0 < 0 ? w - 1 : x0;
	y0 = y0 < 0 ? h - 1 : y0;
	const int x1 = x0 + 1 == w ? 0 : x0 + 1;
	const uint32_t row0 = (uint32_t)y0 * (uint32_t)w;
	const uint32_t row1 = y0 + 1 == h ? 0u : row0 + (uint32_t)w;
	const uint32_t t00 = texels[row0 + (uint32_t)x0], t10 = texels[row0 + (uint32_t)x1];
	const uint32_t t01 = texels[row1 + (uint32_t)x0], t11 = texels[row1 + (uint32_t)x1];
	const float4 c00 = decode_rgba8(t00), c10 = decode_rgba8(t10);
	const float4 c01 = decode_rgba8(t01), c11 = decode_rgba8(t11);
	const float bu = 1.0f - au, bv = 1.0f - av;
	float4 r;
	r.x = (c00.x * bu + c10.x * au) * bv + (c01.x * bu + c11.x * au) * av;
	r.y = (c00.y * bu + c10.y * au) * bv + (c01.y * bu + c11.y * au) * av;
	r.z = (c00.z * bu + c10.z * au) * bv + (c01.z * bu + c11.z * au) * av;
	r.w = (c00.w * bu + c10.w * au) * bv + (c01.w * bu + c11.w * au) * av;
	return r;
}

// tab: the atlas's rows of the table.
__device__ __forceinline__ float4 texture_grad(const uint4 *tab, float s, float v, float dsx,
											   float dvx, float dsy, float dvy) {
	const uint4 top = tab[0], meta = tab[1];
	const float fw = bits2f(top.x), fh = bits2f(top.y);
	const float ux = dsx * fw, vx = dvx * fh, uy = dsy * fw, vy = dvy * fh;
	// the larger of the two lengths: the square root is monotonic, so one is enough
	const float rho = sqrtf(fmx(ux * ux + vx * vx, uy * uy + vy * vy));
	const float lambda = log2f(rho);
	// magnification (or a degenerate footprint): level 0
	const float d = lambda > 0.0f ? fmn(lambda, bits2f(meta.w)) : 0.0f;
	const float fl = floorf(d);
	const int lo = (int)fl;
	const float delta = d - fl;
	const float su = s - floorf(s), sv = v - floorf(v);
	float4 r = tex_bilinear(tab + 2 * lo, su, sv);
	if(delta > 0.0f) {
		const float4 h = tex_bilinear(tab + 2 * min(lo + 1, (int)meta.z - 1), su, sv);
		const float nd = 1.0f - delta;
		r.x = r.x * nd + h.x * delta;
		r.y = r.y * nd + h.y * delta;
		r.z = r.z * nd + h.z * delta;
		r.w = r.w * nd + h.w * delta;
	}
	return r;
}

// Albedo of a textured triangle at a pixel (shading.glsl:111-122,131-159): barycentric
// derivatives from the planes one pixel right and one pixel down, the texture coordinate
// and its derivatives from the triangle's corner coordinates, the instance's uv rectangle,
// then the opaque (alpha 1) or transparent atlas. bary0/1: before the offsets are removed.
__device__ __forceinline__ float4 albedo_sample(const FrameBufs &b, const uint4 *s_tex,
												const uint4 *q, float inv_ray, float e0, float e1,
												float bary0, float bary1, float bp0, float bp1) {
	const uint32_t flags = q[0].w & 0xffffu, inst = q[0].w >> 16, t = q[6].z;
	const float dex = bits2f(q[0].x), dey = bits2f(q[0].y);
	const float ray_posx = __builtin_amdgcn_rcpf(inv_ray + dex);
	const float ray_posy = __builtin_amdgcn_rcpf(inv_ray + dey);
	const float bdx0 = (e0 + bits2f(q[1].x)) * ray_posx - bary0;
	const float bdx1 = (e1 + bits2f(q[2].x)) * ray_posx - bary1;
	const float bdy0 = (e0 + bits2f(q[1].y)) * ray_posy - bary0;
	const float bdy1 = (e1 + bits2f(q[2].y)) * ray_posy - bary1;
	const float b0 = bary0 - bp0, b1 = bary1 - bp1;
	const uint4 *tt = b.tri_tex + 2 * (size_t)tri_rec(b, t);
	const uint4 ta = tt[0], tb = tt[1];
	const float t0x = bits2f(ta.x), t0y = bits2f(ta.y), t1x = bits2f(ta.z), t1y = bits2f(ta.w);
	const float t2x = bits2f(tb.x), t2y = bits2f(tb.y);
	float s = b0 * t1x + (b1 * t2x + t0x), v = b0 * t1y + (b1 * t2y + t0y);
	float dsx = bdx0 * t1x + bdx1 * t2x, dvx = bdx0 * t1y + bdx1 * t2y;
	float dsy = bdy0 * t1x + bdy1 * t2x, dvy = bdy0 * t1y + bdy1 * t2y;
	if(flags & LUCID_INST_HAS_UV_RECT) {
		const float4 rc = b.inst_uv_rects[inst];
		s = rc.z * (s - floorf(s)) + rc.x;
		v = rc.w * (v - floorf(v)) + rc.y;
		dsx = dsx * rc.z, dsy = dsy * rc.z;
		dvx = dvx * rc.w, dvy = dvy * rc.w;
	}
	const bool opaque = (flags & LUCID_INST_TEX_OPAQUE) != 0;
	float4 col = texture_grad(s_tex + (opaque ? 0 : 2 * kMaxTexLevels), s, v, dsx, dvx, dsy, dvy);
	col.w = opaque ? 1.0f : col.w;
	return col;
}

// The shading record of triangle t, built by setup (one 128-byte line per triangle).
__device__ __forceinline__ void load_shading_record(const FrameBufs &b, uint32_t t,
													uint4 (&q)[kRecQuads]) {
	const uint4 *src = b.tri_shade + (size_t)kRecStride * tri_rec(b, t);
#pragma unroll
	for(int j = 0; j < kRecQuads; j++)
		q[j] = src[j];
}

// Depth plane at a pixel: inverse distance along the pixel's ray (shading.glsl:108).
__device__ __forceinline__ float record_inv_depth(uint4 q0, float px, float py) {
	return bits2f(q0.x) * px + (bits2f(q0.y) * py + bits2f(q0.z));
}

// Everything shadeSample (shading.glsl:107-184, no textures) computes before lighting,
// from a shading record (LDS or registers): barycentrics, the vertex colour times the
// instance colour, and the per-channel lighting factors. `inv_ray` is record_inv_depth at
// the same pixel. Returns false when the sample's alpha is 0 (it contributes nothing).
struct ShadeState {
	float bary0, bary1;
	float4 color; // interpolated vertex colour (white without one) times the instance colour
	float4 inst;  // instance colour (white without one)
	float f[3];   // lighting factors
	float fp[3];  // f^(1/2.4)
};

template <bool TEX>
__device__ __forceinline__ bool shade_prepare(const FrameConst &c, const FrameBufs &b,
											  const uint4 *s_tex, const uint4 *q, float px, float py, float inv_ray,
											  ShadeState &st) {
	const uint32_t flags = q[0].w & 0xffffu;
	const uint4 b0 = q[1], b1 = q[2];
	// GLSL's division is specified to 2.5 ulp; v_rcp_f32 (1 ulp) meets that
	float ray_pos = __builtin_amdgcn_rcpf(inv_ray);
	float e0 = bits2f(b0.x) * px + (bits2f(b0.y) * py + bits2f(b0.z));
	float e1 = bits2f(b1.x) * px + (bits2f(b1.y) * py + bits2f(b1.z));
	float bary0 = e0 * ray_pos, bary1 = e1 * ray_pos;
	float4 tex = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
	bool textured = false;
	if constexpr(TEX) {
		if(flags & LUCID_INST_HAS_ALBEDO_TEXTURE) {
			textured = true;
			tex = albedo_sample(b, s_tex, q, inv_ray, e0, e1, bary0, bary1, bits2f(b0.w), bits2f(b1.w));
		}
	}
	bary0 = bary0 - bits2f(b0.w);
	bary1 = bary1 - bits2f(b1.w);
	st.bary0 = bary0, st.bary1 = bary1;

	// vertex colour (or white), then times the instance colour; products by an exact 1.0
	// are skipped, which leaves every result bit-identical
	float4 color = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
	const uint4 q6 = q[6];
	if(flags & LUCID_INST_HAS_VERTEX_COLORS) {
		float w0 = (1.0f - bary0) - bary1;
		const uint4 q3 = q[3];
		if(c.color_mode == kColorRGBA8) {
			float4 c0 = decode_rgba8(q3.x), c1 = decode_rgba8(q3.y), c2 = decode_rgba8(q3.z);
			color.x = w0 * c0.x + (bary0 * c1.x + bary1 * c2.x);
			color.y = w0 * c0.y + (bary0 * c1.y + bary1 * c2.y);
			color.z = w0 * c0.z + (bary0 * c1.z + bary1 * c2.z);
			color.w = w0 * c0.w + (bary0 * c1.w + bary1 * c2.w);
		} else if(c.color_mode == kColorF32) {
			const uint4 q4 = q[4], q5 = q[5];
			color.x = w0 * bits2f(q3.x) + (bary0 * bits2f(q4.x) + bary1 * bits2f(q5.x));
			color.y = w0 * bits2f(q3.y) + (bary0 * bits2f(q4.y) + bary1 * bits2f(q5.y));
			color.z = w0 * bits2f(q3.z) + (bary0 * bits2f(q4.z) + bary1 * bits2f(q5.z));
			color.w = bits2f(q3.w);
		}
	}
	st.inst = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
	if(textured) {
		// shading.glsl: colour = instance colour, times the texture, times the vertex colour
		float4 f = tex;
		if(flags & LUCID_INST_HAS_COLOR) {
			const float4 ic = decode_rgba8(q6.x);
			st.inst = ic;
			f = make_float4(ic.x * tex.x, ic.y * tex.y, ic.z * tex.z, ic.w * tex.w);
		}
		color.x = f.x * color.x;
		color.y = f.y * color.y;
		color.z = f.z * color.z;
		color.w = f.w * color.w;
	} else if(flags & LUCID_INST_HAS_COLOR) {
		const float4 ic = decode_rgba8(q6.x);
		st.inst = ic;
		color.x = ic.x * color.x;
		color.y = ic.y * color.y;
		color.z = ic.z * color.z;
		color.w = ic.w * color.w;
	}
	st.color = color;
	if(color.w == 0.0f)
		return false;
	if(c.identity_light) { // every lighting factor is 1 (no normal or light value is read)
		st.f[0] = st.f[1] = st.f[2] = 1.0f;
		st.fp[0] = st.fp[1] = st.fp[2] = 1.0f;
		return true;
	}
	if(flags & LUCID_INST_HAS_VERTEX_NORMALS) {
		V3 n0 = decode_normal(q[4].w), n1 = decode_normal(q[5].w), n2 = decode_normal(q6.y);
		n1 = sub3(n1, n0);
		n2 = sub3(n2, n0);
		V3 normal = mk3(bary0 * n1.x + (bary1 * n2.x + n0.x), bary0 * n1.y + (bary1 * n2.y + n0.y),
						bary0 * n1.z + (bary1 * n2.z + n0.z));
		const float light = light_value(c, normal);
#pragma unroll
		for(int k = 0; k < 3; k++) {
			st.f[k] = light_factor(c, k, light);
			st.fp[k] = glsl_pow(st.f[k], 1.0f / 2.4f);
		}
	} else {
		const float light = bits2f(q6.w);
#pragma unroll
		for(int k = 0; k < 3; k++)
			st.f[k] = light_factor(c, k, light);
		st.fp[0] = bits2f(q[4].w), st.fp[1] = bits2f(q[5].w), st.fp[2] = bits2f(q6.y);
	}
	return true;
}

// shadeSample (shading.glsl:107-184) without textures: lighting through the sRGB round trip
// of finalShading (funcs.glsl:261-271), then RGBA8 quantisation unless FP32.
template <bool FP32, bool TEX>
__device__ __forceinline__ SampleColor<FP32> shade_record(const FrameConst &c, const FrameBufs &b,
														  const uint4 *s_tex, const uint4 *q,
														  float px, float py, float inv_ray) {
	ShadeState st;
	SampleColor<FP32> out;
	if(!shade_prepare<TEX>(c, b, s_tex, q, px, py, inv_ray, st)) {
		out.zero();
		return out;
	}
	float rgb[3] = {st.color.x, st.color.y, st.color.z};
	if(c.identity_light) {
		// L2S(S2L(x) * 1) = x: the sRGB round trip of a unit lighting factor is skipped
#pragma unroll
		for(int k = 0; k < 3; k++)
			rgb[k] = sat(rgb[k]);
	} else {
#pragma unroll
		for(int k = 0; k < 3; k++)
			rgb[k] = sat(lit_channel<false>(rgb[k], st.f[k], st.fp[k]).s);
	}
	if constexpr(FP32)
		out.col = make_float4(rgb[0], rgb[1], rgb[2], st.color.w);
	else
		out.enc = encode_rgba8_unit_rgb(rgb[0], rgb[1], rgb[2], st.color.w);
	return out;
}

// Shades triangle t at a pixel straight from the setup records (exact fallback path).
template <bool FP32, bool TEX>
__device__ __forceinline__ SampleColor<FP32> shade_sample(const FrameConst &c, const FrameBufs &b,
														  const uint4 *s_tex, uint32_t t,
														  float px, float py, float inv_ray) {
	uint4 q[kRecQuads];
	load_shading_record(b, t, q);
	return shade_record<FP32, TEX>(c, b, s_tex, q, px, py, inv_ray);
}

__device__ __forceinline__ uint64_t pixel_key(float inv_ray, uint32_t t) {
	return ((uint64_t)inv_ord_f32(inv_ray) << 32) | t;
}

// ------------------------------------------------------------------ per-pixel state

struct Accum {
	float cr, cg, cb, tr;
	__device__ __forceinline__ void init() { cr = cg = cb = 0.0f, tr = 1.0f; }
	// shading.glsl:276-283 (front-to-back "over"; additive variant)
	__device__ __forceinline__ void blend(float4 col, bool additive) {
		if(additive) {
			cr = cr + col.x * col.w;
			cg = cg + col.y * col.w;
			cb = cb + col.z * col.w;
		} else {
			cr = cr + (col.x * col.w) * tr;
			cg = cg + (col.y * col.w) * tr;
			cb = cb + (col.z * col.w) * tr;
			tr = tr * (1.0f - col.w);
		}
	}
	// The same for an RGBA8 sample (bytes c and a): the byte scales fold into one weight per
	// sample, so each channel takes one fused multiply-add, cr += c (a tr / 255) with
	// a = byte / 255 (the sums differ from blend()'s by rounding only; the transmittance
	// step is blend()'s, operation for operation).
	__device__ __forceinline__ void blend(SampleColor<false> s, bool additive) {
		const float a = (float)(s.enc >> 24) * (1.0f / 255.0f);
		const float w = (additive ? a : a * tr) * (1.0f / 255.0f);
		cr = fmaf((float)(s.enc & 0xffu), w, cr);
		cg = fmaf((float)((s.enc >> 8) & 0xffu), w, cg);
		cb = fmaf((float)((s.enc >> 16) & 0xffu), w, cb);
		if(!additive)
			tr = tr * (1.0f - a);
	}
	__device__ __forceinline__ void blend(SampleColor<true> s, bool additive) { blend(s.col, additive); }
};

// Sample order key: nearer (larger inverse depth) first, equal depths by triangle id.
constexpr uint64_t kEmptyKey = ~0ull;

// Per-pixel ordering window of kWindow pending samples (payload P) in fixed slots. A
// sample that arrives when the window is full pushes out the nearest of the five, which is
// handed to the emit callback, so samples leave front to back. The pixel is exact iff the
// emitted keys strictly increase; otherwise `bad` marks it for the exact per-pixel sort.
// Slots are updated in place by selects: no register rotation and no dynamic indexing.
// P provides zero() and a component-wise static sel(bool, P, P).
template <class P>
struct OrderWindow {
	uint64_t k0, k1, k2, k3;
	P c0, c1, c2, c3;
	uint32_t n;           // filled slots
	uint64_t first, last; // first and last emitted key (0 before the first)
	bool bad;

	__device__ __forceinline__ void init() {
		k0 = k1 = k2 = k3 = kEmptyKey;
		c0.zero(), c1.zero(), c2.zero(), c3.zero();
		n = 0, first = last = 0, bad = false;
	}

	template <class F> __device__ __forceinline__ void emit(uint64_t k, const P &col, F &&f) {
		bad |= k <= last;
		first = last == 0ull ? k : first;
		last = k;
		f(col);
	}

	template <class F> __device__ __forceinline__ void insert(uint64_t key, const P &col, F &&f) {
		static_assert(kWindow == 4, "window slots are spelled out");
		if(n < (uint32_t)kWindow) {
			k0 = n == 0 ? key : k0, c0 = P::sel(n == 0, col, c0);
			k1 = n == 1 ? key : k1, c1 = P::sel(n == 1, col, c1);
			k2 = n == 2 ? key : k2, c2 = P::sel(n == 2, col, c2);
			k3 = n == 3 ? key : k3, c3 = P::sel(n == 3, col, c3);
			n++;
			return;
		}
		// nearest pending sample by a two-level tournament
		const bool a = k1 < k0, bq = k3 < k2;
		const uint64_t ka = a ? k1 : k0, kb = bq ? k3 : k2;
		const P ca = P::sel(a, c1, c0), cb = P::sel(bq, c3, c2);
		const bool m = kb < ka;
		const uint64_t km = m ? kb : ka;
		const P cm = P::sel(m, cb, ca);
		const bool take_new = key < km;
		emit(take_new ? key : km, P::sel(take_new, col, cm), f);
		// the new sample takes the emitted slot
		const bool s0 = !take_new && !m && !a, s1 = !take_new && !m && a;
		const bool s2 = !take_new && m && !bq, s3 = !take_new && m && bq;
		k0 = s0 ? key : k0, c0 = P::sel(s0, col, c0);
		k1 = s1 ? key : k1, c1 = P::sel(s1, col, c1);
		k2 = s2 ? key : k2, c2 = P::sel(s2, col, c2);
		k3 = s3 ? key : k3, c3 = P::sel(s3, col, c3);
	}

	template <class F> __device__ __forceinline__ void flush(F &&f) {
		for(uint32_t r = 0; r < n; r++) {
			const bool a = k1 < k0, bq = k3 < k2;
			const uint64_t ka = a ? k1 : k0, kb = bq ? k3 : k2;
			const P ca = P::sel(a, c1, c0), cb = P::sel(bq, c3, c2);
			const bool m = kb < ka;
			emit(m ? kb : ka, P::sel(m, cb, ca), f);
			const bool s0 = !m && !a, s1 = !m && a, s2 = m && !bq, s3 = m && bq;
			k0 = s0 ? kEmptyKey : k0;
			k1 = s1 ? kEmptyKey : k1;
			k2 = s2 ? kEmptyKey : k2;
			k3 = s3 ? kEmptyKey : k3;
		}
		n = 0;
	}
};

// Smaller ordering windows (N = 1 or 2 pending samples), same contract as OrderWindow: for
// lists whose block order is already (nearly) each pixel's depth order, where the window
// only has to catch neighbours in the wrong order; a pixel it cannot put in order is still
// detected (bad) and sorted exactly.
//
// The slots are in order, k0 <= k1. While every lane's new sample is behind its pending ones, the
// window is a queue: k0 leaves, no key is compared with the last emitted one and nothing is
// selected; the wave tests for that with one comparison. (A pending key is never before `last`: a
// new key before k0 leaves at once, as the smallest.) Otherwise the wave takes the selects. The
// walks are bound by VALU issue (75 -> 60 instructions per flat sample): both block kernels of 1 M
// soup triangles at 1080p 203 -> 190 us, of the 32-frame batch 1800 -> 1650, pass A of the fp32
// soup (41 M fragments at 512 x 512) 178 -> 160.
template <class P, int N>
struct SmallWindow {
	static_assert(N == 1 || N == 2, "one or two slots");
	static constexpr bool PH = N == 1;
	// Free slots hold placeholders (key 0, below every sample key; a zero payload), which the first
	// samples push out, so no fill count is kept. PH (the forward's one slot): they are emitted like
	// samples, and the blend treats the zero payload as nothing; the backward's order recording (two
	// slots) does not. The keys of one pixel are distinct (one sample per triangle).
	uint64_t k0, k1;
	P c0, c1;
	uint64_t first, last; // first and last emitted key (0 before the first)
	uint32_t bad;         // samples that came after a later one had left

	__device__ __forceinline__ void init() {
		k0 = k1 = 0ull;
		c0.zero(), c1.zero();
		first = last = 0, bad = 0;
	}
	template <class F> __device__ __forceinline__ void emit(uint64_t k, const P &col, F &&f) {
		if(PH || k != 0ull) {
			first = last == 0ull ? k : first;
			last = k;
			f(col);
		}
	}
	template <class F> __device__ __forceinline__ void insert(uint64_t key, const P &col, F &&f) {
		const uint64_t back = N == 1 ? k0 : k1;
		uint64_t ke = k0, n0 = N == 1 ? key : k1, n1 = key;
		P ce, m0, m1;
		ce = c0, m1 = col;
		if constexpr(N == 1)
			m0 = col;
		else
			m0 = c1;
		if(ballot(key < back || (!PH && k0 == 0ull))) {
			const bool a = key < k0, b = key < back;
			bad += key < last ? 1u : 0u;
			ke = a ? key : k0, ce = P::sel(a, col, ce);
			if constexpr(N == 1) {
				n0 = a ? k0 : key, m0 = P::sel(a, c0, col);
			} else {
				n0 = a ? k0 : b ? key : k1, n1 = b ? k1 : key;
				const P t = P::sel(b, col, c1);
				m0 = P::sel(a, c0, t), m1 = P::sel(b, c1, col);
			}
		}
		k0 = n0, c0 = m0;
		if constexpr(N == 2)
			k1 = n1, c1 = m1;
		emit(ke, ce, f);
	}
	template <class F> __device__ __forceinline__ void flush(F &&f) {
		emit(k0, c0, f); // the last samples, or placeholders
		if constexpr(N == 2)
			emit(k1, c1, f);
		k0 = k1 = 0ull;
		c0.zero(), c1.zero();
	}
};

// Forward per-pixel state: the ordering window (N slots) feeding the front-to-back blend.
template <bool FP32, int N = kWindow>
struct PixelState {
	std::conditional_t<N == kWindow, OrderWindow<SampleColor<FP32>>, SmallWindow<SampleColor<FP32>, N>> w;
	Accum acc;

	__device__ __forceinline__ void init() {
		w.init();
		acc.init();
	}
	__device__ __forceinline__ void insert(uint64_t key, SampleColor<FP32> col, bool additive) {
		w.insert(key, col, [&](const SampleColor<FP32> &s) { acc.blend(s, additive); });
	}
	__device__ __forceinline__ void flush(bool additive) {
		w.flush([&](const SampleColor<FP32> &s) { acc.blend(s, additive); });
	}
};

__device__ __forceinline__ void write_pixel(const FrameConst &c, const FrameBufs &b, int px,
											int py, const Accum &a, uint32_t count) {
	if(px >= c.width || py >= c.height)
		return;
	float r = sat(a.cr + a.tr * c.background[0]);
	float g = sat(a.cg + a.tr * c.background[1]);
	float bl = sat(a.cb + a.tr * c.background[2]);
	size_t o = (size_t)py * c.width + px;
	if(b.image) {
		uint32_t v = f2u(r * 255.0f + 0.5f) | (f2u(g * 255.0f + 0.5f) << 8) |
					 (f2u(bl * 255.0f + 0.5f) << 16) | (255u << 24);
		((uint32_t *)b.image)[o] = v;
	}
	if(b.image_f)
		((float4 *)b.image_f)[o] = make_float4(r, g, bl, 1.0f);
	if(b.frag_counts)
		b.frag_counts[o] = count;
}

// ------------------------------------------------------------------ sorts

// Bitonic network on 64 * E keys held by one wave (key e * 64 + lane of the block in v[e]).
// Level K merges runs of K / 2 keys in steps J = K / 2 .. 1, each pairing indices i and i ^ J,
// ascending where (i & K) == 0. A step within a wave is an exchange and one median: of the pair
// and a bound, 0 keeps the smaller key and ~0 the larger, so the lane mask of the upper partner
// and the direction fold into the bound (a constant of the step). The block sorts were bound by
// the LDS pipe when the exchanges went through ds_bpermute_b32 (high_finalize, before -> after:
// 1 M soup triangles at 1080p 124 -> 89 us, 5.2 M mesh triangles at 1440p 272 -> 193 us).
__device__ __forceinline__ uint32_t med3_u32(uint32_t a, uint32_t b, uint32_t c) {
	return max(min(a, b), min(max(a, b), c));
}
// Lanes l of a wave with (l & J) != 0.
constexpr uint64_t upper_lanes(int J) {
	uint64_t m = 0;
	for(int l = 0; l < 64; l++)
		m |= (l & J) ? 1ull << l : 0ull;
	return m;
}

// Steps J, J / 2 .. 1 of level K; K = 0: ascending everywhere (the last level of a sort).
template <int E, int K, int J> __device__ __forceinline__ void bitonic_steps(uint32_t (&v)[E]) {
	if constexpr(J >= 64) {
#pragma unroll
		for(int e = 0; e < E; e++) {
			if((e & (J / 64)) == 0) {
				const int pe = e | (J / 64);
				const uint32_t mn = min(v[e], v[pe]), mx = max(v[e], v[pe]);
				const bool desc = ((e * 64) & K) != 0;
				v[e] = desc ? mx : mn;
				v[pe] = desc ? mn : mx;
			}
		}
	} else {
#pragma unroll
		for(int e = 0; e < E; e++) {
			const uint64_t desc = K == 0 ? 0ull : K < 64 ? upper_lanes(K) : ((e * 64) & K) ? ~0ull : 0ull;
			const uint32_t bound = __builtin_amdgcn_inverse_ballot_w64(upper_lanes(J) ^ desc) ? ~0u : 0u;
			if constexpr(J >= 16) {
				const LanePair p = lane_pair<J>(v[e]);
				v[e] = med3_u32(p.x, p.y, bound);
			} else {
				v[e] = med3_u32(v[e], lane_xor<J>(v[e]), bound);
			}
		}
	}
	if constexpr(J > 1)
		bitonic_steps<E, K, J / 2>(v);
}

// Steps J .. 1 of a level beyond the block (every pair in the block has the same direction):
// ascending for flip = 0, descending for ~0 (the complements ascend).
template <int E, int J>
__device__ __forceinline__ void bitonic_merge(uint32_t (&v)[E], uint32_t flip) {
#pragma unroll
	for(int e = 0; e < E; e++)
		v[e] ^= flip;
	bitonic_steps<E, 0, J>(v);
#pragma unroll
	for(int e = 0; e < E; e++)
		v[e] ^= flip;
}

// Levels K .. 32 * E of a block (the direction depends on the index within it).
template <int E, int K> __device__ __forceinline__ void bitonic_levels(uint32_t (&v)[E]) {
	if constexpr(K < 64 * E) {
		bitonic_steps<E, K, K / 2>(v);
		bitonic_levels<E, 2 * K>(v);
	}
}

// Sorts the block: ascending for flip = 0, descending for flip = ~0 (as the levels of a longer
// sequence expect of every second block).
template <int E> __device__ __forceinline__ void bitonic_regs(uint32_t (&v)[E], uint32_t flip = 0u) {
	bitonic_levels<E, 2>(v);
	bitonic_merge<E, 32 * E>(v, flip);
}

// Sorts the wave's 64 keys, one per lane, ascending.
template <int K, int J> __device__ __forceinline__ void bitonic64_steps(uint64_t &v) {
	const uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
	uint32_t olo, ohi;
	if constexpr(J >= 16) {
		const LanePair a = lane_pair<J>(lo), b = lane_pair<J>(hi);
		const bool upper = (lane_id() & J) != 0;
		olo = upper ? a.x : a.y, ohi = upper ? b.x : b.y;
	} else {
		olo = lane_xor<J>(lo), ohi = lane_xor<J>(hi);
	}
	const uint64_t o = ((uint64_t)ohi << 32) | olo;
	const bool keep_min = ((lane_id() & K) == 0) == ((lane_id() & J) == 0);
	v = (o < v) == keep_min ? o : v;
	if constexpr(J > 1)
		bitonic64_steps<K, J / 2>(v);
}
template <int K = 2> __device__ __forceinline__ void bitonic64_wave(uint64_t &v) {
	bitonic64_steps<K, K / 2>(v);
	if constexpr(K < 64)
		bitonic64_wave<K * 2>(v);
}

// Ascending bitonic sort of P (power of two) keys in LDS by one wave.
__device__ void bitonic_lds_wave(uint64_t *key, uint32_t P) {
	const int lane = lane_id();
	for(uint32_t k = 2; k <= P; k <<= 1) {
		for(uint32_t j = k >> 1; j > 0; j >>= 1) {
			for(uint32_t i = lane; i < P / 2; i += 64) {
				uint32_t lo = ((i & ~(j - 1)) << 1) | (i & (j - 1));
				uint32_t hi = lo | j;
				bool asc = (lo & k) == 0;
				uint64_t a = key[lo], bb = key[hi];
				if((a > bb) == asc) {
					key[lo] = bb;
					key[hi] = a;
				}
			}
			wave_sync_lds();
		}
	}
}

__device__ __forceinline__ uint32_t next_pow2(uint32_t x) {
	return x <= 1 ? 1u : 1u << (32 - __clz(x - 1));
}

// Sorts a pixel's n <= kFallbackCap keys in LDS (its own wave's): up to 64 of them in registers (21
// exchanges through the VALU instead of LDS round trips).
__device__ void sort_pixel_keys(uint64_t *key, uint32_t n) {
	const int lane = lane_id();
	if(n <= 64) {
		wave_sync_lds();
		uint64_t k = (uint32_t)lane < n ? key[lane] : ~0ull;
		bitonic64_wave(k);
		key[lane] = k;
		wave_sync_lds();
		return;
	}
	const uint32_t P = next_pow2(n);
	for(uint32_t i = n + lane; i < P; i += 64)
		key[i] = ~0ull;
	wave_sync_lds();
	bitonic_lds_wave(key, P);
}

// Same on global memory (deep pixels); agent-scope fences make each stage visible.
__device__ void bitonic_global_wave(uint64_t *key, uint32_t P) {
	const int lane = lane_id();
	for(uint32_t k = 2; k <= P; k <<= 1) {
		for(uint32_t j = k >> 1; j > 0; j >>= 1) {
			for(uint32_t i = lane; i < P / 2; i += 64) {
				uint32_t lo = ((i & ~(j - 1)) << 1) | (i & (j - 1));
				uint32_t hi = lo | j;
				bool asc = (lo & k) == 0;
				uint64_t a = __hip_atomic_load(&key[lo], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				uint64_t bb = __hip_atomic_load(&key[hi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				if((a > bb) == asc) {
					__hip_atomic_store(&key[lo], bb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					__hip_atomic_store(&key[hi], a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				}
			}
			__threadfence();
			__builtin_amdgcn_wave_barrier();
		}
	}
}

// ------------------------------------------------------------------ block entries and keys

// A block list entry {triangle, depth key, pixel mask}: everything the sorts and walks need
// to know of a (block, triangle) pair, in list order, so that they read whole lists with
// coalesced loads and gather nothing.
__device__ __forceinline__ uint64_t entry_mask(uint4 e) {
	return ((uint64_t)e.w << 32) | e.z;
}

// Block-level depth key ~ord(inverse depth) of a triangle (depth plane d) inside a block at
// the centroid of its covered pixels, from its pixel mask m (bit 8 r + c: row r, column c of
// the block whose corner pixel is (px0, py0)); ties and centroid error are resolved exactly
// per pixel later. The column and row sums are integers, taken bit by bit with masked
// popcounts: the sum of the columns is sum_k 2^k popcount(m & pixels whose column has bit
// k), likewise for the rows. s_inv[n] = 1 / n.
__device__ __forceinline__ uint32_t mask_depth_key(uint4 d, uint64_t m, int px0, int py0,
												   const float *s_inv) {
	auto pc = [](uint64_t x) { return (int)__popcll(x); };
	const int n = pc(m);
	const int sc = pc(m & 0xAAAAAAAAAAAAAAAAull) + 2 * pc(m & 0xCCCCCCCCCCCCCCCCull) +
				   4 * pc(m & 0xF0F0F0F0F0F0F0F0ull);
	const int sr = pc(m & 0xFF00FF00FF00FF00ull) + 2 * pc(m & 0xFFFF0000FFFF0000ull) +
				   4 * pc(m & 0xFFFFFFFF00000000ull);
	const float inv_n = s_inv[n];
	const float cx = (float)px0 + (float)sc * inv_n;
	const float cy = (float)py0 + (float)sr * inv_n;
	return inv_ord_f32(bits2f(d.x) * cx + (bits2f(d.y) * cy + bits2f(d.z)));
}

// Depth rank of a block entry from its depth key ~ord(inverse depth) (ascending = nearest
// first): the key minus the block's smallest, shifted right just enough that the block's key
// range fits BITS bits. Monotone in the key, and float keys keep relative precision (about
// BITS - log2(binades spanned) mantissa bits), so ties are rare and are resolved per pixel.
struct DepthGrid {
	uint32_t lo;
	int shift;
	__device__ __forceinline__ DepthGrid(uint32_t lo_, uint32_t hi_, int bits) : lo(lo_) {
		const uint32_t span = hi_ - lo_;
		const int need = span ? 32 - __clz(span) : 0;
		shift = need > bits ? need - bits : 0;
	}
	__device__ __forceinline__ uint32_t rank(uint32_t key) const { return (key - lo) >> shift; }
};

// Depth order of a block list of m <= 256 entries, sorted by one wave in registers: sorted
// entry 64 k + lane is list position pos[k]. Keys are (24-bit depth rank << 8 | position).
// Each entry's pixel mask and triangle id are left in s_msk / s_tri (LDS, kRegSortCap entries
// each) at its list position, for the caller to read in sorted order after a wave_sync_lds.
__device__ __forceinline__ void sort_block_positions(const uint4 *list, uint32_t m,
													 uint32_t (&pos)[4], uint64_t *s_msk,
													 uint32_t *s_tri) {
	static_assert(kRegSortCap <= 256, "list positions fit 8 bits of the key");
	const int lane = lane_id();
	uint32_t dk[4];
	uint32_t lo = ~0u, hi = 0u;
	uint4 e[4];
#pragma unroll
	for(int k = 0; k < 4; k++)
		e[k] = k * 64 + lane < (int)m ? list[k * 64 + lane] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
	for(int k = 0; k < 4; k++) {
		const uint32_t j = k * 64 + lane;
		dk[k] = e[k].y;
		if(j < m) {
			s_msk[j] = entry_mask(e[k]);
			s_tri[j] = e[k].x;
			lo = min(lo, dk[k]);
			hi = max(hi, dk[k]);
		}
	}
	const DepthGrid grid(wave_min_u32(lo), wave_max_u32(hi), 24);
	// a real key never equals the padding: position 255 exists only when nothing is padded
	auto key = [&](int k) -> uint32_t {
		const uint32_t j = k * 64 + lane;
		return j < m ? (grid.rank(dk[k]) << 8) | j : ~0u;
	};
	// One key array for the three sort widths (copied in and out of the narrower sorts), so
	// that it stays in registers: positions of empty rows are never read.
	uint32_t w[4] = {key(0), key(1), key(2), key(3)};
	if(m <= 64) {
		uint32_t w1[1] = {w[0]};
		bitonic_regs<1>(w1);
		w[0] = w1[0];
	} else if(m <= 128) {
		uint32_t w2[2] = {w[0], w[1]};
		bitonic_regs<2>(w2);
		w[0] = w2[0], w[1] = w2[1];
	} else {
		bitonic_regs<4>(w);
	}
#pragma unroll
	for(int k = 0; k < 4; k++)
		pos[k] = w[k] & 0xffu;
}

__device__ __forceinline__ uint32_t bin_tri_at(const FrameBufs &b, uint32_t i, uint32_t qc,
											   uint32_t qo, uint32_t to) {
	if(i < 2 * qc) {
		uint32_t e = b.bin_quads[qo + (i >> 1)];
		uint32_t s = i & 1u;
		if((e >> (30 + s)) & 1u)
			return 0xffffffffu;
		return 2 * (e & 0x0fffffffu) + s;
	}
	return b.bin_tris[to + (i - 2 * qc)];
}

// Keeps loads that a return could come before where they are written, in flight together: a block's
// chain of early exits otherwise takes a memory latency for each.
__device__ __forceinline__ void loaded_here() {}
template <class T, class... R> __device__ __forceinline__ void loaded_here(T v, R... rest) {
	asm volatile("" ::"v"(v));
	loaded_here(rest...);
}

struct BinInfo {
	uint32_t qc, tc, qo, to, nlevel;
	int bin_x, bin_y;
};

__device__ __forceinline__ BinInfo load_bin(const FrameConst &c, const FrameBufs &b, int bin) {
	const int NB = c.bin_count;
	const uint32_t *counts = b.info + LUCID_INFO_U32_SIZE;
	BinInfo bi;
	bi.qc = counts[LUCID_COUNTS_QUAD_COUNTS * NB + bin];
	bi.tc = counts[LUCID_COUNTS_TRI_COUNTS * NB + bin];
	bi.qo = counts[LUCID_COUNTS_QUAD_OFFSETS * NB + bin];
	bi.to = counts[LUCID_COUNTS_TRI_OFFSETS * NB + bin];
	bi.nlevel = bi.tc + 2 * bi.qc;
	bi.bin_x = (bin % c.bin_count_x) * kBinSize;
	bi.bin_y = (bin / c.bin_count_x) * kBinSize;
	return bi;
}

// Exact-fallback queue: one uint4 item per pixel, {block slot, px, py, whole}. Called by
// a whole wave; lanes with `mine` set queue their pixel (px, py).
__device__ __forceinline__ void enqueue_pixels(const FrameBufs &b, uint32_t slot, bool mine, int px,
											   int py, bool whole) {
	const int lane = lane_id();
	const uint64_t sel = ballot(mine);
	if(!sel)
		return;
	uint32_t base = 0;
	if(lane == 0)
		base = atomicAdd(&b.ctrl[kCtrlFallbackCount], (uint32_t)__popcll(sel));
	base = wave_read(base, 0);
	if(mine) {
		const uint32_t i = base + (uint32_t)__popcll(sel & ((1ull << lane) - 1ull));
		if(i < b.fallback_cap)
			b.fallback_queue[i] = make_uint4(slot, (uint32_t)px, (uint32_t)py, whole ? 1u : 0u);
		else
			atomicOr(&b.ctrl[kCtrlOverflow], kOvfFallback);
	}
}

// ------------------------------------------------------------------ row generation
//
// Both row generators hand their live triangles to waves 64 at a time (sorted by height, so
// that the lanes of a wave scan about as many rows); rowgen_wave scans them and writes their
// block entries. A lane scans its triangle's rows in one loop, four rows (a group) per step,
// and leaves the row spans in LDS. The wave then lists its (block, triangle) pairs block by
// block, reserves each block's list positions with one atomic instruction, and makes the
// entries with one pair per lane: the pixel mask from the spans, the depth key from the mask
// and the depth plane. All lanes are busy there (a triangle covers a few of a bin's 16 blocks),
// and neighbouring lanes write neighbouring entries of a list.
//
// Both are bound by the latency of their gathers (VALU about half busy), so the staging is
// kept small: 25 KB per work-group of four waves. Masks instead of spans in LDS (46 KB) saved a
// third of the VALU work and was slower (5.2 M mesh triangles: 348 us against 270), as was
// loading the next triangles' records ahead (304). Writing whole entries here instead of row
// records and index lists takes the two dependent gathers per entry out of the sorts and walks
// (before -> after): mesh rowgen_high 350 -> 270, high_finalize 406 -> 274 us; 1 M soup
// triangles 131 -> 116 and 139 -> 113 us, rowgen_low 23 -> 30 us with the register-sorted
// blocks' walk 60 -> 54 us.

// Staging of one wave.
struct RowgenWave {
	uint2 rows[64][8];      // spans of a lane's row groups, group g at g ^ (lane / 2 % 8)
	uint16_t pair[64 * 16]; // lane | block << 6
	uint32_t base[16];      // per block: list entry of pair p of the block, minus p
};
// A work-group's LDS: its sorted triangles (each thread takes its up to kRowgenRound of them
// into registers first), then the waves' staging.
constexpr int kRowgenRound = 1024; // list entries per sorting round
template <int THREADS> union RowgenLds {
	uint32_t sorted[kRowgenRound];
	RowgenWave wave[THREADS / 64];
};
struct RowgenCounts {
	uint32_t cnt[8], off[8], nlive; // the counting sort
	uint32_t blk_n[16];             // list lengths of a low bin
};
// The LDS that low and high bins share (in the launch that takes both, too). Three variables, not
// one struct: accesses with indices known only at run time are then known not to overlap, and the
// compiler keeps them in flight together (one struct: rowgen_high 5 - 10 % slower).
template <int THREADS> __device__ __forceinline__ RowgenLds<THREADS> &rowgen_lds() {
	__shared__ RowgenLds<THREADS> s;
	return s;
}
__device__ __forceinline__ RowgenCounts &rowgen_counts() {
	__shared__ RowgenCounts s;
	return s;
}
__device__ __forceinline__ float *rowgen_inverses() { // [n] = 1 / n, n <= 64
	__shared__ float s[65];
	return s;
}
__device__ __forceinline__ void fill_inverses() {
	if(threadIdx.x <= 64)
		rowgen_inverses()[threadIdx.x] = 1.0f / (float)(threadIdx.x > 0 ? threadIdx.x : 1);
}
// Work-group size: a single frame's low bins take twice the waves, as a low bin's triangles are
// few (each wave then scans one or two chunks); high bins, and a batch, which has bins enough to
// fill the chip, keep to the smaller groups. Low bins: 1280 x 720 lit mesh frame 26.2 -> 23.6 us
// with 512 threads, the 32-frame batch 240 us with 256 and 271 us with 512.
constexpr int kRowgenLowThreads = 512;

// What a lane scans: a triangle (~0: none), its scan parameters and depth plane.
struct ScanTri {
	uint32_t t;
	uint4 s0, s1, depth;
};
__device__ __forceinline__ ScanTri load_scan_tri(const FrameBufs &b, uint32_t t) {
	ScanTri tr;
	tr.t = t;
	tr.s0 = tr.s1 = tr.depth = make_uint4(0u, 0u, 0u, 0u);
	if(t != 0xffffffffu) {
		const size_t i = tri_rec(b, t);
		tr.s0 = b.tri_scan[2 * i], tr.s1 = b.tri_scan[2 * i + 1], tr.depth = b.tri_depth[i];
	}
	return tr;
}

// Scans the lanes' triangles from row group g0 to g1 of the bin at
// (bin_x, bin_y) and appends their entries to the bin's 16 block lists. `first` is the list
// offset of block `lane` (lanes 0-15), `reserve(n)` takes n positions of the list of block
// `lane` and returns the first; positions from `cap` on are not written (lists of a low bin
// that will be promoted).
template <class Reserve>
__device__ __forceinline__ void rowgen_wave(const FrameBufs &b, RowgenWave &w, const float *s_inv,
											int bin_x, int bin_y, const ScanTri &tr, int g0, int g1,
											uint32_t first, uint32_t cap, Reserve &&reserve) {
	const int lane = lane_id();
	uint32_t cols = 0; // blocks the triangle covers, one bit each
	const uint4 d = tr.depth;
	const uint32_t t = tr.t;
	if(t != 0xffffffffu) {
		RowScan rs;
		row_scan_init(rs, tr.s0, tr.s1, (float)bin_x, (float)(bin_y + g0 * 4));
		uint2 *rows = w.rows[lane];
		const int sw = (lane >> 1) & 7;
		const uint2 empty = make_uint2(kBinMask | (kBinMask << 16), kBinMask | (kBinMask << 16));
		if(g0 & 1) // the other half of the first and the last 8-row band
			rows[(g0 - 1) ^ sw] = empty;
		if(!(g1 & 1))
			rows[(g1 + 1) ^ sw] = empty;
		for(int g = g0; g <= g1; g++) {
			uint32_t v[4], any = 0;
#pragma unroll
			for(int r = 0; r < 4; r++) {
				v[r] = row_scan_step(rs);
				any |= span_bits(v[r]);
			}
			rows[g ^ sw] = make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16));
			cols |= nonzero_bytes(any) << (4 * (g >> 1));
		}
	}
	const uint64_t below = (1ull << lane) - 1ull;
	const uint32_t first0 = __builtin_amdgcn_readfirstlane(first);
	uint32_t run = 0, off = 0, num = 0;
#pragma unroll
	for(int k = 0; k < 16; k++) {
		const bool mine = (cols >> k) & 1u;
		const uint64_t sel = ballot(mine);
		if(mine)
			w.pair[run + (uint32_t)__popcll(sel & below)] = (uint16_t)(lane | (k << 6));
		const uint32_t n = (uint32_t)__popcll(sel);
		if(lane == k)
			off = run, num = n;
		run += n;
	}
	if(lane < 16)
		w.base[lane] = first + (num ? reserve(num) : 0u) - off;
	wave_sync_lds();
	for(uint32_t p0 = 0; p0 < run; p0 += 64) {
		// (the whole wave stays in the loop: the planes come from the lanes' registers)
		const uint32_t p = p0 + lane, pr = p < run ? w.pair[p] : 0u;
		const uint32_t l = pr & 63u, k = pr >> 6, by = k >> 2, bx = k & 3u;
		const uint32_t idx = w.base[k] + p;
		const uint32_t sw = (l >> 1) & 7u;
		const uint32_t lo = group_mask(w.rows[l][(2 * by) ^ sw], bx);
		const uint32_t hi = group_mask(w.rows[l][(2 * by + 1) ^ sw], bx);
		const uint4 dl = make_uint4(__shfl(d.x, (int)l, 64), __shfl(d.y, (int)l, 64),
									__shfl(d.z, (int)l, 64), 0u);
		const uint32_t tl = __shfl(t, (int)l, 64);
		const uint64_t m = ((uint64_t)hi << 32) | lo;
		const uint32_t key =
			mask_depth_key(dl, m, bin_x + (int)bx * 8, bin_y + (int)by * 8, s_inv);
		if(p < run && (cap == ~0u || idx - (first0 + k * cap) < cap))
			b.blk_lists[idx] = make_uint4(tl, key, lo, hi);
	}
	wave_sync_lds(); // the staging is used again
}

// ------------------------------------------------------------------ high bins

// Block lists of a high bin with the 4-row rule (raster_high.glsl:54-90): a triangle's scan
// starts at the first row of its 4-row group (the start row fixes the scanline arithmetic).
// Work-group `split` of `splits` that share the bin; block k's list starts at lst + k * nlevel.
// A wave's row loop runs as long as its tallest triangle, so each work-group first sorts its
// triangles by height (a counting sort over the 8 heights in 4-row groups, up to kRowgenRound
// list positions at a time).
template <int THREADS>
__device__ __forceinline__ void rowgen_high_bin(const FrameBufs &b, int bin,
												const BinInfo &bi, uint32_t lst, uint32_t split,
												uint32_t splits) {
	RowgenLds<THREADS> &s = rowgen_lds<THREADS>();
	RowgenCounts &sh = rowgen_counts();
	const int lane = lane_id(), wave = threadIdx.x >> 6;
	const uint32_t first = lst + (uint32_t)(lane & 15) * bi.nlevel;
	uint32_t *blk_n = b.blk_count + (size_t)bin * 16;
	const uint32_t stride = THREADS * splits;
	constexpr int kHeights = kBinSize / 4, kChunks = kRowgenRound / THREADS;
	// first row group and height in row groups of triangle t in this bin
	auto groups = [&](uint32_t yr, int &g0, int &g1) {
		g0 = min(max((int)(yr & 0xffffu) - bi.bin_y, 0), kBinMask) >> 2;
		g1 = min(max((int)(yr >> 16) - bi.bin_y, 0), kBinMask) >> 2;
	};
	// the work-group's list positions: chunks split, split + splits, ... of THREADS entries;
	// culled triangles (every second one of a soup quad) are dropped
	const uint32_t round_len = stride * kChunks;
	for(uint32_t base = split * THREADS; base < bi.nlevel; base += round_len) {
		if(threadIdx.x < kHeights)
			sh.cnt[threadIdx.x] = 0;
		__syncthreads();
		uint32_t tk[kChunks];
		int hk[kChunks];
#pragma unroll
		for(int k = 0; k < kChunks; k++) {
			const uint32_t i = base + k * stride + threadIdx.x;
			const uint32_t t = i < bi.nlevel ? bin_tri_at(b, i, bi.qc, bi.qo, bi.to) : 0xffffffffu;
			int h = -1;
			if(t != 0xffffffffu) {
				int g0, g1;
				groups(b.tri_scan[2 * (size_t)tri_rec(b, t)].w, g0, g1);
				h = g1 > g0 ? g1 - g0 : 0;
				atomicAdd(&sh.cnt[h], 1u);
			}
			tk[k] = t, hk[k] = h;
		}
		__syncthreads();
		if(threadIdx.x == 0) {
			uint32_t run = 0;
			for(int h = 0; h < kHeights; h++)
				sh.off[h] = run, run += sh.cnt[h];
			sh.nlive = run;
		}
		__syncthreads();
#pragma unroll
		for(int k = 0; k < kChunks; k++)
			if(hk[k] >= 0)
				s.sorted[atomicAdd(&sh.off[hk[k]], 1u)] = tk[k];
		__syncthreads();
		const uint32_t n = sh.nlive;
#pragma unroll
		for(int k = 0; k < kChunks; k++)
			tk[k] = k * THREADS + threadIdx.x < n ? s.sorted[k * THREADS + threadIdx.x] : 0xffffffffu;
		__syncthreads(); // the staging takes the sorted list's place
		for(int k = 0; k * THREADS + wave * 64 < (int)n; k++) {
			const ScanTri tr = load_scan_tri(b, k == 0 ? tk[0] : k == 1 ? tk[1] : k == 2 ? tk[2 % kChunks] : tk[3 % kChunks]);
			int g0 = 0, g1 = -1;
			if(tr.t != 0xffffffffu)
				groups(tr.s0.w, g0, g1);
			rowgen_wave(b, s.wave[wave], rowgen_inverses(), bi.bin_x, bi.bin_y, tr, g0, g1, first, ~0u,
						[&](uint32_t num) { return atomicAdd(&blk_n[lane], num); });
		}
		if(base + round_len < bi.nlevel)
			__syncthreads(); // the next round reuses the sorted list
	}
}

// ------------------------------------------------------------------ low bins

// Block lists of a low bin, 256 positions each, with the 8-row rule (raster_low.glsl:39-79): the
// scan starts at the first row of a band. A bin with a longer list is promoted: it joins the
// high list, takes list space of its own and is generated again as a high bin.
template <int THREADS>
__device__ __forceinline__ void rowgen_low_bin(const FrameConst &c, const FrameBufs &b, int bin) {
	RowgenLds<THREADS> &s = rowgen_lds<THREADS>();
	RowgenCounts &sh = rowgen_counts();
	const BinInfo bi = load_bin(c, b, bin);
	uint32_t *flags = b.blk_flags + (size_t)bin * 16;
	if(bi.nlevel == 0) {
		if(threadIdx.x < 16)
			flags[threadIdx.x] = LUCID_BIN_LEVEL_EMPTY;
		return;
	}
	if(bi.nlevel >= (uint32_t)kLowLevelLimit)
		return; // a high bin

	constexpr int kChunks = kRowgenRound / THREADS; // list positions per thread
	// The bin's live triangles (its list has fewer than kLowLevelLimit entries: one position
	// per thread and chunk) are counting-sorted by their number of 8-row bands, so that the
	// waves' row loops run about as long as each of their triangles needs.
	static_assert(kLowLevelLimit <= kRowgenRound, "a low bin's list in one round");
	fill_inverses();
	if(threadIdx.x < 16)
		sh.blk_n[threadIdx.x] = 0;
	if(threadIdx.x < 4)
		sh.cnt[threadIdx.x] = 0;
	__syncthreads();
	uint32_t tk[kChunks];
	int hk[kChunks];
	// first and last 8-row band of a triangle in this bin, from its row range
	auto bands = [&](uint32_t yr, int &lo_by, int &hi_by) {
		lo_by = min(max((int)(yr & 0xffffu) - bi.bin_y, 0), kBinMask) >> 3;
		hi_by = min(max((int)(yr >> 16) - bi.bin_y, 0), kBinMask) >> 3;
	};
#pragma unroll
	for(int k = 0; k < kChunks; k++) {
		const uint32_t i = k * THREADS + threadIdx.x;
		const uint32_t t = i < bi.nlevel ? bin_tri_at(b, i, bi.qc, bi.qo, bi.to) : 0xffffffffu;
		int h = -1;
		if(t != 0xffffffffu) {
			int lo_by, hi_by;
			bands(b.tri_scan[2 * (size_t)tri_rec(b, t)].w, lo_by, hi_by);
			h = hi_by > lo_by ? hi_by - lo_by : 0;
			atomicAdd(&sh.cnt[h], 1u);
		}
		tk[k] = t, hk[k] = h;
	}
	__syncthreads();
	if(threadIdx.x == 0) {
		uint32_t run = 0;
		for(int h = 0; h < 4; h++)
			sh.off[h] = run, run += sh.cnt[h];
		sh.nlive = run;
	}
	__syncthreads();
#pragma unroll
	for(int k = 0; k < kChunks; k++)
		if(hk[k] >= 0)
			s.sorted[atomicAdd(&sh.off[hk[k]], 1u)] = tk[k];
	__syncthreads();
	const uint32_t nlive = sh.nlive;
	const int lane = lane_id(), wave = threadIdx.x >> 6;
#pragma unroll
	for(int k = 0; k < kChunks; k++)
		tk[k] = k * THREADS + threadIdx.x < nlive ? s.sorted[k * THREADS + threadIdx.x] : 0xffffffffu;
	__syncthreads(); // the staging takes the sorted list's place
	const uint32_t first = ((uint32_t)bin * 16 + (uint32_t)(lane & 15)) * kRegSortCap;
	for(int k = 0; k * THREADS + wave * 64 < (int)nlive; k++) {
		const ScanTri tr = load_scan_tri(b, k == 0 ? tk[0] : k == 1 ? tk[1] : k == 2 ? tk[2 % kChunks] : tk[3 % kChunks]);
		int lo_by = 0, hi_by = -1;
		if(tr.t != 0xffffffffu)
			bands(tr.s0.w, lo_by, hi_by);
		rowgen_wave(b, s.wave[wave], rowgen_inverses(), bi.bin_x, bi.bin_y, tr, lo_by * 2, hi_by * 2 + 1, first,
					(uint32_t)kRegSortCap, [&](uint32_t n) { return atomicAdd(&sh.blk_n[lane], n); });
	}
	__syncthreads();
	bool promote = false;
	for(int k = 0; k < 16; k++)
		promote |= sh.blk_n[k] > (uint32_t)kMaxBlockTris;
	if(!promote) {
		if(threadIdx.x < 16) {
			b.blk_slot[(size_t)bin * 16 + threadIdx.x] = make_uint2(first, sh.blk_n[threadIdx.x]);
			flags[threadIdx.x] = LUCID_BIN_LEVEL_LOW;
		}
		return;
	}
	__syncthreads(); // blk_n is read
	if(threadIdx.x == 0) {
		lucid_info *info = (lucid_info *)b.info;
		uint32_t id = atomicAdd((uint32_t *)&info->bin_level_counts[LUCID_BIN_LEVEL_HIGH], 1u);
		b.info[LUCID_INFO_U32_SIZE + LUCID_COUNTS_HIGH_BINS * c.bin_count + id] = (uint32_t)bin;
		const uint64_t list0 = (uint64_t)c.bin_count * 16 * kRegSortCap;
		const uint32_t cursor = atomicAdd(&b.ctrl[kCtrlListCursor], bi.nlevel);
		const bool ok = lists_fit(list0, cursor, bi.nlevel, b.blk_lists_cap);
		if(!ok)
			atomicOr(&b.ctrl[kCtrlOverflow], kOvfLists);
		sh.blk_n[0] = (uint32_t)list_entry(list0, cursor), sh.blk_n[1] = ok ? 1u : 0u;
	}
	__syncthreads();
	const uint32_t lst = sh.blk_n[0];
	const bool ok = sh.blk_n[1] != 0u;
	if(threadIdx.x < 16) {
		b.blk_slot[(size_t)bin * 16 + threadIdx.x] = make_uint2(lst + threadIdx.x * bi.nlevel, 0u);
		flags[threadIdx.x] = ok ? 0u : kSlotPromoted; // (no space: the frame reports an overflow)
	}
	if(ok)
		rowgen_high_bin<THREADS>(b, bin, bi, lst, 0u, 1u);
}

// Work-group id of the kRowgenSplitThreads / THREADS that share each high bin.
template <int THREADS>
__device__ __forceinline__ void rowgen_high_body(const FrameConst &c, const FrameBufs &b, uint32_t id) {
	constexpr uint32_t kSplits = kRowgenSplitThreads / THREADS;
	const uint32_t slot = id / kSplits, split = id % kSplits;
	if((b.ctrl[kCtrlOverflow] & kOvfBinLists) || slot >= b.ctrl[kCtrlFixedHigh])
		return;
	const int bin = (int)b.info[LUCID_INFO_U32_SIZE + LUCID_COUNTS_HIGH_BINS * c.bin_count + slot];
	const BinInfo bi = load_bin(c, b, bin);
	const uint32_t lst = b.blk_slot[(size_t)bin * 16].x;
	// Not kOvfLists: a low bin promoted in the same launch may set that while the waves of this
	// work-group read it, and waves that disagree would miss each other at the barriers below.
	const bool fits = b.ctrl[kCtrlFixedFit] != 0u;
	if(split == 0 && threadIdx.x < 16) {
		if(threadIdx.x > 0)
			b.blk_slot[(size_t)bin * 16 + threadIdx.x] = make_uint2(lst + threadIdx.x * bi.nlevel, 0u);
		b.blk_flags[(size_t)bin * 16 + threadIdx.x] = fits ? 0u : kSlotPromoted;
	}
	if(!fits)
		return;
	fill_inverses();
	rowgen_high_bin<THREADS>(b, bin, bi, lst, split, kSplits);
}
template <int THREADS>
__device__ __forceinline__ void rowgen_low_body(const FrameConst &c, const FrameBufs &b, uint32_t id) {
	const uint32_t overflow = b.ctrl[kCtrlOverflow];
	if(!(overflow & kOvfBinLists))
		rowgen_low_bin<THREADS>(c, b, (int)id);
}

// Low (and empty) bins and high bins apart, and in one launch: the high bins' work-groups first
// (the longest), then the low ones', which fill the chip as the high ones run out.
__global__ __launch_bounds__(kRowgenLowThreads) void rowgen_low_kernel(FrameConst c, FrameBufs b) {
	rowgen_low_body<kRowgenLowThreads>(c, b, blockIdx.x);
}
__global__ __launch_bounds__(kRowgenThreads) void rowgen_high_kernel(FrameConst c, FrameBufs b) {
	rowgen_high_body<kRowgenThreads>(c, b, blockIdx.x);
}
__global__ __launch_bounds__(kRowgenLowThreads) void rowgen_fused_kernel(FrameConst c, FrameBufs b) {
	const uint32_t high = (uint32_t)c.bin_count * (kRowgenSplitThreads / kRowgenLowThreads);
	if(blockIdx.x < high)
		rowgen_high_body<kRowgenLowThreads>(c, b, blockIdx.x);
	else
		rowgen_low_body<kRowgenLowThreads>(c, b, blockIdx.x - high);
}
__global__ __launch_bounds__(kRowgenThreads) void rowgen_low_kernel_batch(const FrameDesc *__restrict__ frames,
		const uint32_t *__restrict__ pre, uint32_t num_frames) {
	const StageBatch sb{frames, pre, num_frames};
	const uint32_t f = batch_frame(sb, blockIdx.x);
	const FrameDesc &d = sb.frames[f];
	rowgen_low_body<kRowgenThreads>(d.c, d.b, blockIdx.x - sb.pre[f]);
}
__global__ __launch_bounds__(kRowgenThreads) void rowgen_high_kernel_batch(const FrameDesc *__restrict__ frames,
		const uint32_t *__restrict__ pre, uint32_t num_frames) {
	const StageBatch sb{frames, pre, num_frames};
	const uint32_t f = batch_frame(sb, blockIdx.x);
	const FrameDesc &d = sb.frames[f];
	rowgen_high_body<kRowgenThreads>(d.c, d.b, blockIdx.x - sb.pre[f]);
}

// Entries (triangles of one block in depth order) are handed to the rasteriser in slices
// of up to kSliceEntries: entry lane + 64 k of the slice sits in register k of that lane.
// (The block rasterisers take the slice width W = 1 or 2 words as a template parameter,
// chosen per renderer by its tuning; the backward kernels use kSliceWords.)
constexpr int kSliceWords = 1;
constexpr int kSliceEntries = 64 * kSliceWords;
constexpr uint32_t kTieRun = 32; // longest run of equal block ranks put in exact order
constexpr int kBigWaves = 4; // waves of block_raster_kernel / the backward block kernels

// Pre-sorted block layout in the sorted pool (offsets in words from an even base):
//   [0] number of waves W, [1 .. W + 1] first entry of each wave's range (then m),
//   [kSortedHeader .. + m) triangle ids, [sorted_mask_offset(m) ..) 64-bit pixel masks.
constexpr uint32_t kSortedHeader = 10;
__device__ __forceinline__ uint32_t sorted_mask_offset(uint32_t m) {
	return (kSortedHeader + m + 1u) & ~1u;
}

// Finalises every block of the high bins: copies the list lengths into the slot table and
// pre-sorts long lists. A long list is sorted once by centroid depth (LDS bitonic by the
// whole work-group) and split into contiguous depth ranges of about equal sample counts, so that
// several waves can rasterise a dense block.
// A work-group is a chain of memory and LDS latencies (VALU busy 0.4), so the loads that decide its
// early exits are made together, the pool is asked for while the entries load, and a list of up to
// 256 keys is sorted by all four waves: 32-frame batch 506 -> 471 us, 5.2 M mesh triangles 192 ->
// 148, 1 M soup triangles 89 -> 80.
// Two passes share the body: CAP = kMidSortCap does the slot bookkeeping of every block,
// sorts the lists of up to kMidSortCap entries (8 KB of keys in LDS, so twice as many
// work-groups per CU as with the full capacity) and queues the longer ones in big_queue;
// CAP = kBigSortCap then takes the queued blocks (a small persistent grid: the queue is
// usually empty). Both sort with the same keys, so the output does not depend on the pass.
constexpr uint32_t kMidSortCap = 2048;

template <uint32_t CAP>
__device__ __forceinline__ void high_finalize_kernel_body(const FrameConst &c, const FrameBufs &b, WgPos wg) {
	const lucid_info *info = (const lucid_info *)b.info;
	const uint32_t hslot = wg.id >> 4;
	const int blk = wg.id & 15, by = blk >> 2, bx = blk & 3;
	const uint32_t *counts = b.info + LUCID_INFO_U32_SIZE;
	const uint32_t overflow = b.ctrl[kCtrlOverflow], nhigh = (uint32_t)info->bin_level_counts[LUCID_BIN_LEVEL_HIGH];
	const int bin = (int)counts[LUCID_COUNTS_HIGH_BINS * c.bin_count + hslot]; // (hslot < bin_count)
	loaded_here(overflow, nhigh, bin);
	if((overflow & (kOvfBinLists | kOvfLists)) || hslot >= nhigh)
		return;
	const uint32_t slot = (uint32_t)bin * 16 + blk;
	const uint32_t flags = b.blk_flags[slot], m = b.blk_count[slot], list0 = b.blk_slot[slot].x;
	loaded_here(flags, m, list0);
	if(flags & kSlotPromoted)
		return; // allocation failed: the frame reports an overflow
	if(CAP == kMidSortCap && threadIdx.x == 0)
		b.blk_slot[slot].y = m;
	if(m <= c.presort_min) { // sorted in registers by the block rasteriser (<= kRegSortCap)
		if(CAP == kMidSortCap && threadIdx.x == 0)
			b.blk_flags[slot] = LUCID_BIN_LEVEL_HIGH;
		return;
	}
	static_assert(CAP == kMidSortCap || CAP == (uint32_t)kBigSortCap, "two sort passes");
	if(CAP == kMidSortCap && m > kMidSortCap) {
		if(threadIdx.x == 0) // the long-list pass takes it
			b.big_queue[atomicAdd(&b.ctrl[kCtrlBigSorts], 1u)] = wg.id;
		return;
	}
	if(m > (uint32_t)kBigSortCap) {
		if(threadIdx.x < 64) {
			const int px = (bin % c.bin_count_x) * kBinSize + bx * 8 + (threadIdx.x & 7);
			const int py = (bin / c.bin_count_x) * kBinSize + by * 8 + (threadIdx.x >> 3);
			if(threadIdx.x == 0) {
				b.blk_flags[slot] = LUCID_BIN_LEVEL_HIGH | kSlotWhole;
				atomicAdd(&((lucid_info *)b.info)->stats[3], 1u); // blocks too long to pre-sort
			}
			enqueue_pixels(b, slot, px < c.width && py < c.height, px, py, true);
		}
		return;
	}
	__shared__ uint32_t s_key[CAP];
	__shared__ uint32_t s_lo[kSortThreads / 64], s_hi[kSortThreads / 64];
	__shared__ uint32_t s_wsum[2][kSortThreads / 64];
	__shared__ uint32_t s_tdk[2][kSortThreads]; // full depth keys of tied entries, per round
	__shared__ uint32_t s_bound[kBigWaves + 1];
	__shared__ uint32_t s_base, s_parts, s_total;
	__shared__ uint8_t s_smp[CAP]; // samples (pixel-mask bits) of each entry, in list order
	static_assert(kBigSortCap <= (1 << 13), "list positions fit 13 bits of the key");
	static_assert(kSortThreads == 256, "four waves share the chunks");
	const uint4 *list = b.blk_lists + list0;
	const int wave_s = threadIdx.x >> 6, lane_s = lane_id();
	const uint32_t P = max(256u, next_pow2(m));
	const uint32_t nchunks = P / 256;
	// a key is (depth rank << pb | list position), with pb = log2(P) position bits, so
	// shorter lists keep more rank bits (24 at P = 256, 19 at 8192)
	const int pb = 31 - __clz(P);
	const uint32_t pmask = P - 1u;
	const bool unsorted = (c.opts & LUCID_OPT_UNSORTED) != 0; // the unsorted baseline
	// the block's pool space (allocated first) for the sorted entries: header, triangle ids,
	// masks
	// (the answer is awaited after pass 1's loads are under way)
	const uint32_t need = sorted_mask_offset(m) + 2 * m + 1; // + 1: even rounding of the base
	const uint32_t stripe = slot % kSortStripes;
	uint32_t off = 0;
	if(threadIdx.x == 0)
		off = atomicAdd(sort_cursor(b.ctrl, stripe), need);
	// Keys are (depth rank << pb | list position). Pass 1 reads the entries once: depth keys
	// (in s_key), sample counts and the block's key range.
	uint32_t lo = ~0u, hi = 0u;
	uint32_t mine = 0;
#pragma unroll 2
	for(uint32_t j = threadIdx.x; j < m; j += kSortThreads) {
		const uint4 en = list[j];
		const uint32_t smp = (uint32_t)__popc(en.z) + (uint32_t)__popc(en.w);
		s_smp[j] = (uint8_t)smp;
		mine += smp;
		// the unsorted baseline: list order (rank 0, the position alone)
		s_key[j] = unsorted ? j : en.y;
		lo = min(lo, en.y);
		hi = max(hi, en.y);
	}
	lo = wave_min_u32(lo);
	hi = wave_max_u32(hi);
	mine = wave_read(wave_inclusive_add(mine), 63);
	if(lane_s == 0)
		s_lo[wave_s] = lo, s_hi[wave_s] = hi, s_wsum[1][wave_s] = mine;
	if(threadIdx.x == 0) {
		const uint64_t region = (b.sorted_cap / kSortStripes) & ~1ull;
		uint32_t base = 0xffffffffu;
		if((uint64_t)off + need <= region) {
			base = (uint32_t)(stripe * region + off);
		} else {
			atomicOr(&b.ctrl[kCtrlOverflow], kOvfSorted);
			const uint64_t want = ((uint64_t)off + need + 2) * kSortStripes; // + even rounding
			atomicMax(&b.ctrl[kCtrlSortedCursor], (uint32_t)min(want, (uint64_t)0xffffffffu));
		}
		s_base = base == 0xffffffffu ? base : (base + 1u) & ~1u;
	}
	__syncthreads();
	if(s_base == 0xffffffffu) {
		if(threadIdx.x == 0)
			b.blk_flags[slot] = kSlotPromoted; // nothing rendered; the frame reports overflow
		return;
	}
	uint32_t *hdr = b.sorted_pool + s_base;
	uint32_t tot = 0;
#pragma unroll
	for(int w = 0; w < kSortThreads / 64; w++)
		lo = min(lo, s_lo[w]), hi = max(hi, s_hi[w]), tot += s_wsum[1][w];
	if(threadIdx.x == 0) {
		uint32_t nw = (tot + c.samples_per_wave - 1) / c.samples_per_wave;
		nw = nw < 1u ? 1u : nw > (uint32_t)kBigWaves ? (uint32_t)kBigWaves : nw;
		s_parts = nw;
		s_total = tot;
		for(int w = 0; w <= kBigWaves; w++)
			s_bound[w] = w == 0 ? 0u : m;
	}
	const DepthGrid grid(lo, hi, 32 - pb);
	// Bitonic sort. Up to 256 keys: one per thread, levels up to 64 within the waves, the two strides
	// across them through LDS (a buffer each, so one barrier each). Longer lists: levels up to 256
	// in registers (one 256-key chunk per wave at a time), then per level the strides >= 256 in LDS
	// and the rest in registers. A real key never equals the padding ~0u: position P - 1 exists
	// only when nothing is padded.
	if(nchunks == 1 && !unsorted) {
		static_assert(CAP >= 4 * kSortThreads, "the exchanges' buffers beside the keys");
		const uint32_t j = threadIdx.x;
		uint32_t v[1] = {j < m ? (grid.rank(s_key[j]) << pb) | j : ~0u};
		bitonic_regs<1>(v, (j & 64u) ? ~0u : 0u);
		auto exchange = [&](uint32_t *buf, uint32_t stride, uint32_t k) {
			buf[j] = v[0];
			__syncthreads();
			const uint32_t o = buf[j ^ stride];
			v[0] = ((j & k) == 0) == ((j & stride) == 0) ? min(v[0], o) : max(v[0], o);
		};
		exchange(s_key + kSortThreads, 64u, 128u);
		bitonic_merge<1, 32>(v, (j & 128u) ? ~0u : 0u);
		exchange(s_key + 2 * kSortThreads, 128u, 256u);
		exchange(s_key + 3 * kSortThreads, 64u, 256u);
		bitonic_merge<1, 32>(v, 0u);
		s_key[j] = v[0];
	}
	for(uint32_t ch = wave_s; ch < nchunks && nchunks > 1 && !unsorted; ch += kSortThreads / 64) {
		uint32_t v[4];
#pragma unroll
		for(int e = 0; e < 4; e++) {
			const uint32_t j = ch * 256 + e * 64 + lane_s;
			v[e] = j < m ? (grid.rank(s_key[j]) << pb) | j : ~0u;
		}
		bitonic_regs<4>(v, (ch & 1u) ? ~0u : 0u); // (alternating chunks for the next level)
#pragma unroll
		for(int e = 0; e < 4; e++)
			s_key[ch * 256 + e * 64 + lane_s] = v[e];
	}
	__syncthreads();
	for(uint32_t k = 512; k <= P && !unsorted; k <<= 1) {
		for(uint32_t j = k >> 1; j >= 256; j >>= 1) {
			for(uint32_t i = threadIdx.x; i < P / 2; i += kSortThreads) {
				uint32_t lo_i = ((i & ~(j - 1)) << 1) | (i & (j - 1));
				uint32_t hi_i = lo_i | j;
				bool asc = (lo_i & k) == 0;
				uint32_t a = s_key[lo_i], bb = s_key[hi_i];
				if((a > bb) == asc) {
					s_key[lo_i] = bb;
					s_key[hi_i] = a;
				}
			}
			__syncthreads();
		}
		for(uint32_t ch = wave_s; ch < nchunks; ch += kSortThreads / 64) {
			uint32_t v[4];
#pragma unroll
			for(int e = 0; e < 4; e++)
				v[e] = s_key[ch * 256 + e * 64 + lane_s];
			bitonic_merge<4, 128>(v, ((ch * 256) & k) ? ~0u : 0u);
#pragma unroll
			for(int e = 0; e < 4; e++)
				s_key[ch * 256 + e * 64 + lane_s] = v[e];
		}
		__syncthreads();
	}
	// s_key[i] & pmask is the list position of the i-th entry in depth order. Entries are
	// visited in rounds of kSortThreads consecutive positions (coalesced LDS and output).
	const uint32_t rounds = (m + kSortThreads - 1) / kSortThreads;
	const uint32_t nw = s_parts, total = s_total;
	uint32_t *tri_out = hdr + kSortedHeader;
	uint64_t *mask_out = (uint64_t *)(hdr + sorted_mask_offset(m));
	// wave w starts at the first entry with at least w * total / nw samples before it whose
	// depth rank differs from its predecessor's: the waves' ranges are chained per pixel
	// and must not split a group of equal ranks (whose order is only the list order). The
	// running prefix is a block scan per round (wave scans, then the wave totals).
	// Equal ranks are ordered by list position only. The forward's ordering window absorbs
	// that, but the backward's pass A flushes its window at every slice, so in frames with
	// fp32 samples (the differentiable ones) each run of equal ranks that lies within one
	// round (and is at most kTieRun long) is put in exact depth-key order here: its members
	// take their place among the run by their full depth keys.
	const bool exact_runs = (c.opts & LUCID_OPT_FP32_SAMPLES) != 0 && !unsorted;
	uint32_t carry = 0, found = 0;
	if(!exact_runs) {
		// Without the exact runs, the range starts need only the sample counts, which pass 1
		// left in LDS: each thread takes a contiguous run of sorted positions, one block scan
		// of the runs' totals gives the samples before each entry, and the output is a copy
		// with no barrier between its loads.
		const uint32_t per = (m + kSortThreads - 1) / kSortThreads;
		const uint32_t i0 = min(m, threadIdx.x * per), i1 = min(m, i0 + per);
		uint32_t sum = 0;
		for(uint32_t i = i0; i < i1; i++)
			sum += s_smp[s_key[i] & pmask];
		const uint32_t inc = wave_inclusive_add(sum);
		if(lane_s == 63)
			s_wsum[0][wave_s] = inc;
		__syncthreads();
		uint32_t run = inc - sum;
#pragma unroll
		for(int w = 0; w < kSortThreads / 64; w++)
			run += w < wave_s ? s_wsum[0][w] : 0u;
		for(uint32_t i = i0; i < i1; i++) {
			const uint32_t key = s_key[i];
			const bool cut = unsorted || i == 0 || (key >> pb) != (s_key[i - 1] >> pb);
			for(uint32_t w = 1; w < nw; w++) {
				const uint32_t target = (uint32_t)(((uint64_t)w * total) / nw);
				if(!((found >> w) & 1u) && run >= target && cut) {
					atomicMin(&s_bound[w], i);
					found |= 1u << w;
				}
			}
			run += s_smp[key & pmask];
		}
		for(uint32_t i = threadIdx.x; i < m; i += 4 * kSortThreads) {
			uint4 en[4];
#pragma unroll
			for(int k = 0; k < 4; k++) {
				const uint32_t ik = i + k * kSortThreads;
				en[k] = ik < m ? list[s_key[ik] & pmask] : make_uint4(0u, 0u, 0u, 0u);
			}
#pragma unroll
			for(int k = 0; k < 4; k++) {
				const uint32_t ik = i + k * kSortThreads;
				if(ik < m)
					tri_out[ik] = en[k].x, mask_out[ik] = entry_mask(en[k]);
			}
		}
	}
	for(uint32_t r = 0; r < rounds && exact_runs; r++) {
		const uint32_t i = r * kSortThreads + threadIdx.x;
		const uint32_t r0 = r * kSortThreads, r1 = min(m, r0 + kSortThreads);
		uint32_t tri = 0, key = 0, dk = 0;
		uint64_t msk = 0;
		bool tie = false;
		if(i < m) {
			key = s_key[i];
			const uint4 en = list[key & pmask];
			tri = en.x, dk = en.y, msk = entry_mask(en);
			tie = exact_runs && ((i > 0 && (s_key[i - 1] >> pb) == (key >> pb)) ||
								 (i + 1 < m && (s_key[i + 1] >> pb) == (key >> pb)));
		}
		s_tdk[r & 1][threadIdx.x] = dk;
		const uint32_t smp = (uint32_t)__popcll(msk);
		const uint32_t inc = wave_inclusive_add(smp);
		if(lane_s == 63)
			s_wsum[r & 1][wave_s] = inc;
		__syncthreads();
		uint32_t before = carry, round_tot = 0;
#pragma unroll
		for(int w = 0; w < kSortThreads / 64; w++) {
			const uint32_t t = s_wsum[r & 1][w];
			before += w < wave_s ? t : 0u;
			round_tot += t;
		}
		carry += round_tot;
		if(i < m) {
			const uint32_t run = before + inc - smp; // samples of the entries before i
			const bool cut = unsorted || i == 0 || (s_key[i] >> pb) != (s_key[i - 1] >> pb);
			for(uint32_t w = 1; w < nw; w++) {
				const uint32_t target = (uint32_t)(((uint64_t)w * total) / nw);
				if(!((found >> w) & 1u) && run >= target && cut) {
					atomicMin(&s_bound[w], i);
					found |= 1u << w;
				}
			}
			uint32_t out = i;
			if(tie) {
				const uint32_t rk = key >> pb;
				uint32_t gs = i, ge = i;
				while(gs > r0 && i - gs < kTieRun && (s_key[gs - 1] >> pb) == rk)
					gs--;
				while(ge + 1 < r1 && ge - i < kTieRun && (s_key[ge + 1] >> pb) == rk)
					ge++;
				// the whole run is [gs, ge]: it starts and ends within this round
				const bool inside = (gs == 0 || (s_key[gs - 1] >> pb) != rk) &&
									(ge + 1 >= m || (s_key[ge + 1] >> pb) != rk) && ge - gs < kTieRun;
				if(inside) {
					uint32_t ahead = 0;
					for(uint32_t k = gs; k <= ge; k++) {
						const uint32_t dk_k = s_tdk[r & 1][k - r0];
						const uint32_t j_k = s_key[k] & pmask;
						ahead += (dk_k < dk || (dk_k == dk && j_k < (key & pmask))) ? 1u : 0u;
					}
					out = gs + ahead;
				}
			}
			tri_out[out] = tri;
			mask_out[out] = msk;
		}
	}
	__syncthreads();
	if(threadIdx.x == 0) {
		hdr[0] = nw;
		for(uint32_t w = 0; w < nw; w++)
			hdr[1 + w] = s_bound[w];
		hdr[1 + nw] = m;
		b.blk_sorted[slot] = s_base;
		b.blk_flags[slot] = LUCID_BIN_LEVEL_HIGH | kSlotPresorted;
	}
}

__global__ __launch_bounds__(kSortThreads) void high_finalize_kernel(FrameConst c, FrameBufs b) {
	high_finalize_kernel_body<kMidSortCap>(c, b, WgPos{bin_run_id<16>(blockIdx.x, gridDim.x), gridDim.x});
}

// The long-list pass over the blocks queued by the first: work-group w of `count` takes
// queue entries w, w + count, ... (the queue is complete: the first pass has finished).
__device__ __forceinline__ void high_finalize_long_body(const FrameConst &c, const FrameBufs &b,
														 WgPos wg) {
	if(b.ctrl[kCtrlOverflow] & (kOvfBinLists | kOvfLists))
		return;
	const uint32_t n = b.ctrl[kCtrlBigSorts];
	for(uint32_t q = wg.id; q < n; q += wg.count) {
		high_finalize_kernel_body<(uint32_t)kBigSortCap>(c, b, WgPos{b.big_queue[q], 0u});
		__syncthreads(); // the next block reuses the work-group's LDS
	}
}
__global__ __launch_bounds__(kSortThreads) void high_finalize_long_kernel(FrameConst c, FrameBufs b) {
	high_finalize_long_body(c, b, WgPos{blockIdx.x, gridDim.x});
}
__global__ __launch_bounds__(kSortThreads) void high_finalize_kernel_batch(const FrameDesc *__restrict__ frames,
		const uint32_t *__restrict__ pre, uint32_t num_frames) {
	const StageBatch sb{frames, pre, num_frames};
	const uint32_t wg = bin_run_id<16>(blockIdx.x, gridDim.x);
	const uint32_t f = batch_frame(sb, wg);
	const FrameDesc &d = sb.frames[f];
	high_finalize_kernel_body<kMidSortCap>(d.c, d.b, WgPos{wg - sb.pre[f], sb.pre[f + 1] - sb.pre[f]});
}
__global__ __launch_bounds__(kSortThreads) void high_finalize_long_kernel_batch(const FrameDesc *__restrict__ frames,
		const uint32_t *__restrict__ pre, uint32_t num_frames) {
	const StageBatch sb{frames, pre, num_frames};
	const uint32_t f = batch_frame(sb, blockIdx.x);
	const FrameDesc &d = sb.frames[f];
	high_finalize_long_body(d.c, d.b, WgPos{blockIdx.x - sb.pre[f], sb.pre[f + 1] - sb.pre[f]});
}

// ------------------------------------------------------------------ block_raster

// 64 x 64 bit-matrix transpose across the wave: lane i holds row i (bit j = column j) and
// receives row i of the transpose. Six butterfly stages; at stage s lanes i and i ^ s swap
// the off-diagonal s x s blocks: the lower lane keeps its columns with (j & s) == 0 and
// takes the partner's as columns j + s, the upper lane keeps its columns with (j & s) != 0
// and takes the partner's, shifted down by s (Hacker's Delight, 7-3, one row per lane).
// Stages 32 and 16 are row swaps of whole words and of packed halves; stage 8 picks bytes; the
// others rotate the partner's word into place and merge it under a column mask, both chosen by
// the lane's bit s.
__device__ __forceinline__ uint64_t transpose64(uint64_t row) {
	int lane = lane_id();
	// The lane's selectors are made here on every call (a dozen instructions): kept across the
	// slice loops they cost a wave per SIMD (fp32 pre-sorted blocks 130 registers instead of 128,
	// 241 us instead of 204 for 41 M fragments at 512 x 512).
	asm volatile("" : "+v"(lane));
	const auto w32 = __builtin_amdgcn_permlane32_swap((uint32_t)row, (uint32_t)(row >> 32), false, false);
	const uint32_t l16 = __builtin_amdgcn_perm(w32[1], w32[0], 0x05040100u); // the low halves
	const uint32_t h16 = __builtin_amdgcn_perm(w32[1], w32[0], 0x07060302u); // the high halves
	const auto w16 = __builtin_amdgcn_permlane16_swap(l16, h16, false, false);
	uint32_t w[2] = {__builtin_amdgcn_perm(w16[1], w16[0], 0x05040100u),
					 __builtin_amdgcn_perm(w16[1], w16[0], 0x07060302u)};
	const uint32_t sel8 = (lane & 8) ? 0x03070105u : 0x06020400u;
#pragma unroll
	for(int k = 0; k < 2; k++)
		w[k] = __builtin_amdgcn_perm(lane_xor<8>(w[k]), w[k], sel8);
	auto stage = [&](auto sh, uint32_t cols) {
		constexpr int s = decltype(sh)::value;
		const uint32_t upper = (lane & s) ? ~0u : 0u;
		const uint32_t keep = cols ^ upper;
		const uint32_t ror = ((32u - s) ^ upper) - upper; // down by s (upper lanes), else up
#pragma unroll
		for(int k = 0; k < 2; k++) {
			const uint32_t p = lane_xor<s>(w[k]);
			const uint32_t moved = __builtin_amdgcn_alignbit(p, p, ror);
			w[k] = (w[k] & keep) | (moved & ~keep);
		}
	};
	stage(std::integral_constant<int, 4>{}, 0x0f0f0f0fu);
	stage(std::integral_constant<int, 2>{}, 0x33333333u);
	stage(std::integral_constant<int, 1>{}, 0x55555555u);
	return ((uint64_t)w[1] << 32) | w[0];
}

// Transposes the coverage masks of a slice (64-bit pixel masks, one per entry) into
// per-pixel entry bitmaps: after the call bit e of bm[k] in lane p is set iff entry
// 64 k + e covers pixel p.
template <int W>
__device__ __forceinline__ void transpose_masks(const uint64_t (&msk)[W], int nwords,
												uint64_t (&bm)[W]) {
#pragma unroll
	for(int k = 0; k < W; k++)
		bm[k] = k < nwords ? transpose64(msk[k]) : 0ull;
}

// ------------------------------------------------------------------ flat colour records
//
// Shading modes of the block rasterisers (ShadeMode): the general record (shade_record),
// the same with albedo textures, and flat colour planes for frames with RGBA8 samples, unit
// lighting (identity_light), vertex colours absent or fp32 with a per-triangle alpha, and
// no textures. There a sample's colour is an affine function of the barycentrics, so per
// channel (with d1 = c1 - c0, d2 = c2 - c0 and the barycentric planes e0, e1 with offsets
// P0, P1 of shading.glsl:116-120)
//   c0 + b0 d1 + b1 d2 = K + ray_pos (Lx px + Ly py + Lz),
//   L = e0 d1 + e1 d2,  K = c0 - P0 d1 - P1 d2,
// which the staging computes once per (block, triangle) and the pixel walk evaluates with
// three fused multiply-adds per channel instead of the barycentric interpolation. The value
// is the same affine function (rounding differs by a few ulps, inside the 1/255 colour bar);
// the depth key keeps its unfused evaluation. The instance colour is folded into the planes.
constexpr int kFlatQuads = 5; // f0 depth plane | triangle id; f1-f3 r, g, b planes; f4 alpha
constexpr int shade_kind(int mode) { return mode & ~kShadeNarrow; }
constexpr bool is_flat(int mode) { return shade_kind(mode) == kShadeFlat; }
constexpr bool is_plain(int mode) { return shade_kind(mode) == kShadePlain; }
constexpr bool is_textured(int mode) { return shade_kind(mode) == kShadeTextured; }
constexpr int window_slots(int mode) { return mode & kShadeNarrow ? kNarrowWindow : kWindow; }
constexpr int rec_quads(int mode) { return is_flat(mode) ? kFlatQuads : kRecQuads; }
// LDS of one wave's slice of 64 W records
template <int W, int MODE> constexpr int slice_quads() { return 64 * W * rec_quads(MODE); }

__device__ __forceinline__ void make_flat_record(const uint4 *src, uint4 *dst) {
	const uint4 q0 = src[0], q1 = src[1], q2 = src[2], q3 = src[3], q4 = src[4], q5 = src[5],
				q6 = src[6];
	const uint32_t flags = q0.w & 0xffffu;
	float c0[3] = {1.0f, 1.0f, 1.0f}, c1[3] = {1.0f, 1.0f, 1.0f}, c2[3] = {1.0f, 1.0f, 1.0f};
	float a = 1.0f;
	if(flags & LUCID_INST_HAS_VERTEX_COLORS) {
		c0[0] = bits2f(q3.x), c0[1] = bits2f(q3.y), c0[2] = bits2f(q3.z), a = bits2f(q3.w);
		c1[0] = bits2f(q4.x), c1[1] = bits2f(q4.y), c1[2] = bits2f(q4.z);
		c2[0] = bits2f(q5.x), c2[1] = bits2f(q5.y), c2[2] = bits2f(q5.z);
	}
	if(flags & LUCID_INST_HAS_COLOR) {
		const float4 ic = decode_rgba8(q6.x);
		const float icc[3] = {ic.x, ic.y, ic.z};
#pragma unroll
		for(int k = 0; k < 3; k++)
			c0[k] = icc[k] * c0[k], c1[k] = icc[k] * c1[k], c2[k] = icc[k] * c2[k];
		a = ic.w * a;
	}
	const float e0[3] = {bits2f(q1.x), bits2f(q1.y), bits2f(q1.z)}, p0 = bits2f(q1.w);
	const float e1[3] = {bits2f(q2.x), bits2f(q2.y), bits2f(q2.z)}, p1 = bits2f(q2.w);
	dst[0] = make_uint4(q0.x, q0.y, q0.z, q6.z);
	// a zero alpha contributes nothing (shading.glsl:167-168): zero planes and a zero alpha
	// byte encode such a sample as 0, the RGBA8 word that contributes nothing
	const bool none = a == 0.0f;
#pragma unroll
	for(int k = 0; k < 3; k++) {
		const float d1 = c1[k] - c0[k], d2 = c2[k] - c0[k];
		const float lx = fmaf(e0[0], d1, e1[0] * d2), ly = fmaf(e0[1], d1, e1[1] * d2);
		const float lz = fmaf(e0[2], d1, e1[2] * d2);
		const float kk = fmaf(-p0, d1, fmaf(-p1, d2, c0[k]));
		dst[1 + k] = none ? make_uint4(0u, 0u, 0u, 0u)
						  : make_uint4(f2bits(lx), f2bits(ly), f2bits(lz), f2bits(kk));
	}
	dst[4] = make_uint4(f2u(a * 255.0f) << 24, 0u, 0u, 0u); // RGBA8 alpha byte
}

// RGBA8 sample of a flat record at pixel (px, py); inv_ray = record_inv_depth(f[0], ...).
__device__ __forceinline__ SampleColor<false> shade_flat(const uint4 *f, float px, float py,
														 float inv_ray) {
	const float rp = __builtin_amdgcn_rcpf(inv_ray);
	float rgb[3];
#pragma unroll
	for(int k = 0; k < 3; k++) {
		const uint4 pl = f[1 + k];
		const float l = fmaf(bits2f(pl.x), px, fmaf(bits2f(pl.y), py, bits2f(pl.z)));
		rgb[k] = sat(fmaf(rp, l, bits2f(pl.w)));
	}
	SampleColor<false> out;
	out.enc = (uint32_t)(rgb[0] * 255.0f) | ((uint32_t)(rgb[1] * 255.0f) << 8) |
			  ((uint32_t)(rgb[2] * 255.0f) << 16) | f[4].x;
	return out;
}

// ------------------------------------------------------------------ plain records
//
// Frames with fp32 samples whose instances all have fp32 vertex colours, unit lighting and no
// instance colour (kShadePlain) keep the general record's planes and colours (its first six
// quads, the triangle id in place of the flags; still kRecQuads apart, as six quads would put
// twice as many entries on one LDS bank) and evaluate the general shading without its tests of
// instance flags and frame options: the same operations on the same values, bit for bit. These
// kernels are bound by VALU issue: 41 M fragments at 512 x 512, forward raster 204 -> 175 us, pass A
// 214 -> 179, pass B 534 -> 441 (with its eight rotated orders and 12.5 KB of LDS instead of 15.5).
constexpr int kPlainQuads = 6; // depth plane | triangle id; two barycentric planes; c0 | alpha; c1; c2

struct PlainShade {
	float b0, b1; // barycentrics
	float x[3];   // interpolated colour, unclamped
	float alpha;
};
__device__ __forceinline__ PlainShade shade_plain(const uint4 *q, float px, float py, float inv_ray) {
	PlainShade o;
	const uint4 p0 = q[1], p1 = q[2], q3 = q[3], q4 = q[4], q5 = q[5];
	const float ray_pos = __builtin_amdgcn_rcpf(inv_ray);
	const float e0 = bits2f(p0.x) * px + (bits2f(p0.y) * py + bits2f(p0.z));
	const float e1 = bits2f(p1.x) * px + (bits2f(p1.y) * py + bits2f(p1.z));
	o.b0 = e0 * ray_pos - bits2f(p0.w);
	o.b1 = e1 * ray_pos - bits2f(p1.w);
	const float w0 = (1.0f - o.b0) - o.b1;
	o.x[0] = w0 * bits2f(q3.x) + (o.b0 * bits2f(q4.x) + o.b1 * bits2f(q5.x));
	o.x[1] = w0 * bits2f(q3.y) + (o.b0 * bits2f(q4.y) + o.b1 * bits2f(q5.y));
	o.x[2] = w0 * bits2f(q3.z) + (o.b0 * bits2f(q4.z) + o.b1 * bits2f(q5.z));
	o.alpha = bits2f(q3.w);
	return o;
}
__device__ __forceinline__ SampleColor<true> plain_sample(const uint4 *q, float px, float py, float inv_ray) {
	const PlainShade p = shade_plain(q, px, py, inv_ray);
	SampleColor<true> out;
	out.col = make_float4(sat(p.x[0]), sat(p.x[1]), sat(p.x[2]), p.alpha);
	return out;
}

// Stages the shading records of a slice in LDS: lane l writes entries l + 64 k.
template <int W, int MODE = kShadeGeneral>
__device__ __forceinline__ void stage_slice(const FrameConst &c, const FrameBufs &b,
											const uint32_t (&tri)[W], uint32_t n,
											uint4 *s_rec) {
	const int lane = lane_id();
#pragma unroll
	for(int k = 0; k < W; k++) {
		const uint32_t i = k * 64 + lane;
		if(i < n) {
			// quad by quad (no staging array: with a record pointer read from memory, as in a
			// batched launch, an array between the load and the LDS store went to scratch)
			const uint4 *src = b.tri_shade + (size_t)kRecStride * tri_rec(b, tri[k]);
			if constexpr(is_flat(MODE)) {
				make_flat_record(src, s_rec + i * kFlatQuads);
			} else if constexpr(is_plain(MODE)) {
				const uint4 q0 = src[0];
				s_rec[i * kRecQuads] = make_uint4(q0.x, q0.y, q0.z, tri[k]);
#pragma unroll
				for(int j = 1; j < kPlainQuads; j++)
					s_rec[i * kRecQuads + j] = src[j];
			} else {
#pragma unroll
				for(int j = 0; j < kRecQuads; j++)
					s_rec[i * kRecQuads + j] = src[j];
			}
		}
	}
}

// LUCID_OPT_ALPHA_THRESHOLD (shading.glsl:62,282-284; raster_low.glsl:258-260): once every
// pixel of a wave has transmittance below 1/128, the wave's later samples are not shaded
// (their fragments are still counted). "Over" blending only.
constexpr float kAlphaThreshold = 1.0f / 128.0f;
__device__ __forceinline__ bool alpha_threshold_on(const FrameConst &c) {
	return (c.opts & LUCID_OPT_ALPHA_THRESHOLD) && !(c.opts & LUCID_OPT_ADDITIVE_BLENDING);
}
__device__ __forceinline__ bool all_below_alpha_threshold(float trans) {
	return ballot(!(trans < kAlphaThreshold)) == 0ull;
}

// Visits this lane's set bitmap bits in increasing entry order, one per step. The loop is
// divergent: a lane leaves when its bits run out (the wave steps until every lane is done),
// so the lane's state needs no copies for lanes that sit out a step.
template <int W, class Visit>
__device__ __forceinline__ void walk_bits(uint64_t (&bm)[W], Visit &&visit) {
	while(true) {
		bool nz[W], any = false;
#pragma unroll
		for(int k = 0; k < W; k++) {
			nz[k] = bm[k] != 0ull;
			any = any || nz[k];
		}
		if(!any)
			break;
		uint64_t cur = bm[W - 1];
		int word = W - 1;
#pragma unroll
		for(int k = W - 2; k >= 0; k--) {
			cur = nz[k] ? bm[k] : cur;
			word = nz[k] ? k : word;
		}
		const uint64_t rest = cur & (cur - 1ull);
#pragma unroll
		for(int k = 0; k < W; k++)
			bm[k] = word == k ? rest : bm[k];
		visit(word * 64 + (int)__builtin_ctzll(cur));
	}
}

// OVER: the common case compiled apart (sorted, front-to-back "over"), so that its loop
// carries no test of the blend options; otherwise they are read per sample.
template <bool FP32, int W, int MODE, bool OVER, class PS>
__device__ __forceinline__ void walk_pixel_t(const FrameConst &c, const FrameBufs &b,
											 const uint4 *s_rec, const uint4 *s_tex,
											 uint64_t (&bm)[W], float px, float py, PS &ps,
											 bool additive_opt) {
	const bool unsorted = !OVER && (c.opts & LUCID_OPT_UNSORTED) != 0;
	const bool additive = !OVER && additive_opt;
	if constexpr(is_flat(MODE)) {
		static_assert(!FP32, "flat records carry RGBA8 samples");
		walk_bits(bm, [&](int e) {
			const uint4 *rec = s_rec + e * kFlatQuads;
			const uint4 f0 = rec[0];
			const float inv = record_inv_depth(f0, px, py);
			const SampleColor<false> col = shade_flat(rec, px, py, inv);
			// a sample that contributes nothing (word 0) blends as nothing, so it is not
			// tested for: it takes its place in the window like any other
			if(unsorted)
				ps.acc.blend(col, additive);
			else
				ps.insert(pixel_key(inv, f0.w), col, additive);
		});
		return;
	}
	if constexpr(is_plain(MODE)) {
		static_assert(FP32, "plain records carry fp32 samples");
		walk_bits(bm, [&](int e) {
			const uint4 *rec = s_rec + e * kRecQuads;
			const uint4 q0 = rec[0];
			const float inv = record_inv_depth(q0, px, py);
			const SampleColor<true> col = plain_sample(rec, px, py, inv);
			if(col.contributes()) {
				if(unsorted)
					ps.acc.blend(col, additive);
				else
					ps.insert(pixel_key(inv, q0.w), col, additive);
			}
		});
		return;
	}
	constexpr bool TEX = is_textured(MODE);
	walk_bits(bm, [&](int e) {
		const uint4 *rec = s_rec + e * kRecQuads;
		const uint4 q0 = rec[0];
		const float inv = record_inv_depth(q0, px, py);
		const SampleColor<FP32> col = shade_record<FP32, TEX>(c, b, s_tex, rec, px, py, inv);
		if(col.contributes()) {
			if(unsorted)
				ps.acc.blend(col, additive); // list order, no depth order
			else
				ps.insert(pixel_key(inv, rec[6].z), col, additive);
		}
	});
}

template <bool FP32, int W, int MODE, class PS>
__device__ __forceinline__ void walk_pixel(const FrameConst &c, const FrameBufs &b,
										   const uint4 *s_rec, const uint4 *s_tex,
										   uint64_t (&bm)[W], float px, float py, PS &ps,
										   bool additive) {
	if(!additive && !(c.opts & LUCID_OPT_UNSORTED))
		walk_pixel_t<FP32, W, MODE, true>(c, b, s_rec, s_tex, bm, px, py, ps, false);
	else
		walk_pixel_t<FP32, W, MODE, false>(c, b, s_rec, s_tex, bm, px, py, ps, additive);
}

template <int W>
__device__ __forceinline__ uint32_t bitmap_count(const uint64_t (&bm)[W]) {
	uint32_t n = 0;
#pragma unroll
	for(int k = 0; k < W; k++)
		n += (uint32_t)__popcll(bm[k]);
	return n;
}

// Writes the pixel, queues the block's mis-ordered pixels for the exact sort and adds the
// frame statistics (one lane per block pixel).
__device__ __forceinline__ void finish_pixels(const FrameConst &c, const FrameBufs &b,
											  const Accum &acc, bool bad, uint32_t count, int px,
											  int py, uint32_t slot, uint32_t m) {
	const int lane = lane_id();
	const bool on_screen = px < c.width && py < c.height;
	write_pixel(c, b, px, py, acc, count);
	enqueue_pixels(b, slot, bad && on_screen, px, py, false);
	const uint32_t frags = wave_read(wave_inclusive_add(on_screen ? count : 0u), 63);
	if(lane == 0) {
		atomicAdd(stat_stripe(b.ctrl, 0, slot % kStatStripes), frags);
		if(m)
			atomicAdd(stat_stripe(b.ctrl, 1, slot % kStatStripes), m);
	}
}

// One wave per block whose list fits the register sort (every low bin, most high blocks):
// sorts the list by centroid depth in registers, then walks every pixel through it slice by
// slice (each slice's shading records staged in LDS: s_rec, the wave's own).
template <bool FP32, int W, int MODE>
__device__ __forceinline__ void raster_sorted_block(const FrameConst &c, const FrameBufs &b,
													uint32_t slot, uint4 *s_rec,
													const uint4 *s_tex) {
	const int lane = lane_id();
	const int bin = slot >> 4, blk = slot & 15, by = blk >> 2, bx = blk & 3;
	const int bin_x = (bin % c.bin_count_x) * kBinSize, bin_y = (bin / c.bin_count_x) * kBinSize;
	const int px0 = bin_x + bx * 8, py0 = bin_y + by * 8;
	const int px = px0 + (lane & 7), py = py0 + (lane >> 3);
	const uint32_t flags = b.blk_flags[slot];
	const uint32_t level = flags & kSlotLevelMask;
	if(flags & (kSlotWhole | kSlotPromoted | kSlotPresorted))
		return; // fallback kernel, overflowed frame, or the pre-sorted blocks' work-groups
	Accum bg;
	bg.init();
	if(level == LUCID_BIN_LEVEL_EMPTY) {
		write_pixel(c, b, px, py, bg, 0u);
		return;
	}
	const uint2 sl = b.blk_slot[slot];
	const uint32_t m = sl.y;
	if(m == 0) {
		write_pixel(c, b, px, py, bg, 0u);
		return;
	}
	if(b.ctrl[kCtrlRecorded])
		return; // the recording pass A renders this block
	const uint4 *list = b.blk_lists + sl.x;
	uint64_t msk_all[4];
	uint32_t tri_all[4];
	if(c.opts & LUCID_OPT_UNSORTED) { // list order
#pragma unroll
		for(int j = 0; j < 4; j++) {
			msk_all[j] = 0, tri_all[j] = 0;
			if(j * 64 + lane < (int)m) {
				const uint4 en = list[j * 64 + lane];
				msk_all[j] = entry_mask(en);
				tri_all[j] = en.x;
			}
		}
	} else {
		// the sort leaves the masks and triangle ids by list position in the (not yet used)
		// slice staging area; the lanes read them back in depth order
		static_assert(slice_quads<W, MODE>() * sizeof(uint4) >=
						  kRegSortCap * (sizeof(uint64_t) + sizeof(uint32_t)),
					  "the sort's masks and ids fit the staging area");
		uint64_t *s_msk = reinterpret_cast<uint64_t *>(s_rec);
		uint32_t *s_tri = reinterpret_cast<uint32_t *>(s_msk + kRegSortCap);
		uint32_t pos[4];
		sort_block_positions(list, m, pos, s_msk, s_tri);
		wave_sync_lds();
#pragma unroll
		for(int j = 0; j < 4; j++) {
			msk_all[j] = 0, tri_all[j] = 0;
			if(j * 64 + lane < (int)m) {
				msk_all[j] = s_msk[pos[j]];
				tri_all[j] = s_tri[pos[j]];
			}
		}
		wave_sync_lds(); // read before the first slice is staged over them
	}
	const bool additive = (c.opts & (1u << 5)) != 0;
	const bool threshold = alpha_threshold_on(c);
	PixelState<FP32, window_slots(MODE)> ps;
	ps.init();
	uint32_t count = 0;
	bool opaque = false; // every pixel of the block is nearly opaque (alpha threshold)
	static_assert(4 % W == 0, "register-sorted lists split into whole slices");
	for(uint32_t s0 = 0; s0 < m; s0 += (64 * W)) {
		const int j0 = (int)(s0 / 64);
		uint64_t msk[W];
		uint32_t tri[W];
#pragma unroll
		for(int k = 0; k < W; k++) {
			msk[k] = msk_all[k], tri[k] = tri_all[k];
#pragma unroll
			for(int j = W; j < 4; j++)
				if(j0 + k == j)
					msk[k] = msk_all[j], tri[k] = tri_all[j];
		}
		const uint32_t n = min(m - s0, (uint32_t)(64 * W));
		if(!opaque)
			stage_slice<W, MODE>(c, b, tri, n, s_rec); // loads in flight during the transpose
		uint64_t bm[W];
		transpose_masks(msk, (int)((n + 63) / 64), bm);
		count += bitmap_count(bm);
		if(opaque)
			continue; // counted, not shaded
		wave_sync_lds();
		walk_pixel<FP32, W, MODE>(c, b, s_rec, s_tex, bm, (float)px, (float)py, ps, additive);
		wave_sync_lds(); // every lane is done with this slice's records
		opaque = threshold && all_below_alpha_threshold(ps.acc.tr);
	}
	ps.flush(additive);
	finish_pixels(c, b, ps.acc, ps.w.bad, count, px, py, slot, m);
}

// Pre-sorted lists longer than one register sort: one work-group per block. Wave w takes
// the contiguous depth range [start[w], start[w + 1]) of the sorted list (ranges balanced
// by sample count), walks it slice by slice with one ordering window per pixel, and leaves
// a partial composite; wave 0 chains the partials front to back. A pixel is exact iff each
// range's blended keys increase and every range starts behind the previous one's last key.
template <bool FP32, int W, int MODE>
__device__ __forceinline__ void raster_presorted_block(const FrameConst &c, const FrameBufs &b,
													   uint32_t id,
													   uint4 (&s_rec)[kBigWaves][slice_quads<W, MODE>()],
													   const uint4 *s_tex) {
	const lucid_info *info = (const lucid_info *)b.info;
	const uint32_t hslot = id >> 4;
	if(hslot >= (uint32_t)info->bin_level_counts[LUCID_BIN_LEVEL_HIGH])
		return;
	const int blk = id & 15, by = blk >> 2, bx = blk & 3;
	const int bin = (int)b.info[LUCID_INFO_U32_SIZE + LUCID_COUNTS_HIGH_BINS * c.bin_count + hslot];
	const uint32_t slot = (uint32_t)bin * 16 + blk;
	const uint32_t flags = b.blk_flags[slot];
	if(!(flags & kSlotPresorted) || (flags & kSlotPromoted) || b.ctrl[kCtrlRecorded])
		return; // (a recording pass A renders the block)
	// Each wave's slice staging area holds, once its walk is done, what the chaining of the
	// ranges reads: 20 KB of LDS per work-group (flat records) instead of 29, so that more
	// work-groups fit on a CU.
	struct RangeEnd {
		float4 part[64]; // the range's partial composite
		uint64_t first[64], last[64];
		uint32_t cnt[64]; // fragments | 0x80000000 when the range's order is not exact
	};
	static_assert(sizeof(RangeEnd) <= sizeof(s_rec[0]), "a range's end state fits its staging");
	auto range_end = [&](int w) -> RangeEnd & { return *reinterpret_cast<RangeEnd *>(&s_rec[w][0]); };
	const int wave = threadIdx.x >> 6, lane = lane_id();
	const uint32_t m = b.blk_slot[slot].y;
	const uint32_t *hdr = b.sorted_pool + b.blk_sorted[slot];
	const uint32_t nw = hdr[0];
	const uint32_t *tri = hdr + kSortedHeader;
	const uint64_t *mask = (const uint64_t *)(hdr + sorted_mask_offset(m));
	const int bin_x = (bin % c.bin_count_x) * kBinSize, bin_y = (bin / c.bin_count_x) * kBinSize;
	const int px0 = bin_x + bx * 8, py0 = bin_y + by * 8;
	const int px = px0 + (lane & 7), py = py0 + (lane >> 3);
	const bool additive = (c.opts & (1u << 5)) != 0;
	if((uint32_t)wave < nw) {
		const uint32_t e0 = hdr[1 + wave], e1 = hdr[2 + wave];
		PixelState<FP32, window_slots(MODE)> ps;
		ps.init();
		uint32_t count = 0;
		const bool threshold = alpha_threshold_on(c);
		bool opaque = false; // every pixel is nearly opaque within this range (alpha threshold)
		for(uint32_t s0 = e0; s0 < e1; s0 += (64 * W)) {
			const uint32_t n = min(e1 - s0, (uint32_t)(64 * W));
			uint64_t msk[W];
			uint32_t t[W];
#pragma unroll
			for(int k = 0; k < W; k++) {
				uint32_t i = k * 64 + lane;
				msk[k] = i < n ? mask[s0 + i] : 0ull;
				t[k] = i < n && !opaque ? tri[s0 + i] : 0u;
			}
			if(!opaque)
				stage_slice<W, MODE>(c, b, t, n, s_rec[wave]); // loads in flight during the transpose
			uint64_t bm[W];
			transpose_masks(msk, (int)((n + 63) / 64), bm);
			count += bitmap_count(bm);
			if(opaque)
				continue; // counted, not shaded
			wave_sync_lds();
			walk_pixel<FP32, W, MODE>(c, b, s_rec[wave], s_tex, bm, (float)px, (float)py, ps, additive);
			wave_sync_lds(); // every lane is done with this slice's records
			// the range's own transmittance bounds the pixel's (earlier ranges only lower it)
			opaque = threshold && all_below_alpha_threshold(ps.acc.tr);
		}
		ps.flush(additive);
		wave_sync_lds(); // every lane is done with the staged records (also after an early end)
		RangeEnd &re = range_end(wave);
		re.part[lane] = make_float4(ps.acc.cr, ps.acc.cg, ps.acc.cb, ps.acc.tr);
		re.first[lane] = ps.w.first;
		re.last[lane] = ps.w.last;
		re.cnt[lane] = count | (ps.w.bad ? 0x80000000u : 0u);
	}
	__syncthreads();
	if(wave != 0)
		return;
	Accum acc;
	acc.init();
	uint64_t last = 0;
	bool bad = false;
	uint32_t count = 0;
	for(uint32_t w = 0; w < nw; w++) {
		const RangeEnd &re = range_end((int)w);
		const uint32_t cw = re.cnt[lane];
		count += cw & 0x7fffffffu;
		bad |= (cw >> 31) != 0;
		const uint64_t f = re.first[lane];
		if(f != 0ull) { // the range has samples here
			bad |= f <= last;
			last = re.last[lane];
			const float4 p = re.part[lane];
			acc.cr = acc.cr + acc.tr * p.x;
			acc.cg = acc.cg + acc.tr * p.y;
			acc.cb = acc.cb + acc.tr * p.z;
			acc.tr = acc.tr * p.w;
		}
	}
	finish_pixels(c, b, acc, bad, count, px, py, slot, m);
}

// Register-sorted blocks alone (one wave each) and pre-sorted blocks alone.
template <bool FP32, int W, int MODE>
__device__ __forceinline__ void block_raster_body(const FrameConst &c, const FrameBufs &b,
												  uint32_t id) {
	__shared__ uint4 s_rec[slice_quads<W, MODE>()];
	__shared__ uint4 s_tex[is_textured(MODE) ? kTexTable : 1];
	if(b.ctrl[kCtrlOverflow] & kOvfBinLists)
		return;
	if constexpr(is_textured(MODE))
		fill_tex_table(b, s_tex); // (one wave: the syncs before the first walk cover it)
	raster_sorted_block<FP32, W, MODE>(c, b, id, s_rec, s_tex);
}
template <bool FP32, int W, int MODE>
__device__ __forceinline__ void block_raster_big_body(const FrameConst &c, const FrameBufs &b,
													  uint32_t id) {
	__shared__ uint4 s_rec[kBigWaves][slice_quads<W, MODE>()];
	__shared__ uint4 s_tex[is_textured(MODE) ? kTexTable : 1];
	if(b.ctrl[kCtrlOverflow] & kOvfBinLists)
		return;
	if constexpr(is_textured(MODE)) {
		fill_tex_table(b, s_tex);
		__syncthreads();
	}
	raster_presorted_block<FP32, W, MODE>(c, b, id, s_rec, s_tex);
}
template <bool FP32, int W, int MODE>
__global__ __launch_bounds__(64) void block_raster_kernel(FrameConst c, FrameBufs b) {
	block_raster_body<FP32, W, MODE>(c, b, bin_run_id<16>(blockIdx.x, gridDim.x));
}
template <bool FP32, int W, int MODE>
__global__ __launch_bounds__(64) void block_raster_kernel_batch(const FrameDesc *__restrict__ frames,
		const uint32_t *__restrict__ pre, uint32_t num_frames) {
	const StageBatch sb{frames, pre, num_frames};
	const uint32_t wg = bin_run_id<16>(blockIdx.x, gridDim.x);
	const uint32_t f = batch_frame(sb, wg);
	const FrameDesc &d = sb.frames[f];
	block_raster_body<FP32, W, MODE>(d.c, d.b, wg - sb.pre[f]);
}
template <bool FP32, int W, int MODE>
__global__ __launch_bounds__(kBigWaves * 64) void block_raster_big_kernel(FrameConst c, FrameBufs b) {
	block_raster_big_body<FP32, W, MODE>(c, b, bin_run_id<16>(blockIdx.x, gridDim.x));
}
template <bool FP32, int W, int MODE>
__global__ __launch_bounds__(kBigWaves * 64) void block_raster_big_kernel_batch(const FrameDesc *__restrict__ frames,
		const uint32_t *__restrict__ pre, uint32_t num_frames) {
	const StageBatch sb{frames, pre, num_frames};
	const uint32_t wg = bin_run_id<16>(blockIdx.x, gridDim.x);
	const uint32_t f = batch_frame(sb, wg);
	const FrameDesc &d = sb.frames[f];
	block_raster_big_body<FP32, W, MODE>(d.c, d.b, wg - sb.pre[f]);
}

// Both kinds in one launch, for frames of few blocks (launch_block_raster): the first 16 work-groups
// per bin take the pre-sorted blocks, the others four register-sorted blocks each (one wave a
// block, on its own quarter of the LDS), which fill the CUs that run out of the long ones. As two
// launches each ends with a nearly empty chip. fp32 samples: four waves per SIMD, as apart.
static_assert(kBigWaves == 4, "a bin's 16 blocks are four work-groups of register-sorted blocks");
template <bool FP32, int MODE>
__global__ __launch_bounds__(kBigWaves * 64, FP32 ? 4 : 1) void block_raster_fused_kernel(FrameConst c, FrameBufs b) {
	static_assert(!is_textured(MODE), "no texture table here");
	__shared__ uint4 s_rec[kBigWaves][slice_quads<1, MODE>()];
	if(b.ctrl[kCtrlOverflow] & kOvfBinLists)
		return;
	const uint32_t big = (uint32_t)c.bin_count * 16, w = blockIdx.x;
	if(w < big) {
		raster_presorted_block<FP32, 1, MODE>(c, b, bin_run_id<16>(w, big), s_rec, nullptr);
	} else {
		const uint32_t id = bin_run_id<4>(w - big, gridDim.x - big), wave = threadIdx.x >> 6;
		raster_sorted_block<FP32, 1, MODE>(c, b, id * kBigWaves + wave, s_rec[wave], nullptr);
	}
}

// ------------------------------------------------------------------ exact fallback

// Collects the keys (depth key << 32 | triangle id) of one pixel's fragments into `dst`
// (LDS or global) from the block's list (the entries whose pixel mask has `bit`); returns the
// count. Entries beyond `cap` are counted but not stored.
__device__ uint32_t gather_pixel_keys(const FrameBufs &b, const uint4 *list, uint32_t m,
									  int bit, float px, float py, uint64_t *dst, uint32_t cap,
									  bool global_dst) {
	constexpr int kU = 4; // entries per lane per step: their loads are issued together
	const int lane = lane_id();
	uint32_t n = 0;
	for(uint32_t base = 0; base < m; base += 64 * kU) {
		uint4 rec[kU];
#pragma unroll
		for(int k = 0; k < kU; k++) {
			const uint32_t j = base + k * 64 + lane;
			rec[k] = j < m ? list[j] : make_uint4(0u, 0u, 0u, 0u);
		}
		bool hit[kU];
		uint4 d[kU];
#pragma unroll
		for(int k = 0; k < kU; k++) {
			hit[k] = (entry_mask(rec[k]) >> bit) & 1ull;
			d[k] = hit[k] ? b.tri_depth[tri_rec(b, rec[k].x)] : make_uint4(0u, 0u, 0u, 0u);
		}
#pragma unroll
		for(int k = 0; k < kU; k++) {
			const uint64_t key = pixel_key(record_inv_depth(d[k], px, py), rec[k].x);
			const uint64_t bal = ballot(hit[k]);
			if(hit[k]) {
				const uint32_t pos = n + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
				if(pos < cap) {
					if(global_dst)
						__hip_atomic_store(&dst[pos], key, __ATOMIC_RELAXED,
										   __HIP_MEMORY_SCOPE_AGENT);
					else
						dst[pos] = key;
				}
			}
			n += (uint32_t)__popcll(bal);
		}
	}
	return n;
}

// Blends n sorted keys front to back: 64 samples are shaded in parallel, then composited
// in order.
template <bool FP32, bool TEX>
__device__ Accum blend_sorted(const FrameConst &c, const FrameBufs &b, const uint4 *s_tex,
							  const uint64_t *keys, uint32_t n, float px, float py,
							  bool global_src) {
	const int lane = lane_id();
	const bool additive = (c.opts & (1u << 5)) != 0;
	Accum acc;
	acc.init();
	for(uint32_t base = 0; base < n; base += 64) {
		const uint32_t i = base + lane;
		SampleColor<FP32> col;
		col.zero();
		if(i < n) {
			const uint64_t k = global_src ? __hip_atomic_load(&keys[i], __ATOMIC_RELAXED,
															  __HIP_MEMORY_SCOPE_AGENT)
										  : keys[i];
			const uint32_t t = (uint32_t)k;
			col = shade_sample<FP32, TEX>(c, b, s_tex, t, px, py, sample_inv_depth(b, t, px, py));
		}
		const uint32_t cnt = min(64u, n - base);
		for(uint32_t j = 0; j < cnt; j++) {
			const SampleColor<FP32> c2 = col.read((int)j);
			if(c2.contributes())
				acc.blend(c2, additive);
		}
	}
	return acc;
}

// Exact path for one queued pixel: gathers its fragments from the block list, sorts the
// keys (LDS bitonic up to kFallbackCap, else a global spill), shades and blends in order.
template <bool FP32, bool TEX>
__device__ void fallback_pixel(const FrameConst &c, const FrameBufs &b, const uint4 *s_tex,
							   uint4 item, uint64_t *s_keys) {
	const int lane = lane_id();
	const uint32_t slot = item.x;
	const int px = (int)item.y, py = (int)item.z;
	const bool whole = item.w != 0;
	const uint2 sl = b.blk_slot[slot];
	const uint4 *list = b.blk_lists + sl.x;
	const uint32_t m = sl.y;
	const int bit = (py & 7) * 8 + (px & 7);
	const float fx = (float)px, fy = (float)py;
	const uint32_t n = gather_pixel_keys(b, list, m, bit, fx, fy, s_keys, kFallbackCap, false);
	Accum acc;
	if(n <= (uint32_t)kFallbackCap) {
		sort_pixel_keys(s_keys, n);
		acc = blend_sorted<FP32, TEX>(c, b, s_tex, s_keys, n, fx, fy, false);
	} else {
		// deep pixel: sort its keys in a global spill region
		const uint32_t P = next_pow2(n);
		uint32_t off = 0;
		if(lane == 0) {
			off = (uint32_t)atomicAdd(&b.ctrl[kCtrlSpillCursor], P);
			if((uint64_t)off + P > b.spill_cap) {
				atomicOr(&b.ctrl[kCtrlOverflow], kOvfSpill);
				off = 0xffffffffu;
			}
		}
		off = wave_read(off, 0);
		if(off == 0xffffffffu)
			return; // the frame reports an overflow and is rendered again
		uint64_t *g = b.spill + off;
		gather_pixel_keys(b, list, m, bit, fx, fy, g, P, true);
		for(uint32_t i = n + lane; i < P; i += 64)
			__hip_atomic_store(&g[i], ~0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		__threadfence();
		__builtin_amdgcn_wave_barrier();
		bitonic_global_wave(g, P);
		acc = blend_sorted<FP32, TEX>(c, b, s_tex, g, n, fx, fy, true);
	}
	if(lane == 0) {
		write_pixel(c, b, px, py, acc, n);
		if(whole) // these pixels skipped the block rasteriser
			atomicAdd(&((lucid_info *)b.info)->stats[0], n);
	}
}

// Persistent over the per-pixel queue: wave w of the grid takes items w, w + waves, ...
template <bool FP32, bool TEX>
__device__ __forceinline__ void fallback_kernel_body(const FrameConst &c, const FrameBufs &b, WgPos wg) {
	__shared__ uint64_t s_keys[kFallbackThreads / 64][kFallbackCap];
	if(wg.id == 0 && threadIdx.x < 64) {
		// the block kernels' statistics stripes into LucidInfo (stats[0] fragments, [1]
		// block-list entries); the block kernels have finished
		static_assert(kStatStripes == 64, "one stripe per lane");
		uint32_t v[2] = {*stat_stripe(b.ctrl, 0, threadIdx.x), *stat_stripe(b.ctrl, 1, threadIdx.x)};
#pragma unroll
		for(int k = 0; k < 2; k++) {
			v[k] = wave_read(wave_inclusive_add(v[k]), 63);
			if(threadIdx.x == 0 && v[k])
				atomicAdd(&((lucid_info *)b.info)->stats[k], v[k]);
		}
	}
	const uint32_t nq = min(b.ctrl[kCtrlFallbackCount], b.fallback_cap);
	__shared__ uint4 s_tex[TEX ? kTexTable : 1];
	if constexpr(TEX) {
		fill_tex_table(b, s_tex);
		__syncthreads();
	}
	const uint32_t waves = wg.count * (kFallbackThreads / 64);
	const uint32_t w = wg.id * (kFallbackThreads / 64) + (threadIdx.x >> 6);
	for(uint32_t qi = w; qi < nq; qi += waves)
		fallback_pixel<FP32, TEX>(c, b, s_tex, b.fallback_queue[qi], s_keys[threadIdx.x >> 6]);
	// The work-group that empties the queue last ends the frame (with an empty queue, the first one).
	// Nothing is counted per pixel: two atomics each, on words of the whole frame, took 130 of the
	// kernel's 157 us for 17 k pixels of 32 fragments.
	const uint32_t busy = min(wg.count, (nq + kFallbackThreads / 64 - 1) / (kFallbackThreads / 64));
	if(nq ? wg.id >= busy || !last_work_group(b.ctrl, kDoneFallback, wg.id, busy) : wg.id != 0)
		return;
	// stats[2]: pixels resolved by the exact per-pixel sort (the reference counts the pixels its
	// 3-deep window gets wrong there, shading.glsl:258-265)
	if(nq && threadIdx.x == 0)
		((lucid_info *)b.info)->stats[2] = nq;
	// The control words go to pinned host memory, where the host reads them once the frame's
	// event has completed (a copy command of 64 bytes: 4 us of the GPU, and its submission).
	if(b.host_status && threadIdx.x < (uint32_t)kCtrlWords)
		__hip_atomic_store(&b.host_status[threadIdx.x], agent_load(&b.ctrl[threadIdx.x]), __ATOMIC_RELAXED,
						   __HIP_MEMORY_SCOPE_SYSTEM);
}

template <bool FP32, bool TEX>
__global__ __launch_bounds__(kFallbackThreads) void fallback_kernel(FrameConst c, FrameBufs b) {
	fallback_kernel_body<FP32, TEX>(c, b, WgPos{blockIdx.x, gridDim.x});
}
template <bool FP32, bool TEX>
__global__ __launch_bounds__(kFallbackThreads) void fallback_kernel_batch(const FrameDesc *__restrict__ frames,
		const uint32_t *__restrict__ pre, uint32_t num_frames) {
	const StageBatch sb{frames, pre, num_frames};
	const uint32_t f = batch_frame(sb, blockIdx.x);
	const FrameDesc &d = sb.frames[f];
	fallback_kernel_body<FP32, TEX>(d.c, d.b, WgPos{blockIdx.x - sb.pre[f], sb.pre[f + 1] - sb.pre[f]});
}

// ------------------------------------------------------------------ backward (adjoint)
//
// The adjoint of sorted front-to-back compositing for the fp32-sample forward. Fragment
// lists are recomputed (the forward stages run again), never stored across calls. Per block
// (its sorted list split into the depth ranges of the forward, one wave each):
//   pass A  (bwd_pass_a_kernel) walks every pixel through its range with the forward's
//           ordering window, records the order in which samples leave the window (one byte
//           per sample), and accumulates the range's partial composite in fp64; the
//           work-group then chains the ranges per pixel (exactness across ranges, the
//           saturation mask of the output, dL/d(pixel)) and stores each range's start state:
//           T before it and the remainder R = out - C_before;
//   pass B  (bwd_pass_b_kernel) replays the recorded order and per fragment forms
//             dout/dc_i = a_i T_i,   dout/da_i = T_i c_i - R_{i+1} / (1 - a_i)
//           (T and R in fp64, so pixels whose transmittance underflows fp32 stay exact),
//           chains them through the sRGB lighting stage and the barycentric weights, and
//           sums them per (block, entry) in LDS.
// The (block, entry) rows are then reduced per triangle and per vertex by sorted segmented
// sums (reduce.hip): no global atomics on gradient values. Pixels whose window order is not
// exact take the per-pixel exact sort, as in the forward.

// One sample with what its gradient needs.
struct BwdSample {
	float r, g, b, a;  // shaded sample (fp32, as the fp32-sample forward)
	float b0, b1;      // barycentrics: corner weights (1 - b0) - b1, b0, b1
	float dr, dg, db;  // d(sample channel) / d(vertex colour channel) per unit corner weight
	float da;          // d(sample alpha) / d(triangle alpha)
	__device__ __forceinline__ void zero() { r = g = b = a = b0 = b1 = dr = dg = db = da = 0.0f; }
};

// The fp32-sample shading of shade_record with the derivative of the lighting stage,
// s = sat(L2S(S2L(x) f)) (lit_channel: ds/dx = fp above both linear segments, f below both).
__device__ __forceinline__ bool shade_grad(const FrameConst &c, const FrameBufs &b, const uint4 *q,
										   float px, float py, float inv_ray, BwdSample &o) {
	ShadeState st;
	if(!shade_prepare<false>(c, b, nullptr, q, px, py, inv_ray, st)) {
		o.zero();
		return false;
	}
	const float x[3] = {st.color.x, st.color.y, st.color.z};
	const float ic[3] = {st.inst.x, st.inst.y, st.inst.z};
	float sv[3], dv[3];
#pragma unroll
	for(int k = 0; k < 3; k++) {
		LitChannel l;
		if(c.identity_light) // s = x, ds/dx = 1 (the round trip of a unit factor)
			l.s = x[k], l.deriv = 1.0f;
		else
			l = lit_channel<true>(x[k], st.f[k], st.fp[k]);
		sv[k] = sat(l.s);
		// clamp passes the gradient on [0, 1] (as torch.clamp does)
		dv[k] = (l.s >= 0.0f && l.s <= 1.0f) ? l.deriv * ic[k] : 0.0f;
	}
	o.r = sv[0], o.g = sv[1], o.b = sv[2], o.a = st.color.w;
	o.b0 = st.bary0, o.b1 = st.bary1;
	o.dr = dv[0], o.dg = dv[1], o.db = dv[2];
	o.da = st.inst.w;
	return true;
}

// Pass A window payload: the fp32 sample and its entry within the slice.
struct BwdColor {
	float r, g, b, a;
	uint32_t e;
	__device__ __forceinline__ void zero() { r = g = b = a = 0.0f, e = 0; }
	static __device__ __forceinline__ BwdColor sel(bool p, const BwdColor &x, const BwdColor &y) {
		BwdColor o;
		o.r = p ? x.r : y.r, o.g = p ? x.g : y.g, o.b = p ? x.b : y.b, o.a = p ? x.a : y.a;
		o.e = p ? x.e : y.e;
		return o;
	}
};

// fp64 composite (C, T) plus the fp32 composite the forward computes (saturation mask).
struct BwdTotals {
	double t, cr, cg, cb;
	Accum acc;
	__device__ __forceinline__ void init() {
		t = 1.0, cr = cg = cb = 0.0;
		acc.init();
	}
	__device__ __forceinline__ void add(float r, float g, float b, float a) {
		const double da = a;
		cr += (double)r * da * t;
		cg += (double)g * da * t;
		cb += (double)b * da * t;
		t *= 1.0 - da;
		acc.blend(make_float4(r, g, b, a), false);
	}
};

// Adjoint of one fragment of front-to-back "over" compositing, out = sum_i s_i a_i T_i +
// T_end bg. State: t = T before the fragment and q = g . R, the gradient-weighted remainder
// R = out - (composite before the fragment), both fp64 (R cancels to tiny values behind
// deep fragments). dL/da = g . (s T - R_after / (1 - a)) = T (g . s) - q_after / (1 - a),
// dL/ds_c = g_c a T.
__device__ __forceinline__ void bwd_fragment(double &t, double &q, float gr, float gg, float gb,
											 const BwdSample &s, float (&out)[kGradWords]) {
	const double a = s.a;
	const double at = a * t;
	const double gs = (double)gr * (double)s.r + (double)gg * (double)s.g + (double)gb * (double)s.b;
	const double q_after = q - at * gs; // g . (remainder behind this fragment)
	const double om = 1.0 - a;          // exact: a is a float in [0, 1]
	// 1 / om: the v_rcp_f32 seed (relative error ~1e-7) refined by one Newton step
	const double r0 = (double)__builtin_amdgcn_rcpf((float)om);
	const double inv_om = om > 0.0 ? r0 * (2.0 - om * r0) : 0.0;
	const double ga = t * gs - q_after * inv_om;
	const float w = (float)at;
	const float xr = gr * w * s.dr, xg = gg * w * s.dg, xb = gb * w * s.db;
	const float w0 = (1.0f - s.b0) - s.b1;
	out[0] = xr * w0, out[1] = xg * w0, out[2] = xb * w0;
	out[3] = xr * s.b0, out[4] = xg * s.b0, out[5] = xb * s.b0;
	out[6] = xr * s.b1, out[7] = xg * s.b1, out[8] = xb * s.b1;
	out[9] = (float)ga * s.da;
	t *= om;
	q = q_after;
}

// Entries of one block in depth order (pre-sorted pool, or a register sort kept in LDS) and
// this wave's depth range [e0, e1) of them.
struct BlockEntries {
	const uint32_t *tri;
	const uint64_t *mask;
	uint32_t nw, e0, e1;
};

// Valid for the blocks the block kernels process (not empty, whole or promoted, m > 0).
// For lists sorted here only wave 0 may call it (it fills s_tri_all / s_mask_all).
__device__ __forceinline__ BlockEntries bwd_block_entries(const FrameConst &c, const FrameBufs &b,
														  uint32_t slot, uint32_t flags, uint2 sl,
														  int wave, uint32_t *s_tri_all,
														  uint64_t *s_mask_all) {
	const int lane = lane_id();
	const uint32_t m = sl.y;
	BlockEntries ent;
	if(flags & kSlotPresorted) {
		const uint32_t *hdr = b.sorted_pool + b.blk_sorted[slot];
		ent.tri = hdr + kSortedHeader;
		ent.mask = (const uint64_t *)(hdr + sorted_mask_offset(m));
		ent.nw = hdr[0];
		ent.e0 = (uint32_t)wave < ent.nw ? hdr[1 + wave] : m;
		ent.e1 = (uint32_t)wave < ent.nw ? hdr[2 + wave] : m;
		return ent;
	}
	uint32_t pos[4], t[4];
	uint64_t k[4];
	sort_block_positions(b.blk_lists + sl.x, m, pos, s_mask_all, s_tri_all);
	wave_sync_lds();
#pragma unroll
	for(int j = 0; j < 4; j++)
		if(j * 64 + lane < (int)m)
			k[j] = s_mask_all[pos[j]], t[j] = s_tri_all[pos[j]];
	wave_sync_lds(); // read in list order before they are written in depth order
#pragma unroll
	for(int j = 0; j < 4; j++)
		if(j * 64 + lane < (int)m)
			s_mask_all[j * 64 + lane] = k[j], s_tri_all[j * 64 + lane] = t[j];
	wave_sync_lds();
	ent.tri = s_tri_all;
	ent.mask = s_mask_all;
	ent.nw = 1, ent.e0 = 0, ent.e1 = m;
	return ent;
}

// Loads and stages slice [s0, s0 + n) of the block's entries; returns the coverage masks.
template <int MODE>
__device__ __forceinline__ void bwd_stage(const FrameConst &c, const FrameBufs &b,
										  const BlockEntries &ent, uint32_t s0, uint32_t n,
										  uint4 *s_rec, uint64_t (&msk)[kSliceWords]) {
	const int lane = lane_id();
	uint32_t t[kSliceWords];
#pragma unroll
	for(int k = 0; k < kSliceWords; k++) {
		const uint32_t i = k * 64 + lane;
		msk[k] = i < n ? ent.mask[s0 + i] : 0ull;
		t[k] = i < n ? ent.tri[s0 + i] : 0u;
	}
	stage_slice<kSliceWords, MODE>(c, b, t, n, s_rec);
	wave_sync_lds();
}

constexpr uint8_t kSeqEnd = 0xff; // end of a pixel's recorded order within a slice
static_assert(kSliceEntries <= 255, "recorded entries are bytes");

// Byte of the j-th sample that leaves pixel `lane`'s window in the slice starting at sorted
// position s0 of a block whose gradient rows start at row0.
__device__ __forceinline__ size_t seq_index(uint32_t row0, uint32_t s0, uint32_t j, int lane) {
	return ((size_t)row0 + s0 + j) * 64 + (size_t)lane;
}

// The recorded order, start states and rows are sized by the host from an earlier pass; a
// frame that needs more skips the block and per-pixel adjoints and reports kOvfGradRows
// (the host grows the buffers and the caller runs the backward pass again).
__device__ __forceinline__ bool bwd_fits(const FrameBufs &b, const BwdBufs &g) {
	const uint32_t rows = b.ctrl[kCtrlBwdRows], ranges = b.ctrl[kCtrlBwdRanges];
	return rows <= g.seq_rows_cap && rows <= g.rows_cap && ranges <= g.start_cap;
}

// RECORD: run by a forward frame (when the record gate admitted it) instead of the block
// rasterisers of the blocks it covers. It writes their pixels as the forward does (image,
// counts, statistics, exact-fallback queue) and, instead of the start states (which need
// dL/dpixel), the BwdRecord of each (range, pixel) and the pixel's clamp/exact flags;
// bwd_start_kernel turns them into start states when the backward runs.
// WIN: slots of the ordering window (4, or 2 with the narrow-window tuning).
// MODE: kShadePlain or kShadeGeneral.
template <bool RECORD, int WIN, int MODE>
__global__ __launch_bounds__(kBigWaves * 64) void bwd_pass_a_kernel(FrameConst c, FrameBufs b,
																	 BwdBufs g) {
	if(b.ctrl[kCtrlOverflow] & kOvfBinLists)
		return;
	if constexpr(RECORD) {
		if(!b.ctrl[kCtrlRecorded])
			return;
	} else if(!bwd_fits(b, g)) {
		if(blockIdx.x == 0 && threadIdx.x == 0)
			atomicOr(&b.ctrl[kCtrlOverflow], kOvfGradRows);
		return;
	}
	// Each wave's slice staging area holds, once its walk is done, what the chaining of the
	// ranges reads (the range's composites and ordering keys per pixel): 31 KB of LDS per
	// work-group instead of 49, so that four work-groups fit on a CU.
	struct RangeEnd {
		double pc[4][64]; // C rgb, T (fp64)
		float4 p32[64];   // fp32 partial composite
		uint64_t first[64], last[64];
		uint32_t bad[64], count[64]; // count: RECORD, fragments per pixel
	};
	__shared__ uint4 s_rec[kBigWaves][kSliceEntries * kRecQuads];
	static_assert(sizeof(RangeEnd) <= sizeof(s_rec[0]), "a range's end state fits its staging");
	__shared__ uint32_t s_tri_all[kRegSortCap];
	__shared__ uint64_t s_mask_all[kRegSortCap];
	auto range_end = [&](int w) -> RangeEnd & { return *reinterpret_cast<RangeEnd *>(&s_rec[w][0]); };
	const int lane = lane_id(), wave = threadIdx.x >> 6;
	const uint32_t slot = blockIdx.x;
	const uint32_t flags = b.blk_flags[slot];
	const uint32_t level = flags & kSlotLevelMask;
	if(level == LUCID_BIN_LEVEL_EMPTY || (flags & (kSlotWhole | kSlotPromoted)))
		return;
	const uint2 sl = b.blk_slot[slot];
	if(sl.y == 0)
		return;
	const bool presorted = (flags & kSlotPresorted) != 0;
	if(!presorted && wave != 0)
		return; // one range: wave 0 alone (no work-group barrier below on this path)
	const int bin = slot >> 4, blk = slot & 15, by = blk >> 2, bx = blk & 3;
	const int px = (bin % c.bin_count_x) * kBinSize + bx * 8 + (lane & 7);
	const int py = (bin / c.bin_count_x) * kBinSize + by * 8 + (lane >> 3);
	const bool on_screen = px < c.width && py < c.height;
	const float fx = (float)px, fy = (float)py;
	const BlockEntries ent = bwd_block_entries(c, b, slot, flags, sl, wave, s_tri_all, s_mask_all);
	const uint32_t row0 = g.row_base[slot];

	if((uint32_t)wave < ent.nw) {
		std::conditional_t<WIN == kWindow, OrderWindow<BwdColor>, SmallWindow<BwdColor, WIN>> w;
		w.init();
		BwdTotals part;
		part.init();
		uint32_t count = 0;
		for(uint32_t s0 = ent.e0; s0 < ent.e1; s0 += kSliceEntries) {
			const uint32_t n = min(ent.e1 - s0, (uint32_t)kSliceEntries);
			uint64_t msk[kSliceWords];
			bwd_stage<MODE>(c, b, ent, s0, n, s_rec[wave], msk);
			// the triangle of each gradient row (pass B fills the row itself)
			for(uint32_t e = lane; e < n; e += 64)
				g.row_tri[(size_t)row0 + s0 + e] = ent.tri[s0 + e];
			uint64_t bm[kSliceWords];
			transpose_masks(msk, (int)((n + 63) / 64), bm);
			if constexpr(RECORD)
				count += bitmap_count(bm);
			uint32_t j = 0;
			auto emit = [&](const BwdColor &s) {
				part.add(s.r, s.g, s.b, s.a);
				g.seq[seq_index(row0, s0, j, lane)] = (uint8_t)s.e;
				j++;
			};
			walk_bits(bm, [&](int e) {
				const uint4 *rec = s_rec[wave] + e * kRecQuads;
				const uint4 q0 = rec[0];
				const float inv = record_inv_depth(q0, fx, fy);
				SampleColor<true> col;
				if constexpr(is_plain(MODE))
					col = plain_sample(rec, fx, fy, inv);
				else
					col = shade_record<true, false>(c, b, nullptr, rec, fx, fy, inv);
				if(col.contributes()) {
					BwdColor bc;
					bc.r = col.col.x, bc.g = col.col.y, bc.b = col.col.z, bc.a = col.col.w;
					bc.e = (uint32_t)e;
					w.insert(pixel_key(inv, is_plain(MODE) ? q0.w : rec[6].z), bc, emit);
				}
			});
			// the window empties at every slice end, so pass B only needs this slice staged
			w.flush(emit);
			if(j < n)
				g.seq[seq_index(row0, s0, j, lane)] = kSeqEnd;
			wave_sync_lds();
		}
		RangeEnd &re = range_end(wave); // every lane is done with the last slice's records
		re.pc[0][lane] = part.cr, re.pc[1][lane] = part.cg;
		re.pc[2][lane] = part.cb, re.pc[3][lane] = part.t;
		re.p32[lane] = make_float4(part.acc.cr, part.acc.cg, part.acc.cb, part.acc.tr);
		re.first[lane] = w.first, re.last[lane] = w.last;
		re.bad[lane] = w.bad ? 1u : 0u;
		re.count[lane] = count;
	}
	if(presorted)
		__syncthreads();
	else
		wave_sync_lds();
	if((uint32_t)wave >= ent.nw)
		return;

	// chain the ranges front to back (each wave for its own start state)
	const float bg[3] = {c.background[0], c.background[1], c.background[2]};
	double ct[3] = {0.0, 0.0, 0.0}, tt = 1.0;   // composite of all ranges
	double cb4[3] = {0.0, 0.0, 0.0}, tb4 = 1.0; // composite of the ranges before this one
	Accum a32;
	a32.init();
	uint64_t last = 0;
	bool bad = false;
	for(uint32_t v = 0; v < ent.nw; v++) {
		if(v == (uint32_t)wave)
			cb4[0] = ct[0], cb4[1] = ct[1], cb4[2] = ct[2], tb4 = tt;
		const RangeEnd &re = range_end((int)v);
		bad |= re.bad[lane] != 0;
		const uint64_t f = re.first[lane];
		if(f != 0ull) {
			bad |= f <= last;
			last = re.last[lane];
		}
		for(int k = 0; k < 3; k++)
			ct[k] = ct[k] + tt * re.pc[k][lane];
		tt = tt * re.pc[3][lane];
		const float4 p = re.p32[lane];
		a32.cr = a32.cr + a32.tr * p.x;
		a32.cg = a32.cg + a32.tr * p.y;
		a32.cb = a32.cb + a32.tr * p.z;
		a32.tr = a32.tr * p.w;
	}
	const float o32[3] = {a32.cr + a32.tr * bg[0], a32.cg + a32.tr * bg[1],
						  a32.cb + a32.tr * bg[2]};
	if constexpr(RECORD) {
		if(wave == 0) {
			uint32_t count = 0;
			for(uint32_t v = 0; v < ent.nw; v++)
				count += range_end((int)v).count[lane];
			finish_pixels(c, b, a32, bad, count, px, py, slot, sl.y);
			if(on_screen) {
				uint32_t pf = bad ? 0u : 8u;
#pragma unroll
				for(int k = 0; k < 3; k++)
					pf |= (o32[k] >= 0.0f && o32[k] <= 1.0f) ? 1u << k : 0u;
				g.pix_flags[(size_t)py * c.width + px] = (uint8_t)pf;
			}
		}
		BwdRecord rc;
		rc.t = tb4;
#pragma unroll
		for(int k = 0; k < 3; k++)
			rc.d[k] = (ct[k] + tt * (double)bg[k]) - cb4[k];
		g.rec[((size_t)g.range_base[slot] + wave) * 64 + lane] = rc;
		return;
	}
	if(wave == 0)
		enqueue_pixels(b, slot, on_screen && bad, px, py, false);
	float gsel[3] = {0.0f, 0.0f, 0.0f};
	if(on_screen && !bad) {
		const float4 gi = g.grad_image[(size_t)py * c.width + px];
		const float gv[3] = {gi.x, gi.y, gi.z};
#pragma unroll
		for(int k = 0; k < 3; k++)
			gsel[k] = (o32[k] >= 0.0f && o32[k] <= 1.0f) ? gv[k] : 0.0f;
	}
	BwdStart st;
	st.t = tb4;
	st.q = 0.0;
#pragma unroll
	for(int k = 0; k < 3; k++)
		st.q += (double)gsel[k] * ((ct[k] + tt * (double)bg[k]) - cb4[k]);
	st.gr = gsel[0], st.gg = gsel[1], st.gb = gsel[2];
	st.pad = 0.0f;
	g.start[((size_t)g.range_base[slot] + wave) * 64 + lane] = st;
}

// Start states of a recorded frame (what pass A computes at its end once dL/dpixel is
// known): one wave per (block, depth range), as pass B.
__global__ __launch_bounds__(kBigWaves * 64) void bwd_start_kernel(FrameConst c, FrameBufs b,
																	BwdBufs g) {
	if((b.ctrl[kCtrlOverflow] & kOvfBinLists) || !bwd_fits(b, g))
		return;
	const int lane = lane_id(), wave = threadIdx.x >> 6;
	const uint32_t slot = blockIdx.x;
	const uint32_t flags = b.blk_flags[slot];
	const uint32_t level = flags & kSlotLevelMask;
	if(level == LUCID_BIN_LEVEL_EMPTY || (flags & (kSlotWhole | kSlotPromoted)))
		return;
	if(b.blk_slot[slot].y == 0)
		return;
	const uint32_t nw = (flags & kSlotPresorted) ? b.sorted_pool[b.blk_sorted[slot]] : 1u;
	if((uint32_t)wave >= nw)
		return;
	const int bin = slot >> 4, blk = slot & 15, by = blk >> 2, bx = blk & 3;
	const int px = (bin % c.bin_count_x) * kBinSize + bx * 8 + (lane & 7);
	const int py = (bin / c.bin_count_x) * kBinSize + by * 8 + (lane >> 3);
	const size_t r = ((size_t)g.range_base[slot] + wave) * 64 + lane;
	const BwdRecord rc = g.rec[r];
	const uint32_t pf = (px < c.width && py < c.height) ? g.pix_flags[(size_t)py * c.width + px] : 0u;
	float gsel[3] = {0.0f, 0.0f, 0.0f};
	if(pf & 8u) {
		const float4 gi = g.grad_image[(size_t)py * c.width + px];
		const float gv[3] = {gi.x, gi.y, gi.z};
#pragma unroll
		for(int k = 0; k < 3; k++)
			gsel[k] = ((pf >> k) & 1u) ? gv[k] : 0.0f;
	}
	BwdStart st;
	st.t = rc.t;
	st.q = 0.0;
#pragma unroll
	for(int k = 0; k < 3; k++)
		st.q += (double)gsel[k] * rc.d[k];
	st.gr = gsel[0], st.gg = gsel[1], st.gb = gsel[2];
	st.pad = 0.0f;
	g.start[r] = st;
}

constexpr int kGradStride = kGradWords + 1; // odd stride against bank conflicts

// One wave per (block, depth range); single-wave work-groups (no LDS is shared between
// waves), so that more of them fit on a CU.
// MODE: kShadePlain or kShadeGeneral.
template <int MODE>
__global__ __launch_bounds__(64) void bwd_pass_b_kernel(FrameConst c, FrameBufs b, BwdBufs g) {
	if((b.ctrl[kCtrlOverflow] & kOvfBinLists) || !bwd_fits(b, g))
		return;
	__shared__ uint4 s_rec[kSliceEntries * kRecQuads];
	__shared__ unsigned long long s_grad[kSliceEntries * kGradStride];
	const int lane = lane_id();
	const uint32_t slot = blockIdx.x / kBigWaves;
	const int wave = (int)(blockIdx.x % kBigWaves);
	const uint32_t flags = b.blk_flags[slot];
	const uint32_t level = flags & kSlotLevelMask;
	if(level == LUCID_BIN_LEVEL_EMPTY || (flags & (kSlotWhole | kSlotPromoted)))
		return;
	const uint2 sl = b.blk_slot[slot];
	if(sl.y == 0)
		return;
	if(!(flags & kSlotPresorted) && wave != 0)
		return;
	if(flags & kSlotPresorted) {
		const uint32_t nw = b.sorted_pool[b.blk_sorted[slot]];
		if((uint32_t)wave >= nw)
			return;
	}
	const int bin = slot >> 4, blk = slot & 15, by = blk >> 2, bx = blk & 3;
	const int px = (bin % c.bin_count_x) * kBinSize + bx * 8 + (lane & 7);
	const int py = (bin / c.bin_count_x) * kBinSize + by * 8 + (lane >> 3);
	const float fx = (float)px, fy = (float)py;
	// The block's triangles in depth order: the pre-sorted pool, or the lane's entries of a register
	// sort. (Kept in LDS, as pass A has them, they took 3 of the wave's 16 KB, and the kernel is
	// short of waves: 10 per CU instead of 12.)
	const uint32_t *sorted = nullptr;
	uint32_t e0 = 0, e1 = sl.y, tri_all[4] = {0u, 0u, 0u, 0u};
	if(flags & kSlotPresorted) {
		const uint32_t *hdr = b.sorted_pool + b.blk_sorted[slot];
		sorted = hdr + kSortedHeader;
		e0 = hdr[1 + wave], e1 = hdr[2 + wave];
	} else {
		uint64_t *s_msk = reinterpret_cast<uint64_t *>(s_rec);
		uint32_t *s_tri = reinterpret_cast<uint32_t *>(s_msk + kRegSortCap);
		static_assert(sizeof(s_rec) >= kRegSortCap * 12, "the sort's ids and masks fit the staging area");
		uint32_t pos[4];
		sort_block_positions(b.blk_lists + sl.x, sl.y, pos, s_msk, s_tri);
		wave_sync_lds();
#pragma unroll
		for(int j = 0; j < 4; j++)
			if(j * 64 + lane < (int)sl.y)
				tri_all[j] = s_tri[pos[j]];
		wave_sync_lds(); // read before the first slice is staged over them
	}
	const uint32_t row0 = g.row_base[slot];
	const BwdStart st = g.start[((size_t)g.range_base[slot] + wave) * 64 + lane];
	double t = st.t, q = st.q;
	const bool live = st.gr != 0.0f || st.gg != 0.0f || st.gb != 0.0f;
	const int fix_k = grad_fixed_exp(c, bits2f(b.ctrl[kCtrlBwdGradMax]));
	const double fix_scale = ldexp(1.0, fix_k);
	// the lane's slots of the ten components: component k of the rotated order is added at kk[k]
	const bool rot1 = (lane & 1) != 0, rot2 = (lane & 2) != 0, rot4 = (lane & 4) != 0;
	const int rot = (rot1 ? 3 : 0) + (rot2 ? 5 : 0) + (rot4 ? 1 : 0);
	static_assert(kSliceEntries == 64, "a lane stages one entry of a slice");
	for(uint32_t s0 = e0; s0 < e1; s0 += kSliceEntries) {
		const uint32_t n = min(e1 - s0, (uint32_t)kSliceEntries);
		uint32_t tri[1] = {0u};
		if(sorted) {
			if((uint32_t)lane < n)
				tri[0] = sorted[s0 + lane];
		} else {
#pragma unroll
			for(uint32_t j = 0; j < 4; j++)
				tri[0] = s0 == j * 64 ? tri_all[j] : tri[0];
		}
		stage_slice<kSliceWords, MODE>(c, b, tri, n, s_rec);
		for(int i = lane; i < kSliceEntries * kGradStride; i += 64)
			s_grad[i] = 0ull;
		wave_sync_lds();
		// replay the order recorded by pass A (byte j of this lane at seq[64 j], read one
		// step ahead; a lane stops at its end marker and reads nothing beyond it). The loop
		// is divergent: each lane leaves at its own end, so its state (t, q) needs no copies.
		const uint8_t *seq = g.seq + seq_index(row0, s0, 0, lane);
		uint8_t next = seq[0];
		for(uint32_t j = 0; j < n && next != kSeqEnd; j++) {
			const uint8_t e = next;
			next = j + 1 < n ? seq[(size_t)(j + 1) * 64] : kSeqEnd;
			const uint4 *rec = s_rec + (uint32_t)e * kRecQuads;
			const float inv = record_inv_depth(rec[0], fx, fy);
			BwdSample smp;
			if constexpr(is_plain(MODE)) {
				const PlainShade p = shade_plain(rec, fx, fy, inv);
				smp.b0 = p.b0, smp.b1 = p.b1;
				smp.r = sat(p.x[0]), smp.g = sat(p.x[1]), smp.b = sat(p.x[2]), smp.a = p.alpha;
				// (recorded samples have an alpha other than 0; the clamp passes the gradient on [0, 1])
				smp.dr = p.x[0] >= 0.0f && p.x[0] <= 1.0f ? 1.0f : 0.0f;
				smp.dg = p.x[1] >= 0.0f && p.x[1] <= 1.0f ? 1.0f : 0.0f;
				smp.db = p.x[2] >= 0.0f && p.x[2] <= 1.0f ? 1.0f : 0.0f;
				smp.da = 1.0f;
			} else {
				shade_grad(c, b, rec, fx, fy, inv, smp);
			}
			float out[kGradWords];
			bwd_fragment(t, q, st.gr, st.gg, st.gb, smp, out);
			if(live) {
				// Lanes add the ten components in eight rotated orders (by pixel column: 0, 3, 5, 8, 1,
				// 4, 6 and 9), so that pixels at the same entry in the same step seldom hit one
				// address (integer sums: the order changes no bit). The rotation is three stages of
				// selects on a lane bit each, as many as one four-way choice per component takes.
				float r1[kGradWords], r2[kGradWords], r3[kGradWords];
				// (by value: a choice between array elements would become one of addresses)
				auto sel = [](bool p, float x, float y) { return p ? x : y; };
#pragma unroll
				for(int k = 0; k < kGradWords; k++)
					r1[k] = sel(rot1, out[(k + 3) % kGradWords], out[k]);
#pragma unroll
				for(int k = 0; k < kGradWords; k++)
					r2[k] = sel(rot2, r1[(k + 5) % kGradWords], r1[k]);
#pragma unroll
				for(int k = 0; k < kGradWords; k++)
					r3[k] = sel(rot4, r2[(k + 1) % kGradWords], r2[k]);
#pragma unroll
				for(int k = 0; k < kGradWords; k++) {
					const int kk0 = k + rot;
					const int kk = kk0 >= kGradWords ? kk0 - kGradWords : kk0;
					atomicAdd(&s_grad[(uint32_t)e * kGradStride + kk], to_fixed(r3[k], fix_scale));
				}
			}
		}
		wave_sync_lds();
		for(uint32_t e = lane; e < n; e += 64) {
			const size_t row = (size_t)row0 + s0 + e;
			if(row < g.rows_cap) {
#pragma unroll
				for(int k = 0; k < kGradWords; k++)
					g.rows[row * kGradWords + k] =
						(float)ldexp((double)(long long)s_grad[e * kGradStride + k], -fix_k);
			}
		}
		wave_sync_lds();
	}
}

// Exclusive scans over the blocks the block kernels process: gradient rows (one per list
// entry) and depth ranges (start states of pass B).
// One thread queues every on-screen pixel of block `slot` for the exact per-pixel path (a
// list too long to pre-sort), as high_finalize does for a new frame.
__device__ void enqueue_block_whole(const FrameConst &c, const FrameBufs &b, uint32_t slot) {
	const int bin = (int)(slot >> 4), blk = (int)(slot & 15);
	const int x0 = (bin % c.bin_count_x) * kBinSize + (blk & 3) * 8;
	const int y0 = (bin / c.bin_count_x) * kBinSize + (blk >> 2) * 8;
	const int w = min(8, c.width - x0), h = min(8, c.height - y0);
	if(w <= 0 || h <= 0)
		return;
	const uint32_t base = atomicAdd(&b.ctrl[kCtrlFallbackCount], (uint32_t)(w * h));
	for(int i = 0; i < w * h; i++) {
		if(base + (uint32_t)i >= b.fallback_cap) {
			atomicOr(&b.ctrl[kCtrlOverflow], kOvfFallback);
			break;
		}
		b.fallback_queue[base + i] =
			make_uint4(slot, (uint32_t)(x0 + i % w), (uint32_t)(y0 + i / w), 1u);
	}
}

// REUSE (a finished frame's lists, reused by the backward): the control words start afresh
// and the exact-fallback queue is rebuilt: the blocks too long to pre-sort are queued here,
// pass A adds the mis-ordered pixels.
template <bool REUSE>
__global__ __launch_bounds__(1024) void grad_row_scan_kernel(FrameConst c, FrameBufs b, BwdBufs g) {
	const uint32_t n = (uint32_t)c.bin_count * 16;
	// Four slots per thread and round, whose loads are in flight together: one work-group's chain of
	// loads and barriers is all this kernel waits for (4096 blocks: 12 -> 9 us).
	constexpr int kSlots = 4;
	__shared__ uint32_t s_wave[2][kSlots * 16];
	__shared__ uint32_t s_carry[2];
	if constexpr(REUSE) {
		if(threadIdx.x < (uint32_t)kCtrlWords)
			b.ctrl[threadIdx.x] = 0u;
	}
	if(threadIdx.x < 2)
		s_carry[threadIdx.x] = 0;
	__syncthreads();
	const int wave = threadIdx.x >> 6, lane = lane_id();
	for(uint32_t base = 0; base < n; base += kSlots * 1024) {
		uint32_t flags[kSlots], m[kSlots], at[kSlots], v[2][kSlots], inc[2][kSlots];
#pragma unroll
		for(int i = 0; i < kSlots; i++) {
			const uint32_t slot = base + i * 1024 + threadIdx.x;
			flags[i] = slot < n ? b.blk_flags[slot] : 0u;
			m[i] = slot < n ? b.blk_slot[slot].y : 0u;
			at[i] = slot < n ? b.blk_sorted[slot] : 0u;
		}
#pragma unroll
		for(int i = 0; i < kSlots; i++) {
			const uint32_t level = flags[i] & kSlotLevelMask;
			const bool live = level != LUCID_BIN_LEVEL_EMPTY && !(flags[i] & (kSlotWhole | kSlotPromoted)) && m[i];
			v[0][i] = live ? m[i] : 0u;
			v[1][i] = !live ? 0u : (flags[i] & kSlotPresorted) ? b.sorted_pool[at[i]] : 1u;
			if(REUSE && (flags[i] & kSlotWhole))
				enqueue_block_whole(c, b, base + i * 1024 + threadIdx.x);
		}
#pragma unroll
		for(int k = 0; k < 2; k++) {
#pragma unroll
			for(int i = 0; i < kSlots; i++) {
				inc[k][i] = wave_inclusive_add(v[k][i]);
				if(lane == 63)
					s_wave[k][i * 16 + wave] = inc[k][i];
			}
		}
		__syncthreads();
		if(wave < 2) { // wave k: the sums before each (slot, wave)
			static_assert(kSlots * 16 == 64, "a lane per sum");
			const uint32_t x = s_wave[wave][lane], ex = wave_inclusive_add(x) - x + s_carry[wave];
			s_wave[wave][lane] = ex;
			if(lane == 63)
				s_carry[wave] = ex + x;
		}
		__syncthreads();
#pragma unroll
		for(int i = 0; i < kSlots; i++) {
			const uint32_t slot = base + i * 1024 + threadIdx.x;
			if(slot < n) {
				g.row_base[slot] = s_wave[0][i * 16 + wave] + inc[0][i] - v[0][i];
				g.range_base[slot] = s_wave[1][i * 16 + wave] + inc[1][i] - v[1][i];
			}
		}
		__syncthreads();
	}
	if(threadIdx.x == 0) {
		b.ctrl[kCtrlBwdRows] = s_carry[0];
		b.ctrl[kCtrlBwdRanges] = s_carry[1];
		b.ctrl[kCtrlBwdExtra] = 0;
		b.ctrl[kCtrlBwdGradMax] = 0;
	}
}

// max |dL/dpixel| (rgb) over the image into kCtrlBwdGradMax (after the row scan cleared it):
// fixes the frame's gradient fixed-point scale.
__global__ __launch_bounds__(256) void grad_max_kernel(FrameConst c, BwdBufs g, uint32_t *ctrl) {
	const uint32_t n = (uint32_t)c.width * (uint32_t)c.height;
	float gm = 0.0f;
	for(uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
		const float4 v = g.grad_image[i];
		gm = fmaxf(gm, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fabsf(v.z)));
	}
#pragma unroll
	for(int d = 1; d < 64; d <<= 1)
		gm = fmaxf(gm, __shfl_xor(gm, d, 64));
	if(lane_id() == 0 && gm > 0.0f)
		atomicMax(&ctrl[kCtrlBwdGradMax], f2bits(gm)); // non-negative floats order as uints
}

// Exact adjoint of one queued pixel: its fragments sorted exactly (as fallback_pixel), then
// both passes over the sorted list; one gradient row per fragment, appended after the
// block rows.
__device__ void bwd_fallback_pixel(const FrameConst &c, const FrameBufs &b, const BwdBufs &g,
								   uint4 item, uint64_t *s_keys) {
	const int lane = lane_id();
	const uint32_t slot = item.x;
	const int px = (int)item.y, py = (int)item.z;
	const uint2 sl = b.blk_slot[slot];
	const uint4 *list = b.blk_lists + sl.x;
	const uint32_t m = sl.y;
	const int bit = (py & 7) * 8 + (px & 7);
	const float fx = (float)px, fy = (float)py;
	const uint32_t n =
		gather_pixel_keys(b, list, m, bit, fx, fy, s_keys, kFallbackCap, false);
	const uint64_t *keys = s_keys;
	bool global_keys = false;
	if(n <= (uint32_t)kFallbackCap) {
		sort_pixel_keys(s_keys, n);
	} else {
		const uint32_t P = next_pow2(n);
		uint32_t off = 0;
		if(lane == 0) {
			off = (uint32_t)atomicAdd(&b.ctrl[kCtrlSpillCursor], P);
			if((uint64_t)off + P > b.spill_cap) {
				atomicOr(&b.ctrl[kCtrlOverflow], kOvfSpill);
				off = 0xffffffffu;
			}
		}
		off = wave_read(off, 0);
		if(off == 0xffffffffu)
			return;
		uint64_t *gk = b.spill + off;
		gather_pixel_keys(b, list, m, bit, fx, fy, gk, P, true);
		for(uint32_t i = n + lane; i < P; i += 64)
			__hip_atomic_store(&gk[i], ~0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		__threadfence();
		__builtin_amdgcn_wave_barrier();
		bitonic_global_wave(gk, P);
		keys = gk;
		global_keys = true;
	}
	auto key_at = [&](uint32_t i) -> uint64_t {
		return global_keys ? __hip_atomic_load(&keys[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
						   : keys[i];
	};
	auto shade_at = [&](uint32_t i, BwdSample &smp) -> bool {
		const uint32_t t = (uint32_t)key_at(i);
		uint4 q[kRecQuads];
		load_shading_record(b, t, q);
		return shade_grad(c, b, q, fx, fy, record_inv_depth(q[0], fx, fy), smp);
	};
	// pass A (serial over the sorted list, 64 samples shaded at a time)
	BwdTotals tot;
	tot.init();
	for(uint32_t base = 0; base < n; base += 64) {
		BwdSample smp;
		smp.zero();
		const bool ok = base + lane < n && shade_at(base + lane, smp);
		const uint32_t cnt = min(64u, n - base);
		for(uint32_t j = 0; j < cnt; j++) {
			BwdSample s;
			s.r = wave_read(smp.r, (int)j), s.g = wave_read(smp.g, (int)j);
			s.b = wave_read(smp.b, (int)j), s.a = wave_read(smp.a, (int)j);
			if(wave_read((uint32_t)ok, (int)j))
				tot.add(s.r, s.g, s.b, s.a);
		}
	}
	const float bg[3] = {c.background[0], c.background[1], c.background[2]};
	const float o32[3] = {tot.acc.cr + tot.acc.tr * bg[0], tot.acc.cg + tot.acc.tr * bg[1],
						  tot.acc.cb + tot.acc.tr * bg[2]};
	const float4 gi = g.grad_image[(size_t)py * c.width + px];
	const float gv[3] = {gi.x, gi.y, gi.z};
	float gsel[3];
#pragma unroll
	for(int k = 0; k < 3; k++)
		gsel[k] = (o32[k] >= 0.0f && o32[k] <= 1.0f) ? gv[k] : 0.0f;
	// pass B: rows [base_row, base_row + n)
	uint32_t base_row = 0;
	if(lane == 0) {
		base_row = atomicAdd(&b.ctrl[kCtrlBwdExtra], n);
		if((uint64_t)b.ctrl[kCtrlBwdRows] + base_row + n > g.rows_cap) {
			atomicOr(&b.ctrl[kCtrlOverflow], kOvfGradRows);
			base_row = 0xffffffffu;
		}
	}
	base_row = wave_read(base_row, 0);
	if(base_row == 0xffffffffu)
		return;
	const size_t row0 = (size_t)b.ctrl[kCtrlBwdRows] + base_row;
	double t = 1.0;
	double q = (double)gsel[0] * (tot.cr + tot.t * (double)bg[0]) +
			   (double)gsel[1] * (tot.cg + tot.t * (double)bg[1]) +
			   (double)gsel[2] * (tot.cb + tot.t * (double)bg[2]);
	for(uint32_t base = 0; base < n; base += 64) {
		BwdSample smp;
		smp.zero();
		const bool ok = base + lane < n && shade_at(base + lane, smp);
		const uint32_t cnt = min(64u, n - base);
		float mine[kGradWords];
#pragma unroll
		for(int k = 0; k < kGradWords; k++)
			mine[k] = 0.0f;
		for(uint32_t j = 0; j < cnt; j++) {
			BwdSample s;
			s.r = wave_read(smp.r, (int)j), s.g = wave_read(smp.g, (int)j);
			s.b = wave_read(smp.b, (int)j), s.a = wave_read(smp.a, (int)j);
			s.b0 = wave_read(smp.b0, (int)j), s.b1 = wave_read(smp.b1, (int)j);
			s.dr = wave_read(smp.dr, (int)j), s.dg = wave_read(smp.dg, (int)j);
			s.db = wave_read(smp.db, (int)j), s.da = wave_read(smp.da, (int)j);
			if(wave_read((uint32_t)ok, (int)j)) {
				float out[kGradWords];
				bwd_fragment(t, q, gsel[0], gsel[1], gsel[2], s, out);
				if((uint32_t)lane == j) {
#pragma unroll
					for(int k = 0; k < kGradWords; k++)
						mine[k] = out[k];
				}
			}
		}
		if(base + lane < n) {
			const size_t r = row0 + base + lane;
			g.row_tri[r] = (uint32_t)key_at(base + lane);
#pragma unroll
			for(int k = 0; k < kGradWords; k++)
				g.rows[r * kGradWords + k] = mine[k];
		}
	}
}

__global__ __launch_bounds__(kFallbackThreads) void bwd_fallback_kernel(FrameConst c, FrameBufs b,
																		 BwdBufs g) {
	__shared__ uint64_t s_keys[kFallbackThreads / 64][kFallbackCap];
	if((b.ctrl[kCtrlOverflow] & kOvfBinLists) || !bwd_fits(b, g))
		return;
	const uint32_t nq = min(b.ctrl[kCtrlFallbackCount], b.fallback_cap);
	const uint32_t waves = gridDim.x * (kFallbackThreads / 64);
	const uint32_t w = blockIdx.x * (kFallbackThreads / 64) + (threadIdx.x >> 6);
	for(uint32_t qi = w; qi < nq; qi += waves)
		bwd_fallback_pixel(c, b, g, b.fallback_queue[qi], s_keys[threadIdx.x >> 6]);
}

// Row generation of small frames in one launch, where two would each end with a nearly empty chip
// (767 x 431 particles 33 + gap -> 24 us, 1280 x 720 lit mesh 49 + gap -> 44); large ones fill it
// and do better apart, with the high bins' smaller groups (1440p mesh 310 us apart, 350 in one
// launch). The line: whole frames of the same scene kinds at ten sizes, one launch against two, us.
//   bins                    520   1024   1435   2040   2800   3600
//   clustered triangles    +4.6   -3.7   -3.3  -13.7  -24.5  +14.6
//   byte-coloured ones     -7.6  -11.4   -6.4   -3.8   +3.7   +8.4
//   fp32 samples           -6.7  -11.2   -7.7   -3.2   +2.7   +8.7
//   384 spheres            -5.3   -3.5   -2.0   -1.6   -0.6   +1.8
//   20 k small triangles   -1.5   -0.3   +1.3   -0.1   +1.0   +1.6
// So the kinds part between 1400 and 3600 bins; up to 1024 one launch is not worse but for +5 of
// 300 us at one size. Timed frames take two launches at every size, with `after_low` (if not null)
// recorded between them.
constexpr int kFusedRowgenBins = 1024;
static void launch_rowgen(const FrameConst &c, const FrameBufs &b, hipStream_t stream,
						  hipEvent_t *after_low = nullptr) {
	constexpr int kHigh = kRowgenSplitThreads / kRowgenThreads, kHighFused = kRowgenSplitThreads / kRowgenLowThreads;
	if(c.bin_count <= kFusedRowgenBins && !after_low) {
		hipLaunchKernelGGL(rowgen_fused_kernel, dim3(c.bin_count * (kHighFused + 1)), dim3(kRowgenLowThreads),
						   0, stream, c, b);
		return;
	}
	hipLaunchKernelGGL(rowgen_low_kernel, dim3(c.bin_count), dim3(kRowgenLowThreads), 0, stream, c, b);
	if(after_low)
		(void)hipEventRecord(*after_low, stream);
	hipLaunchKernelGGL(rowgen_high_kernel, dim3(c.bin_count * kHigh), dim3(kRowgenThreads), 0, stream, c, b);
}

// Block bookkeeping and the pre-sort of long lists (up to kMidSortCap entries), then the
// queued lists longer than that (one work-group per CU).
static void launch_high_finalize(const FrameConst &c, const FrameBufs &b, hipStream_t stream) {
	hipLaunchKernelGGL(high_finalize_kernel, dim3(c.bin_count * 16), dim3(kSortThreads), 0, stream,
					   c, b);
	hipLaunchKernelGGL(high_finalize_long_kernel, dim3(256), dim3(kSortThreads), 0, stream, c, b);
}

// Calls f with the sample format and shading mode as compile-time constants.
template <class F> static void with_shade_mode(bool fp32, int mode, F &&f) {
	const std::integral_constant<int, kShadeGeneral> general;
	const std::integral_constant<int, kShadeTextured> textured;
	const std::integral_constant<int, kShadePlain> plain;
	const std::integral_constant<int, kShadeFlat> flat;
	const std::integral_constant<int, kShadeFlat | kShadeNarrow> flat_narrow;
	const std::true_type f32;
	const std::false_type bytes;
	if(fp32)
		mode == kShadePlain ? f(f32, plain) : is_textured(mode) ? f(f32, textured) : f(f32, general);
	else if(is_flat(mode))
		mode & kShadeNarrow ? f(bytes, flat_narrow) : f(bytes, flat);
	else
		is_textured(mode) ? f(bytes, textured) : f(bytes, general);
}

template <bool FP32, int W, int MODE>
static void launch_block_raster_apart(const FrameConst &c, const FrameBufs &b, hipStream_t stream) {
	hipLaunchKernelGGL((block_raster_kernel<FP32, W, MODE>), dim3(c.bin_count * 16), dim3(64), 0, stream,
					   c, b);
	hipLaunchKernelGGL((block_raster_big_kernel<FP32, W, MODE>), dim3(c.bin_count * 16),
					   dim3(kBigWaves * 64), 0, stream, c, b);
}

// Small frames take one launch (two -> one: 767 x 431 particles, 336 bins, 79 -> 64 us; 1280 x 720
// lit mesh, 920 bins, 104 -> 99 us; 512 x 512 preview, 18 -> 15 us). Large ones fill the chip either
// way, and the register-sorted blocks are better off as work-groups of their own (1440p mesh, 3600
// bins, 336 -> 365 us), as are textured ones, whose blocks differ most in length (768 bins, 261 ->
// 269 us). The line: whole frames as above, one launch against two, us.
//   bins                    520   1024   1435   1750   2040   2800
//   clustered triangles   -25.4  -29.5  -25.5  -15.9  -11.0   -5.6
//   byte-coloured ones    -28.2  -17.0   -1.4   +4.9  +14.1  +24.7
//   fp32 samples          -23.3  -12.8   -4.0   -0.3   +2.7   +9.9
//   384 spheres            -7.1   -5.5   -4.1   -2.3   -0.6   +2.4
//   20 k small triangles   -1.0   -0.5   -0.9   -0.6   -0.6   -0.1
// The first kind turns between 1435 and 1750 bins, the last beyond 2800; up to 1024 all gain.
constexpr int kFusedRasterBins = 1024;
template <bool FP32, int MODE>
static void launch_block_raster(const FrameConst &c, const FrameBufs &b, hipStream_t stream) {
	if constexpr(!is_textured(MODE)) {
		if(c.slice_words == 1 && c.bin_count <= kFusedRasterBins) {
			hipLaunchKernelGGL((block_raster_fused_kernel<FP32, MODE>),
							   dim3(c.bin_count * (16 + 16 / kBigWaves)), dim3(kBigWaves * 64), 0, stream,
							   c, b);
			return;
		}
	}
	if(c.slice_words == 2)
		launch_block_raster_apart<FP32, 2, MODE>(c, b, stream);
	else
		launch_block_raster_apart<FP32, 1, MODE>(c, b, stream);
}

template <bool FP32, int MODE>
static void launch_raster_t(const FrameConst &c, const FrameBufs &b, hipStream_t stream,
							hipEvent_t *ev) {
	constexpr bool TEX = is_textured(MODE);
	launch_rowgen(c, b, stream, ev); // (ev[0] between low and high bins)
	launch_high_finalize(c, b, stream);
	if(ev)
		(void)hipEventRecord(ev[1], stream);
	launch_block_raster<FP32, MODE>(c, b, stream);
	if(ev)
		(void)hipEventRecord(ev[2], stream);
	hipLaunchKernelGGL((fallback_kernel<FP32, TEX>), dim3(1024), dim3(kFallbackThreads), 0, stream,
					   c, b);
	if(ev)
		(void)hipEventRecord(ev[3], stream);
}

template <bool FP32, int W, int MODE>
static void launch_raster_batch_t(const BatchPlan &p, hipStream_t stream) {
	constexpr bool TEX = is_textured(MODE);
	hipLaunchKernelGGL(rowgen_low_kernel_batch, dim3(p.total[kBsRowgenLow]), dim3(kRowgenThreads), 0,
					   stream, p.frames, p.stage_pre(kBsRowgenLow), p.num_frames);
	hipLaunchKernelGGL(rowgen_high_kernel_batch, dim3(p.total[kBsRowgenHigh]), dim3(kRowgenThreads), 0,
					   stream, p.frames, p.stage_pre(kBsRowgenHigh), p.num_frames);
	hipLaunchKernelGGL(high_finalize_kernel_batch, dim3(p.total[kBsHighFinalize]),
					   dim3(kSortThreads), 0, stream, p.frames, p.stage_pre(kBsHighFinalize), p.num_frames);
	hipLaunchKernelGGL(high_finalize_long_kernel_batch, dim3(p.total[kBsHighFinalizeLong]),
					   dim3(kSortThreads), 0, stream, p.frames, p.stage_pre(kBsHighFinalizeLong),
					   p.num_frames);
	hipLaunchKernelGGL((block_raster_kernel_batch<FP32, W, MODE>), dim3(p.total[kBsBlockRaster]),
					   dim3(64), 0, stream, p.frames, p.stage_pre(kBsBlockRaster), p.num_frames);
	hipLaunchKernelGGL((block_raster_big_kernel_batch<FP32, W, MODE>),
					   dim3(p.total[kBsBlockRasterBig]), dim3(kBigWaves * 64), 0, stream,
					   p.frames, p.stage_pre(kBsBlockRasterBig), p.num_frames);
	hipLaunchKernelGGL((fallback_kernel_batch<FP32, TEX>), dim3(p.total[kBsFallback]),
					   dim3(kFallbackThreads), 0, stream, p.frames, p.stage_pre(kBsFallback), p.num_frames);
}

// Row generation, sorting, block rasterisation and the exact fallback of every frame of a
// batch: one launch per stage, kernels chosen by the batch's sample format, slice width and
// shading mode.
template <int W>
static void launch_raster_batch_w(const BatchPlan &p, hipStream_t stream) {
	with_shade_mode(p.fp32, p.mode, [&](auto fp32, auto mode) {
		launch_raster_batch_t<decltype(fp32)::value, W, decltype(mode)::value>(p, stream);
	});
}

hipError_t launch_raster_batch(const BatchPlan &p, hipStream_t stream) {
	if(p.slice_words == 2)
		launch_raster_batch_w<2>(p, stream);
	else
		launch_raster_batch_w<1>(p, stream);
	return hipGetLastError();
}

// events (optional, 4): after the row generation of low bins, after that of high bins and the
// sorting of long block lists, after block rasterisation, after the fallback kernel.
hipError_t launch_raster(const FrameConst &c, const FrameBufs &b, hipStream_t stream,
						 hipEvent_t *events) {
	// frames with albedo textures take kernels built with the texture path (the others carry
	// none of its code or registers); flat-colour frames take the colour-plane records
	with_shade_mode((c.opts & LUCID_OPT_FP32_SAMPLES) != 0, frame_shade_mode(c), [&](auto fp32, auto mode) {
		launch_raster_t<decltype(fp32)::value, decltype(mode)::value>(c, b, stream, events);
	});
	return hipGetLastError();
}

// Backward, first part: the forward's row generation and block sorting (fragment lists are
// recomputed, not stored), then the gradient row allocation.
hipError_t launch_backward_prepare(const FrameConst &c, const FrameBufs &b, const BwdBufs &g,
								   hipStream_t stream) {
	launch_rowgen(c, b, stream);
	launch_high_finalize(c, b, stream);
	hipLaunchKernelGGL(grad_row_scan_kernel<false>, dim3(1), dim3(1024), 0, stream, c, b, g);
	return hipGetLastError();
}

// max |dL/dpixel| for the gradient scale (pass B and the triangle sums read it); it may run
// on a helper stream once the row scan (which clears it) has run.
hipError_t launch_grad_max(const FrameConst &c, const BwdBufs &g, uint32_t *ctrl,
						   hipStream_t stream) {
	hipLaunchKernelGGL(grad_max_kernel, dim3(256), dim3(256), 0, stream, c, g, ctrl);
	return hipGetLastError();
}

// A frame recording the backward's pass A does so only if its gradient rows, recorded
// order and start states fit the buffers (sized by an earlier frame); otherwise the block
// rasterisers render it and the host grows the buffers from the row scan's counts.
__global__ __launch_bounds__(64) void record_gate_kernel(FrameBufs b, BwdBufs g) {
	if(threadIdx.x == 0)
		b.ctrl[kCtrlRecorded] = (!(b.ctrl[kCtrlOverflow] & kOvfBinLists) && bwd_fits(b, g)) ? 1u : 0u;
}

template <bool RECORD>
static void launch_pass_a(const FrameConst &c, const FrameBufs &b, const BwdBufs &g, hipStream_t stream) {
	auto go = [&](auto kernel) {
		hipLaunchKernelGGL(kernel, dim3(c.bin_count * 16), dim3(kBigWaves * 64), 0, stream, c, b, g);
	};
	if(c.window == 1) // narrow-window tuning: two slots
		c.plain_colors ? go(bwd_pass_a_kernel<RECORD, 2, kShadePlain>)
					   : go(bwd_pass_a_kernel<RECORD, 2, kShadeGeneral>);
	else
		c.plain_colors ? go(bwd_pass_a_kernel<RECORD, kWindow, kShadePlain>)
					   : go(bwd_pass_a_kernel<RECORD, kWindow, kShadeGeneral>);
}

// Forward frame that also records pass A (fp32 samples): the raster stage of launch_raster
// with the gradient row scan, the gate and the recording pass before the block kernels
// (which then render only what the recording pass does not).
hipError_t launch_raster_recording(const FrameConst &c, const FrameBufs &b, const BwdBufs &g,
								   hipStream_t stream, hipEvent_t *ev) {
	launch_rowgen(c, b, stream, ev); // (ev[0] between low and high bins)
	launch_high_finalize(c, b, stream);
	hipLaunchKernelGGL(grad_row_scan_kernel<false>, dim3(1), dim3(1024), 0, stream, c, b, g);
	hipLaunchKernelGGL(record_gate_kernel, dim3(1), dim3(64), 0, stream, b, g);
	if(ev)
		(void)hipEventRecord(ev[1], stream);
	launch_pass_a<true>(c, b, g, stream);
	with_shade_mode(true, frame_shade_mode(c), [&](auto, auto mode) {
		if constexpr(!is_textured(decltype(mode)::value) && !is_flat(decltype(mode)::value))
			launch_block_raster<true, decltype(mode)::value>(c, b, stream);
	});
	if(ev)
		(void)hipEventRecord(ev[2], stream);
	hipLaunchKernelGGL((fallback_kernel<true, false>), dim3(1024), dim3(kFallbackThreads), 0, stream,
					   c, b);
	if(ev)
		(void)hipEventRecord(ev[3], stream);
	return hipGetLastError();
}

// Backward of a frame that recorded pass A: fresh backward control words (the frame's row
// scan results and exact-fallback queue stay), then the start states and the exact
// per-pixel adjoints.
__global__ __launch_bounds__(64) void recorded_begin_kernel(uint32_t *ctrl) {
	if(threadIdx.x == 0) {
		ctrl[kCtrlOverflow] = 0;
		ctrl[kCtrlSpillCursor] = 0;
		ctrl[kCtrlBwdExtra] = 0;
		ctrl[kCtrlBwdGradMax] = 0;
		ctrl[kCtrlTopoChanged] = 0;
	}
}

hipError_t launch_backward_recorded(const FrameConst &c, const FrameBufs &b, const BwdBufs &g,
									hipStream_t stream) {
	hipLaunchKernelGGL(recorded_begin_kernel, dim3(1), dim3(64), 0, stream, b.ctrl);
	return hipGetLastError();
}

hipError_t launch_backward_recorded_order(const FrameConst &c, const FrameBufs &b,
										  const BwdBufs &g, hipStream_t stream) {
	hipLaunchKernelGGL(bwd_start_kernel, dim3(c.bin_count * 16), dim3(kBigWaves * 64), 0, stream, c,
					   b, g);
	hipLaunchKernelGGL(bwd_fallback_kernel, dim3(1024), dim3(kFallbackThreads), 0, stream, c, b, g);
	return hipGetLastError();
}

// Backward, first part when the last finished frame's setup, bins and block lists are
// reused: fresh control words, the exact-pixel queue of the too-long blocks and the
// gradient row allocation, in one kernel.
hipError_t launch_backward_reuse(const FrameConst &c, const FrameBufs &b, const BwdBufs &g,
								 hipStream_t stream) {
	hipLaunchKernelGGL(grad_row_scan_kernel<true>, dim3(1), dim3(1024), 0, stream, c, b, g);
	return hipGetLastError();
}

// Backward, second part: the recorded blend order and start states (pass A, which also
// fills the triangle of every block gradient row), then the exact per-pixel adjoints (their
// rows follow the block rows). After these every row's triangle is known.
hipError_t launch_backward_order(const FrameConst &c, const FrameBufs &b, const BwdBufs &g,
								 hipStream_t stream) {
	launch_pass_a<false>(c, b, g, stream);
	hipLaunchKernelGGL(bwd_fallback_kernel, dim3(1024), dim3(kFallbackThreads), 0, stream, c, b, g);
	return hipGetLastError();
}

// Backward, third part: the block gradient rows (pass B replays the recorded order).
hipError_t launch_backward_rows(const FrameConst &c, const FrameBufs &b, const BwdBufs &g,
								hipStream_t stream) {
	if(c.plain_colors)
		hipLaunchKernelGGL(bwd_pass_b_kernel<kShadePlain>, dim3(c.bin_count * 16 * kBigWaves), dim3(64), 0,
						   stream, c, b, g);
	else
		hipLaunchKernelGGL(bwd_pass_b_kernel<kShadeGeneral>, dim3(c.bin_count * 16 * kBigWaves), dim3(64), 0,
						   stream, c, b, g);
	return hipGetLastError();
}

} // namespace lucid

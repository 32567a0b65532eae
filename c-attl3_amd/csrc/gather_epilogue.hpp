/*
 * gather_epilogue.hpp — what the gathered GEMMs do with a finished tile besides storing it (Epilogue, EPI_*): activation,
 * activation and pooling, moments of the columns.
 */
#ifndef CATTLE_HIP_GATHER_EPILOGUE_HPP_
#define CATTLE_HIP_GATHER_EPILOGUE_HPP_

#include "act_math.hpp"
#include "gemm_tiles.hpp"

#include <limits>

namespace cattle_hip {

/* Sum of v over a group of TL consecutive lanes (TL = 16: a row of the wavefront; TL = 32: two rows) with data-parallel
 * primitives of the vector ALU - lane exchanges inside quads, mirrored halves of a row, the last lane of a row broadcast to
 * the next row - so that no step goes through the LDS crossbar, which the wavefronts of a CU share (a butterfly of
 * ds_bpermute over the 64 column sums of a lane was most of the moments epilogue's time). The total is valid in the
 * last lane of the group (for TL = 16 in all of them). */
template<int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_move(float v) {
	return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, false));
}
template<int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_move(double v) {
	const long long bits = __builtin_bit_cast(long long, v);
	const int lo = __builtin_amdgcn_update_dpp(0, (int) (bits & 0xffffffffll), CTRL, ROW_MASK, 0xF, false);
	const int hi = __builtin_amdgcn_update_dpp(0, (int) (bits >> 32), CTRL, ROW_MASK, 0xF, false);
	return __builtin_bit_cast(double, ((long long) hi << 32) | (long long) (unsigned) lo);
}
template<typename T, int TL>
__device__ __forceinline__ T lane_group_sum(T v) {
	static_assert(TL == 16 || TL == 32, "a row or two rows of the wavefront");
	v += dpp_move<0xB1, 0xF>(v);            /* quad_perm [1, 0, 3, 2] */
	v += dpp_move<0x4E, 0xF>(v);            /* quad_perm [2, 3, 0, 1] */
	v += dpp_move<0x141, 0xF>(v);           /* row_half_mirror */
	v += dpp_move<0x140, 0xF>(v);           /* row_mirror */
	if constexpr (TL == 32)
		v += dpp_move<0x142, 0xA>(v);       /* row_bcast:15 into rows 1 and 3 (the other rows receive zero) */
	return v;
}

/* D rows are filters (row rr of block i is filter FB*rr + i), D columns are m (column lc of block j is row MB*lc + j of the
 * tile), so a lane owns MB adjacent outputs. `stage`: STAGE elements of LDS that the block is done with; bias_s: the tile's
 * bias values; mm: the lane's first row of M; vec_out: whether its rows may be stored as vectors. Returns whether the tile is stored; false (EPI_NONE, EPI_STATS): that is left to the caller. */
template<typename T, int WAVES_M, int WAVES_F, int WT_M, int WT_F, int VEC, int EPI, int STAGE>
__device__ __forceinline__ bool gather_epilogue(typename Mfma<T>::acc_t (&acc)[WT_F / Mfma<T>::TL][WT_M / Mfma<T>::TL], const GatherGeom& g,
		const GatherLaunch& L, const Epilogue<T>& E, T* __restrict__ out, const T* bias_s, T* const stage, int tile, int f0, int mm, bool vec_out) {
	typedef Mfma<T> MF;
	constexpr int THREADS = 64 * WAVES_M * WAVES_F, BM = WAVES_M * WT_M, BF = WAVES_F * WT_F, TL = MF::TL;
	constexpr int MB = WT_M / TL, FB = WT_F / TL, VS = MB * (int) sizeof(T) > 16 ? 16 / (int) sizeof(T) : MB;
	const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
	const int wm = wave % WAVES_M, wf = wave / WAVES_M, lc = lane % TL, lk = lane / TL;
	const int sb_shift = EPI == EPI_POOL ? L.sb_shift : 5;
	if constexpr (EPI == EPI_POOL) {
		/* Pre-activation values of a group of output columns go through LDS (the operand buffers are free now), so
		 * that the threads can be dealt out over (column, window, sample): a window's positions lie in different
		 * lanes and waves. A pass stages, for one accumulator block i, the RG accumulator rows of group q of every
		 * wave: FP = WAVES_F * RG columns x BM rows, as many as the buffers hold (every barrier between passes is a
		 * stall of the whole block). */
		constexpr int LROW = BM + 4, ROOM = STAGE / (WAVES_F * LROW), RG_MIN = std::is_same<T, float>::value ? 8 : 4;
		constexpr int RG = ROOM >= TL ? TL : ROOM >= TL / 2 ? TL / 2 : RG_MIN, GROUPS = TL / RG, FP = WAVES_F * RG;
		constexpr int REGS_PER_GROUP = MF::NACC / GROUPS;
		static_assert(FP * LROW <= STAGE, "the staging tile of the pooling epilogue reuses the A operand buffers");
		const int SB = 1 << sb_shift, P = BM >> sb_shift, pa = P / L.pos_b;
		const int W = P / (E.prh * E.prw), wa_n = pa / E.prh;
		const int strip = tile / L.tile_rows, trow = tile - strip * L.tile_rows;
		const int ab = trow / L.sample_blocks, nb = trow - ab * L.sample_blocks;
		const int a_p0 = ab * wa_n, b_p0 = strip * (L.pos_b / E.prw);
		/* What an output's place asks of index arithmetic: the window's first value in a staged column, and the element
		 * offsets of column 0 in the pooled tensors, the arg-max cache and the full-size tensor. */
		struct Spot {
			int col;
			size_t pooled, ind, full;
		};
		const auto spot = [&](int s_i, int w) {
			const int wb = w / wa_n, wa = w - wb * wa_n;
			const int n = (nb << sb_shift) + s_i, a_p = a_p0 + wa, b_p = b_p0 + wb;
			return Spot { s_i + (((wa * E.prh) + pa * (wb * E.prw)) << sb_shift), (size_t) n + (size_t) g.N * (a_p + (size_t) E.OHp * b_p),
					((size_t) b_p * E.OHp + a_p) * ((size_t) g.F * g.N) + n,
					(size_t) n + (size_t) g.N * (a_p * E.prh + (size_t) g.OA * (b_p * E.prw)) };
		};
		/* The threads walk (samples, window, column), samples first and PV of them (one 16-byte access) per thread. When
		 * the windows of a pass divide the threads of a sample block evenly, a thread keeps its samples and window through
		 * every pass and only its column moves on. */
		constexpr int PV = VEC, PV_SHIFT = PV == 4 ? 2 : PV == 2 ? 1 : 0;
		const int sbv_shift = sb_shift - PV_SHIFT, SBV = 1 << sbv_shift;          /* the planner keeps SB >= PV */
		const int tps = THREADS >> sbv_shift, outputs = (FP * W * SBV + THREADS - 1) / THREADS;
		const bool fixed_spot = tps % W == 0;
		const int fl0 = (tid >> sbv_shift) / W, fl_step = tps / W;
		Spot sp = spot((tid & (SBV - 1)) << PV_SHIFT, (tid >> sbv_shift) % W);
		const int kstep = pa << sb_shift;
		const bool two_by_two = E.prh == 2 && E.prw == 2;
		const size_t pooled_plane = (size_t) g.N * E.OHp * E.OWp;
		act_dispatch(E.kind, [&](auto kc) {
			constexpr int KIND = decltype(kc)::value;
			#pragma unroll
			for (int i = 0; i < FB; ++i) {
				#pragma unroll
				for (int q = 0; q < GROUPS; ++q) {
					__syncthreads();
					#pragma unroll
					for (int r = 0; r < MF::NACC; ++r) {
						if (r / REGS_PER_GROUP != q)
							continue;
						const int arow = acc_row<T>(r, lk);
						const T bv = bias_s[wf * WT_F + FB * arow + i];
						T v[MB];
						#pragma unroll
						for (int j = 0; j < MB; ++j)
							v[j] = acc[i][j][r] + bv;
						T* dst = stage + (wf * RG + arow - RG * q) * LROW + wm * WT_M + MB * lc;
						#pragma unroll
						for (int j0 = 0; j0 < MB; j0 += VS)
							vec_store<T, VS>(dst + j0, *reinterpret_cast<T (*)[VS]>(&v[j0]));
					}
					__syncthreads();
					for (int pass = 0; pass < outputs; ++pass) {
						int fl;
						if (fixed_spot) {
							fl = fl0 + pass * fl_step;
							if (fl >= FP)
								break;
						} else {
							const int it = tid + pass * THREADS;
							if (it >= FP * W * SBV)
								break;
							const int t2 = it >> sbv_shift;
							fl = t2 / W;
							sp = spot((it & (SBV - 1)) << PV_SHIFT, t2 - fl * W);
						}
						const int f = f0 + (fl / RG) * WT_F + FB * (RG * q + fl % RG) + i;
						if (f >= g.F)
							continue;
						const T* col = stage + fl * LROW + sp.col;
						T zv[PV];
						if (E.pool_mean) {
							/* the mean of the window, summed width-major / height-minor as the layer of its own does
							 * (MeanPoolLayer.hpp:35-41); what the backward pass needs goes out at every position */
							T sum[PV];
							#pragma unroll
							for (int e = 0; e < PV; ++e)
								sum[e] = (T) 0;
							for (int k = 0; k < E.prw; ++k)
								for (int l = 0; l < E.prh; ++l) {
									vec_load<T, PV>(zv, col + k * kstep + l * SB);
									T y[PV];
									#pragma unroll
									for (int e = 0; e < PV; ++e) {
										y[e] = act_f_coded<T, KIND>(zv[e], E.p);
										sum[e] += y[e];
									}
									if (E.pre)
										vec_store_stream<T, PV>(E.pre + (sp.full + (size_t) g.N * (l + (size_t) g.OA * (k + (size_t) g.OB * f))),
												E.keep_input ? zv : y);
								}
							#pragma unroll
							for (int e = 0; e < PV; ++e)
								sum[e] = sum[e] / (T) (E.prh * E.prw);
							vec_store_stream<T, PV>(out + (sp.pooled + pooled_plane * f), sum);
							continue;
						}
						/* strict '>' from lowest(), width-major / height-minor scan (MaxPoolLayer.hpp:45-56) */
						T best[PV], best_pre[PV];
						unsigned bi[PV];
						vec_load<T, PV>(zv, col);
						#pragma unroll
						for (int e = 0; e < PV; ++e) {
							best[e] = std::numeric_limits<T>::lowest();
							best_pre[e] = zv[e];
							bi[e] = 0;
						}
						const auto consider = [&](const T (&z)[PV], unsigned at) {
							#pragma unroll
							for (int e = 0; e < PV; ++e) {
								const T y = act_f_coded<T, KIND>(z[e], E.p);
								if (y > best[e]) {
									best[e] = y;
									best_pre[e] = z[e];
									bi[e] = at;
								}
							}
						};
						if (two_by_two) {
							/* the usual window: its four positions fetched together, then scanned in the same order */
							T z1[PV], z2[PV], z3[PV];
							vec_load<T, PV>(z1, col + SB);
							vec_load<T, PV>(z2, col + kstep);
							vec_load<T, PV>(z3, col + kstep + SB);
							consider(zv, 0u);
							consider(z1, 1u);
							consider(z2, 2u);
							consider(z3, 3u);
						} else {
							for (int k = 0; k < E.prw; ++k)
								for (int l = 0; l < E.prh; ++l) {
									vec_load<T, PV>(zv, col + k * kstep + l * SB);
									consider(zv, (unsigned) (k * E.prh + l));
								}
						}
						vec_store_stream<T, PV>(out + (sp.pooled + pooled_plane * f), best);
						vec_store_stream<unsigned, PV>(E.inds + (sp.ind + (size_t) f * g.N), bi);
						if (E.pre)
							vec_store_stream<T, PV>(E.pre + (sp.pooled + pooled_plane * f), best_pre);
					}
				}
			}
		});
		return true;
	}
	if constexpr (EPI == EPI_ACT) {
		act_dispatch(E.kind, [&](auto kc) {
			constexpr int KIND = decltype(kc)::value;
			#pragma unroll
			for (int i = 0; i < FB; ++i) {
				#pragma unroll
				for (int r = 0; r < MF::NACC; ++r) {
					const int f = f0 + wf * WT_F + FB * acc_row<T>(r, lk) + i;
					if (f >= g.F)
						continue;
					const T bv = bias_s[wf * WT_F + FB * acc_row<T>(r, lk) + i];
					const size_t o = (size_t) mm + (size_t) g.M * f;
					T z[MB], y[MB];
					#pragma unroll
					for (int j = 0; j < MB; ++j) {
						z[j] = acc[i][j][r] + bv;
						y[j] = act_f_coded<T, KIND>(z[j], E.p);
					}
					if (vec_out) {
						if (mm < g.M) {
							#pragma unroll
							for (int j0 = 0; j0 < MB; j0 += VS) {
								vec_store_stream<T, VS>(out + o + j0, *reinterpret_cast<T (*)[VS]>(&y[j0]));
								if (E.pre)
									vec_store_stream<T, VS>(E.pre + o + j0, *reinterpret_cast<T (*)[VS]>(&z[j0]));
							}
						}
					} else {
						#pragma unroll
						for (int j = 0; j < MB; ++j)
							if (mm + j < g.M) {
								out[o + j] = y[j];
								if (E.pre)
									E.pre[o + j] = z[j];
							}
					}
				}
			}
		});
		return true;
	}
	if constexpr (EPI == EPI_STATS) {
		/* Moments of this tile's rows per output column, from the accumulators: per lane the sums of (z - c) and
		 * (z - c)^2 about a value c of the same column (the first row of the wave's rows: a shift from within the
		 * data, so the squares do not cancel), added over the lanes of a column by a butterfly, then the waves along
		 * m merged in ascending order by the update of Chan et al. */
		T* const red = stage;                    /* [WAVES_M][BF][4]: count, shift, sum, sum of squares */
		static_assert(WAVES_M * (WAVES_F * WT_F) * 4 <= STAGE, "the moment partials reuse the A operand buffers");
		/* The cross-lane sums stay inside the vector ALU (lane_group_sum), and the shift, one value per column from the
		 * first lane of each group, is read as a scalar (fp32; fp64 has few columns per lane and shuffles it). */
		T c[FB][MF::NACC], s1[FB][MF::NACC], s2[FB][MF::NACC];
		#pragma unroll
		for (int i = 0; i < FB; ++i)
			#pragma unroll
			for (int r = 0; r < MF::NACC; ++r)
				c[i][r] = acc[i][0][r] + bias_s[wf * WT_F + FB * acc_row<T>(r, lk) + i];
		#pragma unroll
		for (int i = 0; i < FB; ++i)
			#pragma unroll
			for (int r = 0; r < MF::NACC; ++r) {
				if constexpr (std::is_same<T, float>::value) {
					/* the first lane of each half of the wavefront, read as scalars */
					const int bits = __builtin_bit_cast(int, c[i][r]);
					const int lo = __builtin_amdgcn_readlane(bits, 0), hi = __builtin_amdgcn_readlane(bits, 32);
					c[i][r] = __builtin_bit_cast(float, lk == 0 ? lo : hi);
				} else {
					c[i][r] = __shfl(c[i][r], lane & ~(TL - 1), 64);
				}
			}
		#pragma unroll
		for (int i = 0; i < FB; ++i)
			#pragma unroll
			for (int r = 0; r < MF::NACC; ++r) {
				const T bv = bias_s[wf * WT_F + FB * acc_row<T>(r, lk) + i];
				s1[i][r] = (T) 0;
				s2[i][r] = (T) 0;
				#pragma unroll
				for (int j = 0; j < MB; ++j) {
					const T d = mm + j < g.M ? (acc[i][j][r] + bv) - c[i][r] : (T) 0;
					s1[i][r] += d;
					s2[i][r] += d * d;
				}
			}
		#pragma unroll
		for (int i = 0; i < FB; ++i)
			#pragma unroll
			for (int r = 0; r < MF::NACC; ++r) {
				s1[i][r] = lane_group_sum<T, TL>(s1[i][r]);
				s2[i][r] = lane_group_sum<T, TL>(s2[i][r]);
			}
		/* rows of this wave that exist: all of them in the blocked order, else what is left of M */
		const int wave_rows = L.sample_blocks > 0 ? WT_M : max(0, min(WT_M, g.M - (tile * BM + wm * WT_M)));
		if (lc == TL - 1) {                  /* the lane that holds the group's totals */
			#pragma unroll
			for (int i = 0; i < FB; ++i)
				#pragma unroll
				for (int r = 0; r < MF::NACC; ++r) {
					T* dst = red + ((size_t) wm * BF + wf * WT_F + FB * acc_row<T>(r, lk) + i) * 4;
					dst[0] = (T) wave_rows;
					dst[1] = c[i][r];
					dst[2] = s1[i][r];
					dst[3] = s2[i][r];
				}
		}
		__syncthreads();
		for (int fl = tid; fl < BF; fl += THREADS) {
			if (f0 + fl >= g.F)
				continue;
			T n = (T) 0, mean = (T) 0, m2 = (T) 0;
			#pragma unroll
			for (int w = 0; w < WAVES_M; ++w) {
				const T* src4 = red + ((size_t) w * BF + fl) * 4;
				const T nb_ = src4[0];
				if (nb_ > (T) 0) {
					const T mb = src4[2] / nb_, meanb = src4[1] + mb, m2b = src4[3] - src4[2] * mb;
					const T nt = n + nb_, d = meanb - mean, wgt = nb_ / nt;
					mean += d * wgt;
					m2 += m2b + (d * d) * (n * wgt);
					n = nt;
				}
			}
			T* dst = E.stats + ((size_t) tile * g.F + (f0 + fl)) * 3;
			dst[0] = n;
			dst[1] = mean;
			dst[2] = m2;
		}
		/* the tile itself is stored below, like any other */
	}
	return false;
}

} /* namespace cattle_hip */

#endif /* CATTLE_HIP_GATHER_EPILOGUE_HPP_ */
